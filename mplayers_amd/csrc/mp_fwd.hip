// Forward scan of TRWP / ISGMR for gfx950: one wavefront per chain, see mp_common.h.
//
// Per pixel p of a chain (front pixel q = p - step), following HorizontalKernel /
// DiagonalKernelWide / DiagonalKernelNarrow of the reference (TRWP_forward.cu:82-376,
// ISGMR_forward.cu:123-431):
//     a[fd]  = U[q, fd] + rho * m[q, fd]                  (m[q] = message just computed, 0 at the start)
//     v[cd]  = min_fd a[fd] + w[p] * ctx(cd, fd)          (largest fd on ties)
//     m[p,:] = v - min_cd v                               (largest cd on ties)
// with U = rho * (S - m_dir_old) - m_inv_old taken from the belief plane S = unary + sum_k m_k
// instead of re-summing all messages (UpdateUnaryKernel, TRWP_forward.cu:60-80).  TRWP (Gauss-Seidel
// over directions) forms U on the fly from S, m_dir, m_inv and keeps S up to date; ISGMR (Jacobi)
// finds U of every direction precomputed in place of the old messages.
//
// Compiled once per R (labels per lane) and per kind of scan (with or without argmin labels) with
// -DMPL_INST_R=<R> -DMPL_INST_TRAIN=<0|1>.

#include <type_traits>

#include "mp_fwd_step.h"

namespace mpl {
namespace {

template <int R>
struct PixF {
  float s[R], md[R], mi[R];
  float w;
};

// Several wavefronts on one chain (launches with far fewer chains than the chip has SIMDs, dense
// table): every wavefront of the workgroup walks the chain and holds the same state, but scans only
// its share of the front labels of a pixel; the partial minima (and their labels) meet in LDS,
// one slot per wavefront, and every wavefront folds all of them in the order of the front labels
// (`<=`: the later share wins ties, as the one scan over all front labels does), so the state stays
// identical in all of them, bit for bit what one wavefront computes.  Two sets of slots alternate:
// a wavefront that runs ahead writes the other set, and it cannot reach this set again before the
// barrier of the next step, which every wavefront passes only after it has read this one.
template <int R, bool TRAIN>
__device__ __forceinline__ void split_combine(float* xchg, int n_waves, int wave, int lane, int parity,
                                              float (&v)[R], int (&fd_idx)[R]) {
  constexpr int S = TRAIN ? 2 * R : R;  // dwords per lane and slot
  float* set = xchg + (size_t)parity * n_waves * kWave * S;
  float* mine = set + ((size_t)wave * kWave + lane) * S;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    mine[j] = v[j];
    if (TRAIN) mine[R + j] = __builtin_bit_cast(float, fd_idx[j]);
  }
  __syncthreads();
  for (int k = 0; k < n_waves; ++k) {
    const float* theirs = set + ((size_t)k * kWave + lane) * S;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const float pv = theirs[j];
      if (TRAIN) {
        const int pi = __builtin_bit_cast(int, theirs[R + j]);
        const bool take = (k == 0) || (pv <= v[j]);
        v[j] = take ? pv : v[j];
        fd_idx[j] = take ? pi : fd_idx[j];
      } else {
        v[j] = k == 0 ? pv : fminf(v[j], pv);
      }
    }
  }
}

// One chain.  KT: > 0 band with compile-time K, 0 band with run-time K, -1 dense, -21 dense with
// exactly 21 labels, -2 truncated linear context of any width (linear_step), -3 dense 1-D table with
// the front labels split over the wavefronts of the workgroup (split_combine; xchg: its LDS slots).
// VEC: L % R == 0 (vector accesses).  MASK: some lanes own labels >= L.
// C0: the table's entry 0 is its smallest (band steps only; CtxDesc::c0_is_min), which gives the
// normalisation minimum without a second reduction.
// THROUGH: store_through (mp_common.h).
template <int R, bool VEC, bool MASK, bool TRAIN, int JACOBI, int KT, bool C0 = false, bool THROUGH = false>
__device__ __forceinline__ void run_chain_fwd(const SweepParams& p, const CtxDesc& desc,
                                              const ChainCtx& ch, float* a_s, const float* ctx_s,
                                              const bool skip_s_store_in, float* xchg = nullptr) {
  constexpr bool SPLIT = (KT == -3);
  // (every lane full: 64, 128, 192 or 256 labels, whole cache lines)
  constexpr int kLd = load_policy(!MASK);
  constexpr int kSt = THROUGH ? kStoreThrough : store_policy(R, !MASK);
  const int L = p.L;
  // The caller's initial messages turned out to be all zero (the usual case: the reference's
  // callers pass a cleared tensor) and this is a sweep that can profit: S = Q = U = unary, so the
  // unary terms are read in place of the plane, and the even sweep of the first pair has nothing to
  // store (the odd one reads the unary terms again).  Wave-uniform, the same for every chain.
  const bool zfirst = JACOBI != 2 && p.zero_first && desc.msg_nonzero == 0;
  const bool skip_s_store = skip_s_store_in || (!JACOBI && zfirst && (ch.dir & 1) == 0);
  const int64_t HW = (int64_t)p.H * p.W;
  const int64_t P = (int64_t)p.B * HW;
  const int64_t N = P * L;
  const int dir = ch.dir;
  const int64_t img_p = (int64_t)ch.bv * HW;  // first pixel of this batch item
  const int64_t img_e = img_p * L;
  const int vbytes = L * 4;
  // plane bases of this batch item and direction; descriptors are formed per access
  // Jacobi: the plane of this direction in msg_in holds U itself (written by the host's
  // element-wise pass before the sweeps), so one plane is read per pixel instead of three
  // JACOBI == 2 (four directions, rho == 1): no U plane either; U of the pair {dir, dir^1} is the
  // unary plus the old messages of the other pair, read here (three planes in, but the pass that
  // stores U, five planes in and two out per iteration, is not run)
  const int oth = (dir & ~1) ^ 2;  // the even direction of the other pair
  const float* __restrict__ bS =
      (zfirst ? p.belief_zero
              : (JACOBI == 1 ? p.msg_in + (int64_t)(p.u_pair_share ? (dir & ~1) : dir) * p.u_stride
                             : p.belief)) + img_e;
  const float* __restrict__ bMd = p.msg_in + (int64_t)(JACOBI == 2 ? oth : dir) * N + img_e;
  const float* __restrict__ bMi = p.msg_in + (int64_t)(JACOBI == 2 ? oth + 1 : (dir ^ 1)) * N + img_e;
  float* __restrict__ bMo = p.msg_out + (int64_t)dir * N + img_e;
  float* __restrict__ bSo = (JACOBI ? nullptr : p.belief_out + img_e);
  uint8_t* __restrict__ bImin = TRAIN ? p.idx_min + (int64_t)dir * N + img_e : nullptr;
  const int img_bytes_p = (int)(HW * 4 > 0x7fffffff ? 0x7fffffff : HW * 4);
  const rsrc_t dW = make_rsrc(p.edge + (int64_t)dir * P + img_p, img_bytes_p);
  const rsrc_t dInorm = make_rsrc(TRAIN ? p.idx_norm + (int64_t)dir * P + img_p : nullptr,
                                  TRAIN ? (int)HW : 0);
  const float rho = p.rho;
  const float inf = INFINITY;
  const int lane = SPLIT ? (int)(threadIdx.x & (kWave - 1)) : (int)threadIdx.x;
  const int lab0 = R * lane;
  const int foff = lab0 * 4;  // byte offset of this lane's block inside a pixel's float vector
  const int n = ch.n;
  // SPLIT: the wavefronts of the workgroup share the front labels; the first one stores
  const int wave = SPLIT ? uniform_i((int)(threadIdx.x / kWave)) : 0;
  const int n_waves = SPLIT ? (int)(blockDim.x / kWave) : 1;
  const bool store_ok = !SPLIT || wave == 0;
  // front labels per wavefront: whole trips of the dense scan
  // (the division by the number of wavefronts runs on the vector unit: without the explicit
  // read-back the bounds, and with them the loop counter of the scan and every address it forms,
  // would stay in vector registers)
  const int fd_chunk = SPLIT ? uniform_i(split_share(L, R, n_waves)) : L;
  const int fd_lo = SPLIT ? uniform_i(min(wave * fd_chunk, L)) : 0;
  const int fd_hi = SPLIT ? uniform_i(min(fd_lo + fd_chunk, L)) : L;
  // dense scan, several labels per lane: this wavefront's copy of a[], the table moved down by one
  // entry, and the sliding table values of the lane's labels at the first front label
  float* a_w = a_s + (SPLIT ? wave * kMaxL : 0);
  const float* c1_s = ctx_s + dense_c1_offset(L);
  const float* csym_s = c1_s + dense_c1_floats(L);  // the table around its centre (dense1d_argmin)
  // (only where the dense scan is the kernel's step: a kernel compiled for a band or a
  // truncated-linear table meets it at pixels with a negative edge weight and takes
  // dense1d_step_lanes)
  constexpr bool kDenseMain = KT == -1 || KT == -3;
  float cv0_chain[R];
  if constexpr (kDenseMain) {
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int l = lab0 + j < L ? lab0 + j : L - 1;
      cv0_chain[j] = ctx_s[l > fd_lo ? l - fd_lo : fd_lo - l];
    }
  }

  bool valid[R];
  // a lane's labels beyond the last one are kept at +inf by a maximum with +inf (-inf for the
  // others, which changes nothing): one instruction in the short encoding, no lane masks to hold
  float floor_l[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    valid[j] = MASK ? (lab0 + j < L) : true;
    floor_l[j] = valid[j] ? -INFINITY : INFINITY;
  }

  float c_reg[KT > 0 ? KT : 1];
  if (KT > 0) {
#pragma unroll
    for (int k = 0; k < KT; ++k) c_reg[k] = p.ctx[k];
  }
  // KT == -21: dense path with the label count fixed at 21 (the segmentation case)
  constexpr int LT = (KT == -21) ? 21 : 0;
  float tcol[LT > 0 ? LT : 1];
  if (LT > 0) {
#pragma unroll
    for (int fd = 0; fd < LT; ++fd) tcol[fd] = ctx_s[fd * LT + (lane < LT ? lane : LT - 1)];
  }
  const int K = desc.band_k;
  // (in a vector register for the whole chain: the far candidate multiplies it by the edge weight
  // and adds the minimum, both scalars, and a multiply-add takes one scalar operand)
  float cmax = desc.cmax;
  asm volatile("" : "+v"(cmax));

  // first Gauss-Seidel iteration over all-zero initial messages: the plane of this direction has
  // not been swept yet, and neither has the opposite one when this direction is the even one
  const bool md_zero = !JACOBI && p.first_iter && desc.msg_nonzero == 0;
  const bool mi_zero = md_zero && (dir & 1) == 0;
  // Gauss-Seidel pairs (p.pair_q): between the sweep of an even direction and the sweep of its
  // opposite the belief plane holds Q = S - m_dir - m_inv, which neither sweep changes:
  //   first sweep  (even):  reads S, m_dir, m_inv; stores m_dir' and Q
  //   second sweep (odd):   reads Q and m_inv (= m_even'), not its own old messages:
  //                         S - m_dir = Q + m_inv;  stores m_dir' and S = Q + m_inv + m_dir'
  // (at a chain start, where no message is written, the plane is converted with the old values)
  const bool pair_first = !JACOBI && p.pair_q && (dir & 1) == 0;
  const bool pair_second = !JACOBI && p.pair_q && (dir & 1) == 1;
  // VEC: one descriptor per plane for the whole kernel, covering the batch item's image; a lane
  // reaches its labels of a pixel through its vector offset, and a lane without labels (or a step
  // that must not store) through an offset no descriptor covers.  Nothing but one multiply, one
  // add and one select per pixel is then spent on addressing (descriptors formed per access cost
  // some eight scalar instructions each, which a chain-starved launch -- one wavefront per SIMD,
  // every instruction an issue slot of its own -- cannot hide).  Planes that are not to be read
  // (all-zero initial messages, the odd sweep's own old messages) or stored get an empty descriptor.
  const bool lane_ok = !MASK || lab0 < L;
  const int img_bytes = (int)(unsigned)(HW * L * 4);
  // (VEC and MASK: a lane without labels carries the size of the image in place of its offset, which
  // takes every access of its past the end of every plane without a select per access; the host
  // gives images beyond 2 GiB, where that sum could wrap, to the kernels that form a descriptor per
  // access)
  // (one label per lane: every image goes through these kernels, and the select stays)
  constexpr bool kAddDead = R > 1;
  const unsigned foff_ok = lane_ok ? (unsigned)foff : (unsigned)img_bytes;
  const rsrc_t rS = make_rsrc(bS, img_bytes);
  const rsrc_t rMd0 = make_rsrc(bMd, md_zero ? 0 : img_bytes);  // chain start
  const rsrc_t rMd = make_rsrc(bMd, (md_zero || pair_second) ? 0 : img_bytes);
  const rsrc_t rMi = make_rsrc(bMi, mi_zero ? 0 : img_bytes);
  const rsrc_t rMo = make_rsrc(bMo, img_bytes);
  const rsrc_t rSo = make_rsrc(bSo, (JACOBI || skip_s_store) ? 0 : img_bytes);
  const rsrc_t rImin = make_rsrc(bImin, TRAIN ? (int)(HW * L) : 0);
  // loads of the next pixel; past the end of the chain the last pixel is fetched again
  const int last_p = ch.pix0 + (n - 1) * ch.pstep;
  int ld_p = ch.pix0;
  int ld_t = 0;
  auto load_next = [&](const bool first = false) __attribute__((always_inline)) {
    PixF<R> r;
    // VEC: the prefetch simply runs on past the end of the chain: what lies there is another pixel
    // of the image or outside the descriptors (reads as 0), and no step uses it
    const unsigned pp = (unsigned)uniform_i((VEC || ld_t < n) ? ld_p : last_p);
    const unsigned so = pp * (unsigned)vbytes;
    if constexpr (VEC) {
      const int vo = (int)(kAddDead ? so + foff_ok : (lane_ok ? so + (unsigned)foff : kDeadWide));
      buf_load<R, true, kLd>(rS, vo, 0u, r.s);
      if (JACOBI == 0) {
        buf_load<R, true, kLd>(first ? rMd0 : rMd, vo, 0u, r.md);
        buf_load<R, true, kLd>(rMi, vo, 0u, r.mi);
      } else if (JACOBI == 2) {
        buf_load<R, true, kLd>(rMd0, vo, 0u, r.md);
        buf_load<R, true, kLd>(rMi, vo, 0u, r.mi);
      }
    } else {
      const int nrec = (int)(so + (unsigned)vbytes);
      buf_load<R, VEC, kLd>(make_rsrc(bS, nrec), foff, so, r.s);
      if (JACOBI == 0) {
        // planes that still hold all-zero initial messages are read through an empty descriptor
        buf_load<R, VEC, kLd>(make_rsrc(bMd, (md_zero || (pair_second && ld_t > 0)) ? 0 : nrec), foff, so,
                         r.md);
        buf_load<R, VEC, kLd>(make_rsrc(bMi, mi_zero ? 0 : nrec), foff, so, r.mi);
      } else if (JACOBI == 2) {
        buf_load<R, VEC, kLd>(make_rsrc(bMd, nrec), foff, so, r.md);
        buf_load<R, VEC, kLd>(make_rsrc(bMi, nrec), foff, so, r.mi);
      }
    }
    r.w = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(dW, (int)(pp * 4u), 0, 0));
    ld_p += ch.pstep;
    ld_t += 1;
    return r;
  };

  // chain start: its front lies outside the image and the reference never writes it.  The Jacobi
  // buffers alternate, so there the start pixel is written with the zeros it keeps in the reference.
  float prev[R], uf[R];
  {
    const PixF<R> p0 = load_next(true);
    MPL_ORDER_LOADS();  // (the chain start's loads stay ahead of the ring's)
    float conv[R];  // the start pixel's belief-plane value in the other representation
#pragma unroll
    for (int j = 0; j < R; ++j) conv[j] = 0.f;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      prev[j] = 0.f;
      float un = JACOBI == 2 ? (p0.s[j] + p0.md[j]) + p0.mi[j] : p0.s[j];
      if (!JACOBI) {
        const float t0 = pair_second ? p0.s[j] + p0.mi[j] : p0.s[j] - p0.md[j];
        un = fmaf(t0, rho, -p0.mi[j]);
        conv[j] = pair_second ? t0 + p0.md[j] : t0 - p0.mi[j];
      }
      uf[j] = valid[j] ? un : inf;
    }
    if constexpr (SPLIT) {
      // the first wavefront is about to overwrite the start pixel's entry of the belief plane, in
      // place: not before every wavefront of the chain has read it
      wait_vmem<0>();
      __syncthreads();
    }
    const unsigned so0 = (unsigned)ch.pix0 * (unsigned)vbytes;
    const int vo0 = (int)((lane_ok && store_ok) ? so0 + (unsigned)foff : kDeadWide);
    const int nrec0 = store_ok ? (int)(so0 + (unsigned)vbytes) : 0;
    if (!JACOBI && p.pair_q && !skip_s_store) {
      if constexpr (VEC)
        buf_store<R, true, kSt>(rSo, vo0, 0u, conv);
      else
        buf_store<R, VEC, kSt>(make_rsrc(bSo, nrec0), foff, so0, conv);
    }
    if (JACOBI || p.zero_start) {
      float z[R];
#pragma unroll
      for (int j = 0; j < R; ++j) z[j] = 0.f;
      if constexpr (VEC)
        buf_store<R, true, kSt>(rMo, vo0, 0u, z);
      else
        buf_store<R, VEC, kSt>(make_rsrc(bMo, nrec0), foff, so0, z);
    }
  }

  // memory instructions per step: 1 or 3 label vectors + the weight in, 1-2 label vectors
  // (+ indices) out
  constexpr int kOps = (JACOBI == 1 ? 1 : 3) * vec_ops(R, VEC) + 1 + (JACOBI ? 1 : 2) * vec_ops(R, VEC) +
                       (TRAIN ? byte_ops(R, VEC) + 1 : 0);
  constexpr int D = ring_depth(kOps);
  // Two banks of D pixels in flight: while the steps consume one, the loads of D pixels ahead land
  // in the other, so that after 2 D steps every value sits in the register it started in (with a
  // single bank the loop ends in one register move per value in flight).
  PixF<R> ring[D], ring2[D];
#pragma unroll
  for (int u = 0; u < D; ++u) {
    ring[u] = load_next();
    // keeps the pixels' loads in this order: the compiler's own waits in the loop are sized for
    // the order it sees here, and a later pixel's loads placed first would make them drain the queue
    MPL_ORDER_LOADS();
  }

  // The dense 1-D steps leave out candidates that are no number, so a term that is none must not become the -inf
  // that a maximum with the floor makes of it.
  const bool keep_nan = kDenseMain && !(R == 1 && (p.ctx2d || (KT == -1 && L < kSlidingMinL)));
  int st_p = ch.pix0 + ch.pstep;
  // in_chain: a constant `true` where the caller knows that step t lies inside the chain and that
  // no edge weight of the chain is negative
  auto step = [&](const PixF<R>& px, const int t, const auto in_chain) __attribute__((always_inline)) {
      constexpr bool kPlain = decltype(in_chain)::value;
      // steps past the end compute on stale data and store nothing
      const bool live = kPlain || t < n;
      float tt[R], un[R];
#pragma unroll
      for (int j = 0; j < R; ++j) {
        float x = JACOBI == 2 ? (px.s[j] + px.md[j]) + px.mi[j] : px.s[j];
        if (!JACOBI) {
          // unary + the other directions' messages
          tt[j] = pair_second ? px.s[j] + px.mi[j] : px.s[j] - px.md[j];
          x = fmaf(tt[j], rho, -px.mi[j]);  // UpdateUnaryKernel, TRWP_forward.cu:70-78
        } else {
          tt[j] = 0.f;
        }
        un[j] = !MASK ? x : keep_nan ? (valid[j] ? x : inf) : fmaxf(x, floor_l[j]);
      }
      const float w = uniform_f(px.w);
      float a[R], v[R];
      int fd_idx[R];
#pragma unroll
      for (int j = 0; j < R; ++j) a[j] = fmaf(rho, prev[j], uf[j]);
      // the normalisation minimum of v (every path ends with it or with a cheaper way to it: the
      // usual path then runs through without a flag to test)
      float nmin;
      auto norm_min = [&]() __attribute__((always_inline)) {
        float vm = inf;
#pragma unroll
        for (int j = 0; j < R; ++j) vm = fminf(vm, MASK ? fmaxf(v[j], floor_l[j]) : v[j]);
        return wave_min_fast(vm);
      };
      // (the usual case falls through; the trips of steps that the caller vouches for do not ask)
      if ((KT >= 0 || KT == -2) && (kPlain || __builtin_expect(w >= 0.f, 1))) {
        // (several labels per lane without argmin labels: the reduction and the first tap in one
        // block)
        constexpr bool kHead = R >= 2 && !TRAIN && KT >= 2;
        float amin;
        float hup[R], hdn[R];
        if constexpr (kHead) {
          float red;
          band_head(a, px.w, c_reg[0], c_reg[1], red, v, hup, hdn);
          amin = readlane_f(red, 63);
        } else {
          float am = a[0];
#pragma unroll
          for (int j = 1; j < R; ++j) am = fminf(am, a[j]);
          amin = wave_min_fast(am);
        }
        int fstar = L - 1;
        if (TRAIN) {
          bool pr[R];
#pragma unroll
          for (int j = 0; j < R; ++j) pr[j] = (a[j] == amin);
          fstar = last_label<R>(pr, L - 1);
        }
        if constexpr (KT == -2) {
          linear_step<R, TRAIN>(a, w, desc.slope, cmax, amin, fstar, lab0, lane, L, a_s, ctx_s, v,
                                fd_idx);
        } else {
          // (after the head the weight is taken from the vector register every lane loaded it
          // into: the minimum arrives in a scalar register, and a multiply-add reads one scalar)
          band_step<R, TRAIN, (KT > 0 ? KT : 0), kHead>(a, kHead ? px.w : w, K, c_reg, ctx_s, cmax, amin,
                                                        fstar, lab0, v, fd_idx, hup, hdn);
        }
        if constexpr (KT != -2 && C0) {
          // every candidate is >= amin + w*c[0], which the centre tap of label argmin(a) attains
          nmin = fmaf(kHead ? px.w : w, KT > 0 ? c_reg[0] : ctx_s[0], amin);
        } else {
          nmin = norm_min();
        }
      } else if (R == 1 && KT < 0 && (p.ctx2d || (KT == -1 && L < kSlidingMinL))) {  // (the full table is in LDS then)
        if constexpr (LT > 0) {
          // 21 labels: the scan over front labels fully unrolled, context column in registers.
          // The edge weight stays in a vector register (every lane loaded the same one): a[fd]
          // arrives in a scalar register, and a multiply-add takes one scalar operand only.
          float af[LT], val[LT];
#pragma unroll
          for (int fd = 0; fd < LT; ++fd) af[fd] = readlane_f(a[0], fd);
          // (a multiply-add may read a[fd] only two issue slots after it reached its scalar
          // register: all of them first, then the multiply-adds)
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int fd = 0; fd < LT; ++fd) val[fd] = fmaf(px.w, tcol[fd], af[fd]);
          float best = val[LT - 1];
#pragma unroll
          for (int fd = LT - 2; fd >= 1; fd -= 2) best = fminf(fminf(val[fd], val[fd - 1]), best);
          if ((LT & 1) == 0) best = fminf(best, val[0]);
          v[0] = best;
          if (TRAIN) {
            // the scan in descending order with a strict comparison keeps the largest front label
            // that attains the minimum
            float red = valid[0] ? best : inf;
            argmin_and_lane_min_21(val, best, red, fd_idx[0]);
            nmin = readlane_f(red, 31);
          } else {
            fd_idx[0] = LT - 1;
            nmin = norm_min();
          }
        } else {
          dense_step_r1<TRAIN>(a[0], L, w, lane, ctx_s, v[0], fd_idx[0]);
          nmin = norm_min();
        }
      } else if (live) {
        if constexpr (R > 1 || KT < 0) {  // (one label per lane: 1-D tables)
          if constexpr (kDenseMain) {
            dense1d_step<R, TRAIN>(a, w, lab0, a_w, c1_s, cv0_chain, v, fd_idx, fd_lo, fd_hi);
            if constexpr (SPLIT) split_combine<R, TRAIN>(xchg, n_waves, wave, lane, t & 1, v, fd_idx);
            // (fd_idx holds the first front label of the trip with the argmin; only a wavefront
            // that stores needs the label itself)
            if (TRAIN && store_ok) dense1d_argmin<R>(v, fd_idx, w, lab0, L, a_w, csym_s, fd_idx);
          } else {
            // a pixel with a negative edge weight in a kernel compiled for a band or a
            // truncated-linear table: the same candidates, broadcast from the lanes
            dense1d_step_lanes<R, TRAIN, VEC>(a, w, L, lab0, ctx_s, v, fd_idx, 0, L);
          }
        } else {
          dense_step<R, TRAIN>(a, valid, w, L, p.ctx2d, lab0, a_s, ctx_s, v, fd_idx);
        }
        nmin = norm_min();
      } else {
#pragma unroll
        for (int j = 0; j < R; ++j) {
          v[j] = 0.f;
          fd_idx[j] = 0;
        }
        nmin = 0.f;
      }
      float m[R], sn[R];
#pragma unroll
      for (int j = 0; j < R; ++j) {
        m[j] = v[j] - nmin;  // MsgNormNaive, commonCUDA.cuh:126-128
        sn[j] = pair_first ? tt[j] - px.mi[j] : tt[j] + m[j];
        prev[j] = m[j];  // (a lane without a label keeps a = +inf through uf, whatever prev is)
        uf[j] = un[j];
      }
      const unsigned sp = (unsigned)uniform_i(st_p);
      const unsigned so = sp * (unsigned)vbytes;
      const unsigned sob = sp * (unsigned)L;
      if constexpr (VEC) {
        const bool on = lane_ok && live && store_ok;  // nothing is stored past the end
        const int vo = (int)(kAddDead ? ((live && store_ok) ? so + foff_ok : kDeadWide)
                                      : (on ? so + (unsigned)foff : kDeadWide));
        buf_store<R, true, kSt>(rMo, vo, 0u, m);
        if (!JACOBI) buf_store<R, true, kSt>(rSo, vo, 0u, sn);
        if (TRAIN) buf_store_u8<R, true, kSt>(rImin, (int)(on ? sob + (unsigned)lab0 : kDeadWide), 0u, fd_idx);
      } else {
        const int nrec = (live && store_ok) ? (int)(so + (unsigned)vbytes) : 0;
        buf_store<R, VEC, kSt>(make_rsrc(bMo, nrec), foff, so, m);
        if (!JACOBI) buf_store<R, VEC, kSt>(make_rsrc(bSo, skip_s_store ? 0 : nrec), foff, so, sn);
        if (TRAIN)
          buf_store_u8<R, VEC, kSt>(make_rsrc(bImin, (live && store_ok) ? (int)(sob + (unsigned)L) : 0), lab0, sob, fd_idx);
      }
      if (TRAIN) {
        bool pr[R];
#pragma unroll
        for (int j = 0; j < R; ++j) pr[j] = valid[j] && (v[j] == nmin);
        const int nidx = last_label<R>(pr, L - 1);
        // every lane stores the same byte to the same address
        __builtin_amdgcn_raw_buffer_store_b8((unsigned char)nidx, dInorm, (live && store_ok) ? (int)sp : kDeadOffset, 0, 0);
      }
      st_p += ch.pstep;
  };
  // Trips of 2 D steps that lie inside the chain, on a chain without negative edge weights (the
  // band and the label scans hold for every step then): nothing in them asks whether a step is past
  // the end or which way its weight points, and the step for negative weights is not part of their
  // code.  A chain with such a weight takes the loop below from its first step.  Without argmin
  // labels, or with one label per lane (the scans of the usual training sizes with more labels
  // share their SIMDs and wait for memory, not for issue slots; their code is large enough as it is).
  int t0 = 1;
  if constexpr (!TRAIN || R == 1) {
    bool plain = true;
    if constexpr (KT >= 0 || KT == -2) {
      if (n > 2 * D) {  // (there is such a trip)
        bool bad = false;
        for (int i = lane; i < n; i += kWave) {
          const unsigned pi = (unsigned)(ch.pix0 + i * ch.pstep);
          const float wi = __builtin_bit_cast(
              float, __builtin_amdgcn_raw_buffer_load_b32(dW, (int)(pi * 4u), 0, 0));
          bad |= !(wi >= 0.f);
        }
        plain = ballot(bad) == 0;
      }
    }
    for (; plain && t0 + 2 * D <= n; t0 += 2 * D) {
#pragma unroll
      for (int u = 0; u < D; ++u) {
        // the loads of this ring slot were followed by at most D-1 steps' worth of memory operations
        wait_vmem<(D - 1) * kOps>();
        const PixF<R> px = ring[u];
        ring2[u] = load_next();
        step(px, t0 + u, std::true_type());
        // (the steps have no branch left between them; kept apart, the scalars of one step do not
        // pile up on those of the next, and none of them is spilled inside the loop)
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int u = 0; u < D; ++u) {
        wait_vmem<(D - 1) * kOps>();
        const PixF<R> px = ring2[u];
        ring[u] = load_next();
        step(px, t0 + D + u, std::true_type());
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  for (; t0 < n; t0 += 2 * D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      wait_vmem<(D - 1) * kOps>();
      const PixF<R> px = ring[u];
      ring2[u] = load_next();
      step(px, t0 + u, std::false_type());
    }
    if (t0 + D >= n) break;  // wave-uniform
#pragma unroll
    for (int u = 0; u < D; ++u) {
      wait_vmem<(D - 1) * kOps>();
      const PixF<R> px = ring2[u];
      ring[u] = load_next();
      step(px, t0 + D + u, std::false_type());
    }
  }
}

template <int R, bool VEC, bool MASK, bool TRAIN, int JACOBI, bool THROUGH = false>
__global__ void __launch_bounds__(kWave) sweep_fwd_kernel(const SweepParams p) {
  extern __shared__ __align__(16) float smem[];
  float* a_s = smem;            // kMaxL floats
  float* ctx_s = smem + kMaxL;  // L*L floats, or L and the table moved down by one and around its centre
  const int lane = threadIdx.x;
  const int L = p.L;
  const ChainCtx ch = locate_chain(p);
  if (!JACOBI && !p.pair_q && ch.n < 2) return;  // nothing to write

  CtxDesc desc;
  if (p.desc != nullptr) {
    desc = *p.desc;
  } else {
    desc.band_k = 0;
    desc.c0_is_min = 0;
    desc.cmax = 0.f;
    desc.msg_nonzero = 1;
    desc.linear = 0;
    desc.slope = 0.f;
  }
  // context table into LDS (dense path, run-time band taps, negative-weight fallback)
  if (R == 1 && (p.ctx2d || (is_dense(desc) && L < kSlidingMinL))) {
    // full symmetric table for dense_step_r1: tab[fd * L + cd] = ctx(cd, fd), TRWP_forward.cu:101-113
    for (int i = lane; i < L * L; i += kWave) {
      const int fd = i / L, cd = i - fd * L;
      const int lo = cd < fd ? cd : fd, hi = cd < fd ? fd : cd;
      ctx_s[i] = p.ctx[p.ctx2d ? lo * L + hi : hi - lo];
    }
  } else {
    const int n_ctx = p.ctx2d ? L * L : L;
    for (int i = lane; i < n_ctx; i += kWave) ctx_s[i] = p.ctx[i];
    if (desc.band_k == 0) {  // (the dense scan is this kernel's step)
      float* c1_s = ctx_s + dense_c1_offset(L);
      for (int i = lane; i < dense_c1_floats(L); i += kWave) c1_s[i] = i + 1 < L ? p.ctx[i + 1] : 0.f;
      if (TRAIN) fill_dense_sym<R>(c1_s + dense_c1_floats(L), p.ctx, L, lane, kWave);
    }
  }
  __syncthreads();

  // Gauss-Seidel, chain-starved launches: the sweep of the opposite direction visits the same
  // pixels in reverse and depends on nothing but this chain's own first sweep, so the wavefront
  // runs it right away (p.fused_pair) instead of a second launch doing so.  What the first sweep
  // stored is read back by the same wavefront, in program order.
  const int halves = (!JACOBI && p.fused_pair) ? 2 : 1;
#pragma clang loop unroll(disable)
  for (int half = 0; half < halves; ++half) {
    ChainCtx c = ch;
    bool skip_s = p.skip_s_store != 0;
    if (half) {
      c.dir = ch.dir ^ 1;
      c.pix0 = ch.pix0 + (ch.n - 1) * ch.pstep;
      c.pstep = -ch.pstep;
      skip_s = p.skip_s_store2 != 0;
      wait_vmem<0>();
      __syncthreads();
    }
    // wide truncated-linear contexts: two label scans instead of 2K-1 taps or the dense scan
    if (desc.linear && !p.ctx2d && (desc.band_k == 0 || desc.band_k > 4)) {
      run_chain_fwd<R, VEC, MASK, TRAIN, JACOBI, -2, false, THROUGH>(p, desc, c, a_s, ctx_s, skip_s);
      continue;
    }
    // (a band whose entry 0 is not its smallest -- no Potts, linear or quadratic table -- takes the
    // taps at run time and reduces for the normalisation minimum)
    if (desc.band_k > 0 && !desc.c0_is_min) {
      run_chain_fwd<R, VEC, MASK, TRAIN, JACOBI, 0, false, THROUGH>(p, desc, c, a_s, ctx_s, skip_s);
      continue;
    }
    switch (desc.band_k) {
      case 0:
        if (R == 1 && L == 21 && p.ctx2d)
          run_chain_fwd<R, VEC, MASK, TRAIN, JACOBI, (R == 1 ? -21 : -1), false, THROUGH>(p, desc, c, a_s, ctx_s, skip_s);
        else
          run_chain_fwd<R, VEC, MASK, TRAIN, JACOBI, -1, false, THROUGH>(p, desc, c, a_s, ctx_s, skip_s);
        break;
      case 2: run_chain_fwd<R, VEC, MASK, TRAIN, JACOBI, 2, true, THROUGH>(p, desc, c, a_s, ctx_s, skip_s); break;
      case 3: run_chain_fwd<R, VEC, MASK, TRAIN, JACOBI, 3, true, THROUGH>(p, desc, c, a_s, ctx_s, skip_s); break;
      case 4: run_chain_fwd<R, VEC, MASK, TRAIN, JACOBI, 4, true, THROUGH>(p, desc, c, a_s, ctx_s, skip_s); break;
      default:
        // wider bands with the taps in registers: the table is constant from band_k on, so the
        // taps between band_k and the compiled width are the dense scan's own candidates
        // (only with several labels per lane: the short chains of small label counts gain nothing
        // and pay for the larger kernel)
        if constexpr (R >= 2) {
          if (desc.band_k <= 8) {
            run_chain_fwd<R, VEC, MASK, TRAIN, JACOBI, 8, true, THROUGH>(p, desc, c, a_s, ctx_s, skip_s);
            break;
          }
          if (desc.band_k <= 16) {
            run_chain_fwd<R, VEC, MASK, TRAIN, JACOBI, 16, true, THROUGH>(p, desc, c, a_s, ctx_s, skip_s);
            break;
          }
        }
        run_chain_fwd<R, VEC, MASK, TRAIN, JACOBI, 0, true, THROUGH>(p, desc, c, a_s, ctx_s, skip_s);
        break;
    }
  }
}

// A dense 1-D table in a launch with far fewer chains than the chip has SIMDs (p.split wavefronts
// per chain, chosen by the host; several labels per lane only).  Every wavefront of the workgroup
// runs the chain; see split_combine.
constexpr int kSplitMaxWaves = 8;
template <int R, bool VEC, bool MASK, bool TRAIN, int JACOBI>
__global__ void __launch_bounds__(kSplitMaxWaves * kWave) sweep_fwd_split_kernel(const SweepParams p) {
  extern __shared__ __align__(16) float smem[];
  const int L = p.L;
  float* a_s = smem;  // kMaxL floats per wavefront
  float* ctx_s = smem + (blockDim.x / kWave) * kMaxL;  // L floats, and the table moved down by one
  float* c1_s = ctx_s + dense_c1_offset(L);
  float* csym_s = c1_s + dense_c1_floats(L);
  float* xchg = csym_s + dense_sym_floats(R);
  const ChainCtx ch = locate_chain(p);
  if (!JACOBI && !p.pair_q && ch.n < 2) return;  // nothing to write (the same for every wavefront)
  CtxDesc desc;
  desc.band_k = 0;  // the dense scan is exact for any table; the descriptor only says whether
  desc.c0_is_min = 0;  // the initial messages are zero
  desc.cmax = 0.f;
  desc.msg_nonzero = p.desc != nullptr ? p.desc->msg_nonzero : 1;
  desc.linear = 0;
  desc.slope = 0.f;
  for (int i = threadIdx.x; i < L; i += blockDim.x) ctx_s[i] = p.ctx[i];
  for (int i = threadIdx.x; i < dense_c1_floats(L); i += blockDim.x) c1_s[i] = i + 1 < L ? p.ctx[i + 1] : 0.f;
  if (TRAIN) fill_dense_sym<R>(csym_s, p.ctx, L, (int)threadIdx.x, (int)blockDim.x);
  __syncthreads();
  const int halves = (!JACOBI && p.fused_pair) ? 2 : 1;
#pragma clang loop unroll(disable)
  for (int half = 0; half < halves; ++half) {
    ChainCtx c = ch;
    bool skip_s = p.skip_s_store != 0;
    if (half) {
      c.dir = ch.dir ^ 1;
      c.pix0 = ch.pix0 + (ch.n - 1) * ch.pstep;
      c.pstep = -ch.pstep;
      skip_s = p.skip_s_store2 != 0;
      wait_vmem<0>();
      __syncthreads();
    }
    run_chain_fwd<R, VEC, MASK, TRAIN, JACOBI, -3>(p, desc, c, a_s, ctx_s, skip_s, xchg);
  }
}

inline size_t split_lds_bytes(int L, int R, int waves, bool train) {
  return sizeof(float) * ((size_t)waves * kMaxL + dense_c1_offset(L) + dense_c1_floats(L) +
                          dense_sym_floats(R) + (size_t)2 * waves * kWave * (train ? 2 * R : R));
}

template <int R, bool VEC, bool MASK, bool TRAIN>
void launch_vm_split(const SweepParams& p, bool jacobi, hipStream_t st) {
  const int blocks = p.block_prefix[p.n_dirs];
  const int threads = p.split * kWave;
  const size_t lds = split_lds_bytes(p.L, R, p.split, TRAIN);
  const int mode = jacobi ? (p.u_fused ? 2 : 1) : 0;
  if (mode == 2)
    sweep_fwd_split_kernel<R, VEC, MASK, TRAIN, 2><<<blocks, threads, lds, st>>>(p);
  else if (mode == 1)
    sweep_fwd_split_kernel<R, VEC, MASK, TRAIN, 1><<<blocks, threads, lds, st>>>(p);
  else
    sweep_fwd_split_kernel<R, VEC, MASK, TRAIN, 0><<<blocks, threads, lds, st>>>(p);
}

template <int R, bool VEC, bool MASK, bool TRAIN>
void launch_vm(const SweepParams& p, bool jacobi, hipStream_t st) {
  if constexpr (R > 1) {
    if (p.split >= 2 && !p.ctx2d) {
      launch_vm_split<R, VEC, MASK, TRAIN>(p, jacobi, st);
      return;
    }
  }
  const int blocks = p.block_prefix[p.n_dirs];
  const size_t lds = fwd_lds_bytes(p.L, p.ctx2d);
  const int mode = jacobi ? (p.u_fused ? 2 : 1) : 0;
  if constexpr (!MASK && (!TRAIN || R <= 2)) {
    if (jacobi && store_through(p)) {
      if (mode == 2)
        sweep_fwd_kernel<R, VEC, MASK, TRAIN, 2, true><<<blocks, kWave, lds, st>>>(p);
      else
        sweep_fwd_kernel<R, VEC, MASK, TRAIN, 1, true><<<blocks, kWave, lds, st>>>(p);
      return;
    }
  }
  if (mode == 2)
    sweep_fwd_kernel<R, VEC, MASK, TRAIN, 2><<<blocks, kWave, lds, st>>>(p);
  else if (mode == 1)
    sweep_fwd_kernel<R, VEC, MASK, TRAIN, 1><<<blocks, kWave, lds, st>>>(p);
  else
    sweep_fwd_kernel<R, VEC, MASK, TRAIN, 0><<<blocks, kWave, lds, st>>>(p);
}

}  // namespace

// (the scans that keep argmin labels and those that do not are compiled as separate units)
template <int R, bool TRAIN>
void launch_sweep_fwd_t(const SweepParams& p, bool jacobi, hipStream_t st) {
  if (p.block_prefix[p.n_dirs] <= 0) return;
  const bool mask = p.L != R * kWave;
  // one descriptor per plane for the whole kernel: whole lanes of labels, and, where some lanes have
  // none, an image of at most 2 GiB (run_chain_fwd, foff_ok)
  const bool vec = (p.L % R) == 0 &&
                   (!mask || (int64_t)p.H * p.W * p.L * 4 <= (int64_t)1 << 31);
  if constexpr (R > 1) {
    if (!vec) {
      launch_vm<R, false, true, TRAIN>(p, jacobi, st);
      return;
    }
  }
  if (mask)
    launch_vm<R, true, true, TRAIN>(p, jacobi, st);
  else
    launch_vm<R, true, false, TRAIN>(p, jacobi, st);
}

template void launch_sweep_fwd_t<MPL_INST_R, (MPL_INST_TRAIN != 0)>(const SweepParams&, bool, hipStream_t);

}  // namespace mpl
