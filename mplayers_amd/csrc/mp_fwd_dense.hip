// Forward scan of TRWP for tables declared dense (learned ones: every pair of labels counts) with four
// wavefronts per chain, in launches of few chains.  The recurrence and what each plane holds: mp_fwd.hip;
// the results are the same bits, but for a linear table of 65 labels or more, which takes the scan over all pairs
// of labels here and the minima from both sides there: they agree to the parity tolerance.
//
// Such a launch is bound by the scan over all pairs of labels of one pixel, so the front labels are split
// over the wavefronts: each holds the chain's state, takes the minimum over its quarter, and the four partial
// minima meet in LDS, with their least entries (one barrier per pixel).  Next to sweep_fwd_split_kernel, which does
// the same,
//   * the table entries a lane needs for its wavefront's front labels stay in registers for the whole chain
//     (they differ between lanes, but not between pixels), so a front label costs a multiply-add and half a
//     minimum per label, and of LDS only its belief, four to a broadcast read;
//   * nothing but the recurrence is the scanners' work.  Loads, the update of the unary terms, argmin labels and
//     stores are four more wavefronts', one beside each scanner on its SIMD, a pixel of every block of four each:
//     while a block is scanned they finish the one before and prepare the one after it.  They issue where the
//     scanners wait for LDS and for each other, some half of the time.
// Measured, argmin labels kept / not, rows of 257 on 256 chains, ns per pixel, every wavefront serving two pixels of a
// block it has scanned -> this: 64 labels 443 / 385 -> 323 / 312, 96 labels 697 / 608 -> 453 / 445, 128 labels 811 / 652 ->
// 522 / 509; 192 labels, rows of 129, 1290 / 973 -> 891 / 845.  A third of that is that what follows the barrier reads
// everything it needs before it waits for any of it.
// The argmin labels take two steps, as in dense1d_step: the scan notes the trip (eight front labels) whose
// candidates last reached the running minimum; the servers evaluate that one trip again.
//
// With one label per lane (17 to 64 labels), where the scans of mp_fwd_team.hip take a third to half of this one's
// time for a band or a truncated linear table, the declaration alone does not decide: both kernels are
// launched, and the one whose kind of table it is not ends at once (is_dense).
//
// Compiled once per R (labels per lane, 1 to 3) with -DMPL_INST_R=<R>.

#include <type_traits>

#include "mp_fwd_step.h"

namespace mpl {
namespace {

constexpr int kWaves = 4;              // that scan; as many serve, one of either on every SIMD of the unit
constexpr int kTeam = 2 * kWaves * kWave;
constexpr int kBlock = kWaves;         // pixels of a block, one to a server
constexpr int kTrip = 8;               // front labels

template <int R>
struct alignas(16) Set {
  float in[kBlock][kWave][R == 1 ? 2 : 4];            // U, edge weight
  float part[kBlock][kWaves][kWave][R == 1 ? 2 : 4];  // partial minima, the trips they were found in (a byte each)
  float a[kBlock][kWave * R];                         // beliefs the pixel's message comes from (scanner 0)
  float pmin[kBlock][kWaves];                         // minima over the labels of the partial minima
};
template <int R>
struct alignas(16) Slots {
  Set<R> set[2];                    // by the parity of the block
  float copy[kWaves][kWave * R];    // each scanner's own copy of the beliefs
};

// workgroup barrier over LDS contents only: global loads in flight stay in flight
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// R words and one more, of a lane's slot
template <int R>
__device__ __forceinline__ void get_slot(const float* src, float (&x)[R], float& extra) {
  if constexpr (R == 1) {
    const f32x2 v = *reinterpret_cast<const f32x2*>(src);
    x[0] = v[0];
    extra = v[1];
  } else {
    const f32x4 v = *reinterpret_cast<const f32x4*>(src);
#pragma unroll
    for (int j = 0; j < R; ++j) x[j] = v[j];
    extra = v[R];
  }
}
template <int R>
__device__ __forceinline__ void put_slot(float* dst, const float (&x)[R], float extra) {
  if constexpr (R == 1)
    *reinterpret_cast<f32x2*>(dst) = f32x2{x[0], extra};
  else if constexpr (R == 2)
    *reinterpret_cast<f32x4*>(dst) = f32x4{x[0], x[1], extra, 0.f};
  else
    *reinterpret_cast<f32x4*>(dst) = f32x4{x[0], x[1], x[2], extra};
}

// its R words alone (read together, the extra ones would be reads into registers that the next read wants)
template <int R>
__device__ __forceinline__ void get_words(const float* src, float (&x)[R]) {
  if constexpr (R == 1) {
    x[0] = *src;
  } else if constexpr (R == 2) {
    const f32x2 v = *reinterpret_cast<const f32x2*>(src);
    x[0] = v[0];
    x[1] = v[1];
  } else {
    const f32x4 v = *reinterpret_cast<const f32x4*>(src);
#pragma unroll
    for (int j = 0; j < R; ++j) x[j] = v[j];
  }
}

// +inf that the compiler cannot see through: what starts from it is +inf where no candidate is a number (a candidate
// that is none drops out of a minimum; left to itself the compiler leaves out a minimum with +inf), so a share without
// a number says nothing about the labels or their least one.  Argmin labels kept, rows of 257 on 256 chains, with what
// finds the labels of such pixels, over neither: 17 to 64 labels 1.01 to 1.025, 96 and 128 labels 1.00 to 1.01, 192 labels 1.00.
__device__ __forceinline__ float opaque_inf() {
  float x = INFINITY;
  asm volatile("" : "+s"(x));
  return x;
}

constexpr int kNoLabel = kMaxL;
// the candidates of label l in the trip from front label f0 on (the same multiply-adds on the same operands as in the
// scan: the same bits)
template <int R>
__device__ __forceinline__ void trip_candidates(const float* a, const float* csym_s, const float w, const int f0, const int l,
                                                float (&val)[kTrip]) {
  const f32x4 a0 = *reinterpret_cast<const f32x4*>(a + f0);
  const f32x4 a1 = *reinterpret_cast<const f32x4*>(a + f0 + 4);
  const float* cp = csym_s + (dense_sym_centre<R>() + l - f0 - (kTrip - 1));  // entry of front label f0 + kTrip - 1
#pragma unroll
  for (int u = 0; u < kTrip; ++u) val[u] = fmaf(w, cp[kTrip - 1 - u], u < 4 ? a0[u & 3] : a1[u & 3]);
}
// the largest front label of them whose candidate is the minimum v; kNoLabel or more: none
__device__ __forceinline__ int trip_label(const float (&val)[kTrip], const float v, const int f0) {
  int arg = kNoLabel;
#pragma unroll
  for (int u = 0; u < kTrip; ++u) arg = equal(val[u], v) ? u : arg;
  return f0 + arg;
}
// The labels that trip_label has not found: of a minimum of +inf, which a share without a number reaches too and whose
// trip it then is.  All front labels are looked at, and the last one is taken where no candidate is a number, as in
// the other scans.  stored: uniform; the labels are kept (a chain start's beliefs are zero, also past the last label, and
// its trips end there).
template <int R>
__device__ __forceinline__ void labels_without_trip(const float* a, const float* csym_s, const float w, const float (&v)[R],
                                                    const bool stored, const int lab0, const int L, int (&fd_idx)[R]) {
  bool none[R], any = false;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    none[j] = fd_idx[j] >= L;
    any |= none[j];
    fd_idx[j] = min(fd_idx[j], L - 1);
  }
  if (__builtin_expect(!stored || ballot(any) == 0, 1)) return;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const float* cp = csym_s + (dense_sym_centre<R>() + lab0 + j);
#pragma clang loop unroll(disable)
    for (int fd = 0; fd < L; ++fd) {
      const bool is_min = equal(fmaf(w, cp[-fd], a[fd]), v[j]);
      fd_idx[j] = none[j] && is_min ? fd : fd_idx[j];
    }
  }
}

// NT: trips per wavefront
template <int R, bool TRAIN, int NT>
__device__ __forceinline__ void walk_chain(const SweepParams& p, const ChainCtx& ch0, const bool msg_zero,
                                           Slots<R>& s, const float* csym_s) {
  constexpr int kShare = NT * kTrip;  // front labels per wavefront
  constexpr int kAhead = 2;           // blocks of pixels whose loads are in flight
  const int L = p.L;
  const int lane = threadIdx.x & (kWave - 1);
  const int role = uniform_i((int)threadIdx.x / kWave);
  const bool serves = role >= kWaves;
  const int wave = role & (kWaves - 1);
  const int lab0 = R * lane;
  const bool whole = L % R == 0;      // every lane's labels exist or none does
  const int n = ch0.n;
  const float rho = p.rho;
  const int64_t HW = (int64_t)p.H * p.W;
  const int64_t P = (int64_t)p.B * HW;
  const int64_t N = P * L;
  const int blocks = (n + kBlock - 1) / kBlock;
  const int fd_lo = wave * kShare;
  const float inf = opaque_inf();

  float floor_l[R];
#pragma unroll
  for (int j = 0; j < R; ++j) floor_l[j] = lab0 + j < L ? -INFINITY : INFINITY;
  auto norm_min = [&](const float (&v)[R]) __attribute__((always_inline)) {
    float vm = INFINITY;
#pragma unroll
    for (int j = 0; j < R; ++j) vm = fminf(vm, fmaxf(v[j], floor_l[j]));
    return wave_min_fast(vm);
  };

  // the minimum over all labels, from the scanners' own
  auto joint_min = [&](const Set<R>& st, const int i) __attribute__((always_inline)) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(st.pmin[i]);
    return fminf(fminf(x[0], x[1]), fminf(x[2], x[3]));
  };

  // The scan of a block's pixels.  tab: c[|label - front label|] of this wavefront's front labels; prev, uf: message
  // and U of the front pixel.
  auto fill_tab = [&](float (&tab)[kShare][R]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kShare; ++u)
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int d = lab0 + j - (fd_lo + u);
        tab[u][j] = csym_s[dense_sym_centre<R>() + (d < -R * kWave ? -R * kWave : d)];
        asm volatile("" : "+v"(tab[u][j]));  // (not to be read again for every pixel)
      }
  };
  auto scan_block = [&](Set<R>& st, const bool first, const float (&tab)[kShare][R], float (&prev)[R], float (&uf)[R])
      __attribute__((always_inline)) {
    float un[R], w;
    get_slot<R>(st.in[0][lane], un, w);
#pragma unroll
    for (int i = 0; i < kBlock; ++i) {
      // (the first wavefront's copy is the one the service reads)
      float* const mine = wave == 0 ? st.a[i] : s.copy[wave];
#pragma unroll
      for (int j = 0; j < R; ++j) mine[lab0 + j] = fmaf(rho, prev[j], uf[j]);
      lds_order();
      float v[R];
      int trip[R];
#pragma unroll
      for (int j = 0; j < R; ++j) {
        v[j] = inf;
        trip[j] = wave * NT;
      }
      f32x4 x[2 * NT];
#pragma unroll
      for (int k = 0; k < 2 * NT; ++k) x[k] = *reinterpret_cast<const f32x4*>(&mine[fd_lo + 4 * k]);
      __builtin_amdgcn_sched_barrier(0);  // (all of them on their way before the first is waited for)
#pragma unroll
      for (int k = 0; k < NT; ++k) {
        const f32x4 x0 = x[2 * k], x1 = x[2 * k + 1];
#pragma unroll
        for (int j = 0; j < R; ++j) {
          float c[kTrip];
#pragma unroll
          for (int u = 0; u < kTrip; ++u) c[u] = fmaf(w, tab[k * kTrip + u][j], u < 4 ? x0[u & 3] : x1[u & 3]);
          if constexpr (TRAIN) {
            const float lm = fminf(fminf(fminf(fminf(fminf(c[0], c[1]), c[2]), fminf(fminf(c[3], c[4]), c[5])), c[6]), c[7]);
            if (k > 0) trip[j] = at_most(lm, v[j]) ? wave * NT + k : trip[j];
            v[j] = fminf(lm, v[j]);
          } else {
#pragma unroll
            for (int u = 0; u < kTrip; u += 2) v[j] = fminf(fminf(v[j], c[u]), c[u + 1]);
          }
        }
      }
      int trips = 0;
      if (TRAIN) {
#pragma unroll
        for (int j = 0; j < R; ++j) trips |= trip[j] << (8 * j);
      }
      put_slot<R>(st.part[i][wave][lane], v, __builtin_bit_cast(float, trips));
      const float pm = norm_min(v);
      if (lane == 0) st.pmin[i][wave] = pm;
#pragma unroll
      for (int j = 0; j < R; ++j) uf[j] = un[j];
      if (i + 1 < kBlock) get_slot<R>(st.in[i + 1][lane], un, w);
      lds_barrier();
      float pv[kWaves - 1][R];
#pragma unroll
      for (int k = 1; k < kWaves; ++k) get_words<R>(st.part[i][(wave + k) & 3][lane], pv[k - 1]);
      const float nmin = joint_min(st, i);
#pragma unroll
      for (int k = 1; k < kWaves; ++k)
#pragma unroll
        for (int j = 0; j < R; ++j) v[j] = fminf(v[j], pv[k - 1][j]);
      const bool start = first && i == 0;
#pragma unroll
      for (int j = 0; j < R; ++j) prev[j] = start ? 0.f : v[j] - nmin;  // (the chain start has no front pixel)
    }
  };

  // even_walk: a constant; the first (even direction) or the second sweep of a pair (run_chain_fwd)
  auto serve = [&](const ChainCtx& ch, const bool skip_s_in, const auto even_walk) __attribute__((always_inline)) {
    constexpr bool EVEN = decltype(even_walk)::value;
    const int dir = ch.dir;
    const int64_t img_p = (int64_t)ch.bv * HW;
    const int64_t img_e = img_p * L;
    const bool zfirst = p.zero_first && msg_zero;
    const bool skip_s = skip_s_in || (EVEN && zfirst);
    const bool md_zero = p.first_iter && msg_zero;
    const bool mi_zero = md_zero && EVEN;
    const int img_bytes = (int)(unsigned)(HW * L * 4);
    const int img_bytes_p = (int)(HW * 4 > 0x7fffffff ? 0x7fffffff : HW * 4);
    const rsrc_t rS = make_rsrc((zfirst ? p.belief_zero : p.belief) + img_e, img_bytes);
    const rsrc_t rMd = make_rsrc(p.msg_in + (int64_t)dir * N + img_e, md_zero ? 0 : img_bytes);
    const rsrc_t rMi = make_rsrc(p.msg_in + (int64_t)(dir ^ 1) * N + img_e, mi_zero ? 0 : img_bytes);
    const rsrc_t rMo = make_rsrc(p.msg_out + (int64_t)dir * N + img_e, img_bytes);
    const rsrc_t rSo = make_rsrc(p.belief_out + img_e, skip_s ? 0 : img_bytes);
    const rsrc_t rImin = make_rsrc(TRAIN ? p.idx_min + (int64_t)dir * N + img_e : nullptr, TRAIN ? (int)(HW * L) : 0);
    const rsrc_t dInorm = make_rsrc(TRAIN ? p.idx_norm + (int64_t)dir * P + img_p : nullptr, TRAIN ? (int)HW : 0);
    const rsrc_t dW = make_rsrc(p.edge + (int64_t)dir * P + img_p, img_bytes_p);

    auto pixel_at = [&](const int t) __attribute__((always_inline)) { return (unsigned)(ch.pix0 + t * ch.pstep); };
    auto label_off = [&](bool on, unsigned so, int j) __attribute__((always_inline)) {
      return (int)((on && lab0 + j < L) ? so + (unsigned)(lab0 + j) * 4u : kDeadWide);
    };
    // (one access per lane whatever the label count: of a lane with labels and places past the last one, the
    // places read another pixel's or, past the plane, zero)
    auto load_plane = [&](rsrc_t r, bool on, unsigned so, float (&x)[R]) __attribute__((always_inline)) {
      buf_load<R, true, load_policy(false)>(r, label_off(on, so, 0), 0u, x);
    };
    auto store_plane = [&](rsrc_t r, bool on, unsigned so, const float (&x)[R]) __attribute__((always_inline)) {
      if (R == 1 || whole) {
        buf_store<R, true>(r, label_off(on, so, 0), 0u, x);
      } else {
#pragma unroll
        for (int j = 0; j < R; ++j)
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x[j]), r, label_off(on, so, j), 0, MPL_ST_AUX);
      }
    };
    struct Pix {
      float s[R], md[R], mi[R], w;
    };
    // the loads of chain position t (nothing is read past the end of the chain)
    auto load_pix = [&](const int t) __attribute__((always_inline)) {
      Pix r;
      const bool on = t < n;
      const unsigned pp = pixel_at(t);
      const unsigned so = pp * (unsigned)L * 4u;
      load_plane(rS, on, so, r.s);
      if (EVEN) load_plane(rMd, on, so, r.md);
      load_plane(rMi, on, so, r.mi);
      r.w = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(dW, on ? (int)(pp * 4u) : kDeadOffset, 0, 0));
      return r;
    };
    float tt[2][R];  // of this server's pixels of the blocks in the sets
    const int i = wave;
    auto prepare = [&](const Pix& px, const int t, Set<R>& st, float (&tk)[R]) __attribute__((always_inline)) {
      float un[R], q[R];
#pragma unroll
      for (int j = 0; j < R; ++j) {
        tk[j] = EVEN ? px.s[j] - px.md[j] : px.s[j] + px.mi[j];
        // UpdateUnaryKernel, TRWP_forward.cu:70-78 (no maximum with the floor, which is -inf where a term is no number)
        un[j] = lab0 + j < L ? fmaf(tk[j], rho, -px.mi[j]) : INFINITY;
        q[j] = tk[j] - px.mi[j];
      }
      put_slot<R>(st.in[i][lane], un, px.w);
      // Q of the pixel is known already, whatever its message
      if (EVEN) store_plane(rSo, t < n, pixel_at(t) * (unsigned)L * 4u, q);
    };
    float md0[R];  // second sweep: the old message of the chain start (wavefront 0)
    if (!EVEN) load_plane(rMd, wave == 0, pixel_at(0) * (unsigned)L * 4u, md0);

    // what is left of a pixel of the block that has been scanned
    auto finish = [&](const int t, const Set<R>& st, const float (&tk)[R], const auto& pause) __attribute__((always_inline)) {
      const bool on = t < n;
      const unsigned pp = pixel_at(t);
      const unsigned so = pp * (unsigned)L * 4u;
      float v[R], m[R];
      int trips = 0;
#pragma unroll
      for (int k = 0; k < kWaves; ++k) {
        float pv[R], pt;
        get_slot<R>(st.part[i][k][lane], pv, pt);
        const int theirs = __builtin_bit_cast(int, pt);
#pragma unroll
        for (int j = 0; j < R; ++j) {
          const bool take = k == 0 || pv[j] <= v[j];  // (the later share wins ties)
          v[j] = take ? pv[j] : v[j];
          const int byte = 0xff << (8 * j);
          if (TRAIN) trips = take ? (trips & ~byte) | (theirs & byte) : trips;
        }
      }
      const float nmin = joint_min(st, i);
#pragma unroll
      for (int j = 0; j < R; ++j) m[j] = t == 0 ? 0.f : v[j] - nmin;
      if constexpr (TRAIN) {
        float un[R], w;
        get_slot<R>(st.in[i][lane], un, w);
        int fd_idx[R], f0[R];
        bool pr[R];
        float val[R][kTrip];
#pragma unroll
        for (int j = 0; j < R; ++j) {
          f0[j] = ((trips >> (8 * j)) & 0xff) * kTrip;
          trip_candidates<R>(st.a[i], csym_s, w, f0[j], lab0 + j, val[j]);
        }
        pause();
#pragma unroll
        for (int j = 0; j < R; ++j) {
          fd_idx[j] = trip_label(val[j], v[j], f0[j]);
          pr[j] = lab0 + j < L && v[j] == nmin;
        }
        const bool idx_on = on && t > 0;
        labels_without_trip<R>(st.a[i], csym_s, w, v, idx_on, lab0, L, fd_idx);
        const int nidx = last_label<R>(pr, L - 1);
        const unsigned sob = pp * (unsigned)L;
        if (R == 1 || whole) {
          buf_store_u8<R, true>(rImin, (int)((idx_on && lab0 < L) ? sob + (unsigned)lab0 : kDeadWide), 0u, fd_idx);
        } else {
#pragma unroll
          for (int j = 0; j < R; ++j)
            __builtin_amdgcn_raw_buffer_store_b8((unsigned char)fd_idx[j], rImin,
                                                 (int)((idx_on && lab0 + j < L) ? sob + (unsigned)(lab0 + j) : kDeadWide), 0, MPL_ST_AUX);
        }
        // every lane stores the same byte to the same address
        __builtin_amdgcn_raw_buffer_store_b8((unsigned char)nidx, dInorm, idx_on ? (int)pp : kDeadOffset, 0, 0);
      } else {
        pause();
      }
      pause();
      // (the reference never writes the chain start)
      store_plane(rMo, on && (t > 0 || p.zero_start), so, m);
      if constexpr (!EVEN) {
        float sn[R];
#pragma unroll
        for (int j = 0; j < R; ++j) sn[j] = tk[j] + (t == 0 ? md0[j] : m[j]);
        store_plane(rSo, on, so, sn);
      }
    };

    Pix ring[kAhead];
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
      ring[q] = load_pix(q * kBlock + i);
      MPL_ORDER_LOADS();
    }
    prepare(ring[0], i, s.set[0], tt[0]);
    ring[0] = load_pix(kAhead * kBlock + i);
    lds_barrier();
    // Period b, a barrier per pixel of block b, which the scanners walk: the server finishes its pixel of block
    // b - 1, prepares that of block b + 1 in the same set and loads that of block b + 3, in four parts
#pragma clang loop unroll(disable)
    for (int b0 = 0; b0 <= blocks; b0 += 2) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int b = b0 + q;
        Set<R>& st = s.set[(q + 1) & 1];
        auto pause = [&]() __attribute__((always_inline)) {
          if (b < blocks) lds_barrier();
        };
        if (b > 0 && b <= blocks) finish((b - 1) * kBlock + i, st, tt[(q + 1) & 1], pause);
        else if (b == 0) {
          pause();
          pause();
        }
        lds_order();
        if (b < blocks) {
          prepare(ring[(q + 1) % kAhead], (b + 1) * kBlock + i, st, tt[(q + 1) & 1]);
          lds_barrier();
          ring[(q + 1) % kAhead] = load_pix((b + 1 + kAhead) * kBlock + i);
          lds_barrier();
        }
      }
    }
  };

  if (!serves) {
    __builtin_amdgcn_s_setprio(3);
    float tab[kShare][R];
    fill_tab(tab);
    const int walks = !(ch0.dir & 1) && p.fused_pair ? 2 : 1;
#pragma clang loop unroll(disable)
    for (int k = 0; k < walks; ++k) {
      if (k > 0) __syncthreads();
      float prev[R], uf[R];
#pragma unroll
      for (int j = 0; j < R; ++j) prev[j] = uf[j] = 0.f;
      lds_barrier();  // block 0 is prepared
#pragma clang loop unroll(disable)
      for (int b = 0; b < blocks; ++b) scan_block(s.set[b & 1], b == 0, tab, prev, uf);
    }
    return;
  }
  if (!(ch0.dir & 1)) serve(ch0, p.skip_s_store != 0, std::true_type());
  if ((ch0.dir & 1) || p.fused_pair) {
    ChainCtx ch = ch0;
    bool skip_s = p.skip_s_store != 0;
    if (!(ch0.dir & 1)) {
      // the second sweep of a pair reads what the first one stored: on the same compute unit, once the
      // stores are complete
      ch.dir = ch0.dir ^ 1;
      ch.pix0 = ch0.pix0 + (n - 1) * ch0.pstep;
      ch.pstep = -ch0.pstep;
      skip_s = p.skip_s_store2 != 0;
      wait_vmem<0>();
      __syncthreads();
    }
    serve(ch, skip_s, std::false_type());
  }
}

// ---- the scan without servers ------------------------------------------------------------------------
// The four wavefronts serve two pixels each of every block they have scanned (launch).
constexpr int kTeamAlone = kWaves * kWave;
constexpr int kPer = 2;                // pixels of a block that a wavefront serves
constexpr int kBlockAlone = kWaves * kPer;

template <int R>
struct alignas(16) SlotsAlone {
  float in[kBlockAlone][kWave][R == 1 ? 2 : 4];            // U, edge weight
  float part[kBlockAlone][kWaves][kWave][R == 1 ? 2 : 4];  // partial minima, the trips they were found in (a byte each)
  float a[kBlockAlone][kWave * R];                         // beliefs the pixel's message comes from (wavefront 0)
  float copy[kWaves][kWave * R];                      // each wavefront's own copy of them
};

template <int R, bool TRAIN, int NT>
__device__ __forceinline__ void walk_chain_alone(const SweepParams& p, const ChainCtx& ch0, const bool msg_zero,
                                           SlotsAlone<R>& s, const float* csym_s) {
  constexpr int kShare = NT * kTrip;  // front labels per wavefront
  const int L = p.L;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = uniform_i((int)threadIdx.x / kWave);
  const int lab0 = R * lane;
  const bool whole = L % R == 0;      // every lane's labels exist or none does
  const int n = ch0.n;
  const float rho = p.rho;
  const int64_t HW = (int64_t)p.H * p.W;
  const int64_t P = (int64_t)p.B * HW;
  const int64_t N = P * L;
  const int blocks = (n + kBlockAlone - 1) / kBlockAlone;
  const int fd_lo = wave * kShare;
  const float inf = opaque_inf();

  float floor_l[R];
#pragma unroll
  for (int j = 0; j < R; ++j) floor_l[j] = lab0 + j < L ? -INFINITY : INFINITY;
  float tab[kShare][R];  // c[|label - front label|]
#pragma unroll
  for (int u = 0; u < kShare; ++u)
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int d = lab0 + j - (fd_lo + u);
      tab[u][j] = csym_s[dense_sym_centre<R>() + (d < -R * kWave ? -R * kWave : d)];
    }
  auto norm_min = [&](const float (&v)[R]) __attribute__((always_inline)) {
    float vm = INFINITY;
#pragma unroll
    for (int j = 0; j < R; ++j) vm = fminf(vm, fmaxf(v[j], floor_l[j]));
    return wave_min_fast(vm);
  };

  // even_walk: a constant; the first (even direction) or the second sweep of a pair (run_chain_fwd)
  auto walk = [&](const ChainCtx& ch, const bool skip_s_in, const auto even_walk) __attribute__((always_inline)) {
    constexpr bool EVEN = decltype(even_walk)::value;
    const int dir = ch.dir;
    const int64_t img_p = (int64_t)ch.bv * HW;
    const int64_t img_e = img_p * L;
    const bool zfirst = p.zero_first && msg_zero;
    const bool skip_s = skip_s_in || (EVEN && zfirst);
    const bool md_zero = p.first_iter && msg_zero;
    const bool mi_zero = md_zero && EVEN;
    const int img_bytes = (int)(unsigned)(HW * L * 4);
    const int img_bytes_p = (int)(HW * 4 > 0x7fffffff ? 0x7fffffff : HW * 4);
    const rsrc_t rS = make_rsrc((zfirst ? p.belief_zero : p.belief) + img_e, img_bytes);
    const rsrc_t rMd = make_rsrc(p.msg_in + (int64_t)dir * N + img_e, md_zero ? 0 : img_bytes);
    const rsrc_t rMi = make_rsrc(p.msg_in + (int64_t)(dir ^ 1) * N + img_e, mi_zero ? 0 : img_bytes);
    const rsrc_t rMo = make_rsrc(p.msg_out + (int64_t)dir * N + img_e, img_bytes);
    const rsrc_t rSo = make_rsrc(p.belief_out + img_e, skip_s ? 0 : img_bytes);
    const rsrc_t rImin = make_rsrc(TRAIN ? p.idx_min + (int64_t)dir * N + img_e : nullptr, TRAIN ? (int)(HW * L) : 0);
    const rsrc_t dInorm = make_rsrc(TRAIN ? p.idx_norm + (int64_t)dir * P + img_p : nullptr, TRAIN ? (int)HW : 0);
    const rsrc_t dW = make_rsrc(p.edge + (int64_t)dir * P + img_p, img_bytes_p);

    auto pixel_at = [&](const int t) __attribute__((always_inline)) { return (unsigned)(ch.pix0 + t * ch.pstep); };
    auto label_off = [&](bool on, unsigned so, int j) __attribute__((always_inline)) {
      return (int)((on && lab0 + j < L) ? so + (unsigned)(lab0 + j) * 4u : kDeadWide);
    };
    // (one access per lane whatever the label count: of a lane with labels and places past the last one, the
    // places read another pixel's or, past the plane, zero)
    auto load_plane = [&](rsrc_t r, bool on, unsigned so, float (&x)[R]) __attribute__((always_inline)) {
      buf_load<R, true, load_policy(false)>(r, label_off(on, so, 0), 0u, x);
    };
    auto store_plane = [&](rsrc_t r, bool on, unsigned so, const float (&x)[R]) __attribute__((always_inline)) {
      if (R == 1 || whole) {
        buf_store<R, true>(r, label_off(on, so, 0), 0u, x);
      } else {
#pragma unroll
        for (int j = 0; j < R; ++j)
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x[j]), r, label_off(on, so, j), 0, MPL_ST_AUX);
      }
    };
    struct Pix {
      float s[R], md[R], mi[R], w;
    };
    // the loads of chain position t (nothing is read past the end of the chain)
    auto load_pix = [&](const int t) __attribute__((always_inline)) {
      Pix r;
      const bool on = t < n;
      const unsigned pp = pixel_at(t);
      const unsigned so = pp * (unsigned)L * 4u;
      load_plane(rS, on, so, r.s);
      if (EVEN) load_plane(rMd, on, so, r.md);
      load_plane(rMi, on, so, r.mi);
      r.w = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(dW, on ? (int)(pp * 4u) : kDeadOffset, 0, 0));
      return r;
    };
    float tt[kPer][R];  // of this wavefront's pixels of the block that is being scanned
    auto prepare = [&](const Pix& px, const int t, const int i, float (&tk)[R]) __attribute__((always_inline)) {
      float un[R], q[R];
#pragma unroll
      for (int j = 0; j < R; ++j) {
        tk[j] = EVEN ? px.s[j] - px.md[j] : px.s[j] + px.mi[j];
        // UpdateUnaryKernel, TRWP_forward.cu:70-78 (no maximum with the floor, which is -inf where a term is no number)
        un[j] = lab0 + j < L ? fmaf(tk[j], rho, -px.mi[j]) : INFINITY;
        q[j] = tk[j] - px.mi[j];
      }
      put_slot<R>(s.in[i][lane], un, px.w);
      // Q of the pixel is known already, whatever its message
      if (EVEN) store_plane(rSo, t < n, pixel_at(t) * (unsigned)L * 4u, q);
    };
    float md0[R];  // second sweep: the old message of the chain start (wavefront 0)
    if (!EVEN) load_plane(rMd, wave == 0, pixel_at(0) * (unsigned)L * 4u, md0);

    // what is left of a pixel of the block that has been scanned
    auto finish = [&](const int t, const int i, const float (&tk)[R]) __attribute__((always_inline)) {
      const bool on = t < n;
      const unsigned pp = pixel_at(t);
      const unsigned so = pp * (unsigned)L * 4u;
      float v[R], m[R];
      int trips = 0;
#pragma unroll
      for (int k = 0; k < kWaves; ++k) {
        float pv[R], pt;
        get_slot<R>(s.part[i][k][lane], pv, pt);
        const int theirs = __builtin_bit_cast(int, pt);
#pragma unroll
        for (int j = 0; j < R; ++j) {
          const bool take = k == 0 || pv[j] <= v[j];  // (the later share wins ties)
          v[j] = take ? pv[j] : v[j];
          const int byte = 0xff << (8 * j);
          if (TRAIN) trips = take ? (trips & ~byte) | (theirs & byte) : trips;
        }
      }
      const float nmin = norm_min(v);
#pragma unroll
      for (int j = 0; j < R; ++j) m[j] = t == 0 ? 0.f : v[j] - nmin;
      if constexpr (TRAIN) {
        float un[R], w;
        get_slot<R>(s.in[i][lane], un, w);
        int fd_idx[R];
        bool pr[R];
#pragma unroll
        for (int j = 0; j < R; ++j) {
          const int f0 = ((trips >> (8 * j)) & 0xff) * kTrip;
          float val[kTrip];
          trip_candidates<R>(s.a[i], csym_s, w, f0, lab0 + j, val);
          fd_idx[j] = trip_label(val, v[j], f0);
          pr[j] = lab0 + j < L && v[j] == nmin;
        }
        const bool idx_on = on && t > 0;
        labels_without_trip<R>(s.a[i], csym_s, w, v, idx_on, lab0, L, fd_idx);
        const int nidx = last_label<R>(pr, L - 1);
        const unsigned sob = pp * (unsigned)L;
        if (R == 1 || whole) {
          buf_store_u8<R, true>(rImin, (int)((idx_on && lab0 < L) ? sob + (unsigned)lab0 : kDeadWide), 0u, fd_idx);
        } else {
#pragma unroll
          for (int j = 0; j < R; ++j)
            __builtin_amdgcn_raw_buffer_store_b8((unsigned char)fd_idx[j], rImin,
                                                 (int)((idx_on && lab0 + j < L) ? sob + (unsigned)(lab0 + j) : kDeadWide), 0, MPL_ST_AUX);
        }
        // every lane stores the same byte to the same address
        __builtin_amdgcn_raw_buffer_store_b8((unsigned char)nidx, dInorm, idx_on ? (int)pp : kDeadOffset, 0, 0);
      }
      // (the reference never writes the chain start)
      store_plane(rMo, on && (t > 0 || p.zero_start), so, m);
      if constexpr (!EVEN) {
        float sn[R];
#pragma unroll
        for (int j = 0; j < R; ++j) sn[j] = tk[j] + (t == 0 ? md0[j] : m[j]);
        store_plane(rSo, on, so, sn);
      }
    };

    float prev[R], uf[R];
#pragma unroll
    for (int j = 0; j < R; ++j) prev[j] = uf[j] = 0.f;
    auto scan = [&](const int i, const float w, const bool start) __attribute__((always_inline)) {
      // (the first wavefront's copy is the one the service reads)
      float* const mine = wave == 0 ? s.a[i] : s.copy[wave];
#pragma unroll
      for (int j = 0; j < R; ++j) mine[lab0 + j] = fmaf(rho, prev[j], uf[j]);
      lds_order();
      float v[R];
      int trip[R];
#pragma unroll
      for (int j = 0; j < R; ++j) {
        v[j] = inf;
        trip[j] = wave * NT;
      }
#pragma unroll
      for (int k = 0; k < NT; ++k) {
        const f32x4 x0 = *reinterpret_cast<const f32x4*>(&mine[fd_lo + k * kTrip]);
        const f32x4 x1 = *reinterpret_cast<const f32x4*>(&mine[fd_lo + k * kTrip + 4]);
#pragma unroll
        for (int j = 0; j < R; ++j) {
          float c[kTrip];
#pragma unroll
          for (int u = 0; u < kTrip; ++u) c[u] = fmaf(w, tab[k * kTrip + u][j], u < 4 ? x0[u & 3] : x1[u & 3]);
          if constexpr (TRAIN) {
            const float lm = fminf(fminf(fminf(fminf(fminf(c[0], c[1]), c[2]), fminf(fminf(c[3], c[4]), c[5])), c[6]), c[7]);
            if (k > 0) trip[j] = at_most(lm, v[j]) ? wave * NT + k : trip[j];
            v[j] = fminf(lm, v[j]);
          } else {
#pragma unroll
            for (int u = 0; u < kTrip; u += 2) v[j] = fminf(fminf(v[j], c[u]), c[u + 1]);
          }
        }
      }
      int trips = 0;
      if (TRAIN) {
#pragma unroll
        for (int j = 0; j < R; ++j) trips |= trip[j] << (8 * j);
      }
      put_slot<R>(s.part[i][wave][lane], v, __builtin_bit_cast(float, trips));
      lds_barrier();
      float pv[kWaves - 1][R];
#pragma unroll
      for (int k = 1; k < kWaves; ++k) get_words<R>(s.part[i][(wave + k) & 3][lane], pv[k - 1]);
#pragma unroll
      for (int k = 1; k < kWaves; ++k)
#pragma unroll
        for (int j = 0; j < R; ++j) v[j] = fminf(v[j], pv[k - 1][j]);
      const float nmin = norm_min(v);
#pragma unroll
      for (int j = 0; j < R; ++j) prev[j] = start ? 0.f : v[j] - nmin;  // (the chain start has no front pixel)
    };

    Pix px[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) px[u] = load_pix(kPer * wave + u);
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      prepare(px[u], kPer * wave + u, kPer * wave + u, tt[u]);
      px[u] = load_pix(kBlockAlone + kPer * wave + u);
    }
    lds_barrier();
#pragma clang loop unroll(disable)
    for (int b = 0; b < blocks; ++b) {
#pragma clang loop unroll(disable)
      for (int i = 0; i < kBlockAlone; ++i) {
        float un[R], w;
        get_slot<R>(s.in[i][lane], un, w);
        scan(i, w, b == 0 && i == 0);
#pragma unroll
        for (int j = 0; j < R; ++j) uf[j] = un[j];
      }
      lds_barrier();
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int i = kPer * wave + u;
        finish(b * kBlockAlone + i, i, tt[u]);
        lds_order();
        prepare(px[u], (b + 1) * kBlockAlone + i, i, tt[u]);
        px[u] = load_pix((b + 2) * kBlockAlone + i);
      }
      lds_barrier();
    }
  };

  if (!(ch0.dir & 1)) walk(ch0, p.skip_s_store != 0, std::true_type());
  if ((ch0.dir & 1) || p.fused_pair) {
    ChainCtx ch = ch0;
    bool skip_s = p.skip_s_store != 0;
    if (!(ch0.dir & 1)) {
      // the second sweep of a pair reads what the first one stored: on the same compute unit, once the
      // stores are complete
      ch.dir = ch0.dir ^ 1;
      ch.pix0 = ch0.pix0 + (n - 1) * ch0.pstep;
      ch.pstep = -ch0.pstep;
      skip_s = p.skip_s_store2 != 0;
      wait_vmem<0>();
      __syncthreads();
    }
    walk(ch, skip_s, std::false_type());
  }
}

template <int R, bool TRAIN, int NT, bool SERVED>
__global__ void __launch_bounds__(SERVED ? kTeam : kTeamAlone) sweep_fwd_dense_kernel(const SweepParams p) {
  if (R == 1 && p.skip_dense && p.desc != nullptr && !is_dense(*p.desc)) return;
  extern __shared__ __align__(16) char smem_raw[];
  using S = std::conditional_t<SERVED, Slots<R>, SlotsAlone<R>>;
  S* s = reinterpret_cast<S*>(smem_raw);
  float* csym_s = reinterpret_cast<float*>(s + 1);
  fill_dense_sym<R>(csym_s, p.ctx, p.L, (int)threadIdx.x, SERVED ? kTeam : kTeamAlone);
  __syncthreads();
  const bool msg_zero = p.desc != nullptr && p.desc->msg_nonzero == 0;
  if constexpr (SERVED)
    walk_chain<R, TRAIN, NT>(p, locate_chain(p), msg_zero, *s, csym_s);
  else
    walk_chain_alone<R, TRAIN, NT>(p, locate_chain(p), msg_zero, *s, csym_s);
}

template <int R, int NT>
void launch(const SweepParams& p, bool train, hipStream_t st) {
  const int blocks = p.block_prefix[p.n_dirs];
  const size_t table = sizeof(float) * dense_sym_floats(R);
  // Three labels per lane: the table entries of a scanner and a server beside it leave the registers of a SIMD to one
  // chain.  Keeping argmin labels, rows of 129, ms for five pairs of sweeps, alone / served: 192 labels 256 chains 1.67 /
  // 1.15, 400 chains 1.97 / 2.26, 150 labels 700 chains (three pairs) 1.34 / 1.64.
  if constexpr (R == 3) {
    if (blocks > launch_policy().n_simd / 4) {
      auto kernel = train ? sweep_fwd_dense_kernel<R, true, NT, false> : sweep_fwd_dense_kernel<R, false, NT, false>;
      kernel<<<blocks, kTeamAlone, sizeof(SlotsAlone<R>) + table, st>>>(p);
      return;
    }
  }
  auto kernel = train ? sweep_fwd_dense_kernel<R, true, NT, true> : sweep_fwd_dense_kernel<R, false, NT, true>;
  kernel<<<blocks, kTeam, sizeof(Slots<R>) + table, st>>>(p);
}

}  // namespace

template <int R>
void launch_dense_fwd(const SweepParams& p, bool train, hipStream_t st) {
  if (p.block_prefix[p.n_dirs] <= 0) return;
  constexpr int kFull = 2 * R;  // trips of a wavefront that cover R labels per lane
  // (one trip fewer covers label counts up to 32 less)
  if (p.L <= kWaves * kTrip * (kFull - 1))
    launch<R, kFull - 1>(p, train, st);
  else
    launch<R, kFull>(p, train, st);
}

template void launch_dense_fwd<MPL_INST_R>(const SweepParams&, bool, hipStream_t);

}  // namespace mpl
