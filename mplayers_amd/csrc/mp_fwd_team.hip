// Forward scan of TRWP with four wavefronts per chain, in launches with fewer chains than the chip has
// SIMDs.  The recurrence and what each plane holds: mp_fwd.hip; the results are the same bits.
//
// What bounds such a launch is the length of one pixel's step, not memory: a wavefront that has its SIMD
// to itself issues one instruction every four clocks or more, and of the instructions of a step the next
// pixel waits for the beliefs, the minimum over front labels and the normalisation only.  So the work is
// divided by what the recurrence needs:
//   * three helper wavefronts (six where argmin labels are kept and chains are few: launch_v), every third (sixth)
//     pixel each, load the planes, form U of the pixel and put it
//     into an LDS slot; two blocks of pixels later they take the message from the slot and store the
//     planes.  Where argmin labels are kept they take the beliefs from the slot instead and run the
//     whole step again, with the labels: the same operations on the same operands, so the same message,
//   * the main wavefront touches LDS only: beliefs, minimum over front labels, normalisation.
// The wavefronts meet once per block of kT pixels: in iteration k the helpers finish block k - 2 and
// prepare block k while the main wavefront runs block k - 1.  The slots of a block are reused two
// iterations on by the helpers that own them, so two sets suffice.
//
// Measured, ns per pixel of rows of 256 / 512 chains, one wavefront per chain -> this: 60 labels, Potts, no
// argmin labels 150 / 158 -> 90 / 101; 96 labels, min(k, 3), kept 418 / 439 -> 204 / 241; 192 labels 469 / 500 ->
// 241 / 364 (with six helpers 183 / 236 and 228 / 385 on rows of 129), where the planes move at 4.7 TB/s.  The main wavefront of the first issues 29 instructions per
// pixel, of the last 57.  Which launches take it: team_fwd_chains_per_cu (mp_api.hip).
//
// Compiled once per R (labels per lane) with -DMPL_INST_R=<R>.

#include <type_traits>

#include "mp_fwd_step.h"

namespace mpl {
namespace {

constexpr int kT = 6;                // pixels per block, shared out among three or six helpers (launch_h)

constexpr int kAhead = 2;            // blocks of pixels whose loads are in flight (four and six measure the same)

// Slot of a pixel, per lane: U and the edge weight (one read; with four labels the weight has a word of
// its own for the pixel), and the message or, where argmin labels are kept, the beliefs it comes from.
constexpr int in_words(int R) { return R == 1 ? 2 : 4; }
constexpr int out_words(int R) { return R == 3 ? 4 : R; }
template <int R>
struct alignas(16) Slot {
  float in[kWave][in_words(R)];
  float out[kWave][out_words(R)];
};
struct Flags {
  int neg[kT];   // the pixel's edge weight is not >= 0: the band and the label scans do not hold there
  float w[kT];   // the edge weight (four labels per lane)
};

template <int N>
__device__ __forceinline__ void lds_get(const float* src, float (&x)[N]) {
  if constexpr (N == 4) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(src);
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = v[i];
  } else if constexpr (N == 2) {
    const f32x2 v = *reinterpret_cast<const f32x2*>(src);
    x[0] = v[0];
    x[1] = v[1];
  } else {
    static_assert(N == 1, "words of a slot");
    x[0] = *src;
  }
}
template <int N>
__device__ __forceinline__ void lds_put(float* dst, const float (&x)[N]) {
  if constexpr (N == 4) {
    *reinterpret_cast<f32x4*>(dst) = f32x4{x[0], x[1], x[2], x[3]};
  } else if constexpr (N == 3) {
    *reinterpret_cast<f32x4*>(dst) = f32x4{x[0], x[1], x[2], 0.f};
  } else if constexpr (N == 2) {
    *reinterpret_cast<f32x2*>(dst) = f32x2{x[0], x[1]};
  } else {
    static_assert(N == 1, "words of a slot");
    *dst = x[0];
  }
}
template <int R>
__device__ __forceinline__ void get_in(const Slot<R>& s, const Flags& f, int i, int lane, float (&un)[R], float& w) {
  float t[in_words(R)];
  lds_get(s.in[lane], t);
#pragma unroll
  for (int j = 0; j < R; ++j) un[j] = t[j];
  w = R == 4 ? f.w[i] : t[R < 4 ? R : 0];
}
template <int R>
__device__ __forceinline__ void put_in(Slot<R>& s, Flags& f, int i, int lane, const float (&un)[R], float w) {
  float t[in_words(R)];
#pragma unroll
  for (int j = 0; j < in_words(R); ++j) t[j] = j < R ? un[j < R ? j : 0] : w;
  lds_put(s.in[lane], t);
  if (R == 4) f.w[i] = w;  // (every lane the same value)
}
template <int R>
__device__ __forceinline__ void get_out(const Slot<R>& s, int lane, float (&x)[R]) {
  float t[out_words(R)];
  lds_get(s.out[lane], t);
#pragma unroll
  for (int j = 0; j < R; ++j) x[j] = t[j];
}

// workgroup barrier over LDS contents only: global loads in flight stay in flight
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// what every step of a walk needs
template <int R, int KT>
struct StepCtx {
  int L, lab0, lane, K;
  bool full_table;            // ctx_s holds the (L, L) table (2-D, or few labels; 21 labels: mp_team21.hip)
  float cmax, slope;
  float floor_l[R];           // -inf, +inf where the lane's label does not exist
  float c_reg[KT > 0 ? KT : 1];
  float cv0[R];               // dense 1-D table: c[label]
  float* a_w;                 // this wavefront's scratch, kMaxL floats
  const float* ctx_s;
  const float* c1_s;
  const float* csym_s;
  int ctx2d;
};

// The step of one pixel from the beliefs of its front pixel: v, the normalisation minimum and, where they
// are kept, the argmin labels.  KT, C0: run_chain_fwd (mp_fwd.hip).  PLAIN: no edge weight of the block is
// negative.
template <int R, int KT, bool C0, bool TRAIN, bool PLAIN>
__device__ __forceinline__ void team_step(const StepCtx<R, KT>& c, const float (&a)[R], const float wv,
                                          float (&v)[R], int (&fd_idx)[R], float& nmin) {
  constexpr bool kDenseMain = KT == -1;
  auto norm_min = [&]() __attribute__((always_inline)) {
    float vm = INFINITY;
#pragma unroll
    for (int j = 0; j < R; ++j) vm = fminf(vm, fmaxf(v[j], c.floor_l[j]));
    return wave_min_fast(vm);
  };
  const int L = c.L;
  bool fast = KT >= 0 || KT == -2;
  if constexpr ((KT >= 0 || KT == -2) && !PLAIN) fast = uniform_f(wv) >= 0.f;
  if (fast) {
    if constexpr (KT >= 0 || KT == -2) {
      constexpr bool kHead = !TRAIN && (KT >= 2 || (KT == 1 && R == 1));
      float amin;
      float hup[R], hdn[R];
      if constexpr (kHead) {
        float red;
        if constexpr (R == 1)
          band_head<KT>(a, wv, c.c_reg[0], c.c_reg[KT > 1 ? 1 : 0], red, v, hup, hdn);
        else
          band_head(a, wv, c.c_reg[0], c.c_reg[KT > 1 ? 1 : 0], red, v, hup, hdn);
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
        linear_step<R, TRAIN>(a, wv, c.slope, c.cmax, amin, fstar, c.lab0, c.lane, L, c.a_w, c.ctx_s, v, fd_idx);
      } else if constexpr (kHead && KT == 1) {
        v[0] = fminf(v[0], fmaf(wv, c.cmax, amin));
      } else {
        band_step<R, TRAIN, KT, kHead>(a, wv, c.K, c.c_reg, c.ctx_s, c.cmax, amin, fstar, c.lab0, v, fd_idx,
                                       hup, hdn);
      }
      if constexpr (KT != -2 && C0)
        nmin = fmaf(wv, KT > 0 ? c.c_reg[0] : c.ctx_s[0], amin);
      else
        nmin = norm_min();
    }
  } else if (R == 1 && KT < 0 && c.full_table) {
    dense_step_r1<TRAIN>(a[0], L, uniform_f(wv), c.lane, c.ctx_s, v[0], fd_idx[0]);
    nmin = norm_min();
  } else {
    const float w = uniform_f(wv);
    if constexpr (kDenseMain) {
      dense1d_step<R, TRAIN>(a, w, c.lab0, c.a_w, c.c1_s, c.cv0, v, fd_idx, 0, L);
      if (TRAIN) dense1d_argmin<R>(v, fd_idx, w, c.lab0, L, c.a_w, c.csym_s, fd_idx);
    } else if constexpr (R > 1 || KT == -2) {
      dense1d_step_lanes<R, TRAIN, false>(a, w, L, c.lab0, c.ctx_s, v, fd_idx, 0, L);
    } else {
      bool valid[R];
#pragma unroll
      for (int j = 0; j < R; ++j) valid[j] = c.lab0 + j < L;
      dense_step<R, TRAIN>(a, valid, w, L, c.ctx2d, c.lab0, c.a_w, c.ctx_s, v, fd_idx);
    }
    nmin = norm_min();
  }
}

template <int R>
struct PixT {
  float s[R], md[R], mi[R];
};

template <int R, bool VEC, bool TRAIN, int KT, bool C0, int kHelpers, bool THROUGH>
__device__ __forceinline__ void team_walk(const SweepParams& p, const CtxDesc& desc, const ChainCtx& ch0,
                                          Slot<R>* slots, Flags* flags, float* a_s, const float* ctx_s,
                                          const int role) {
  constexpr int kPer = kT / kHelpers;  // pixels of a block per helper
  const int L = p.L;
  const int lane = threadIdx.x & (kWave - 1);
  const int lab0 = R * lane;
  const bool lane_ok = lab0 < L;
  const int n = ch0.n;
  const float rho = p.rho;
  const int64_t HW = (int64_t)p.H * p.W;
  const int64_t P = (int64_t)p.B * HW;
  const int64_t N = P * L;
  const int blocks = (n + kT - 1) / kT;
  const int iters = (blocks + 2 + kAhead - 1) / kAhead * kAhead;  // (the helpers' loop is unrolled)

  StepCtx<R, KT> c;
  c.L = L;
  c.lab0 = lab0;
  c.lane = lane;
  c.K = desc.band_k;
  c.full_table = R == 1 && (p.ctx2d || (KT == -1 && L < kSlidingMinL));
  c.cmax = desc.cmax;
  asm volatile("" : "+v"(c.cmax));
  c.slope = desc.slope;
  c.a_w = a_s + role * kMaxL;
  c.ctx_s = ctx_s;
  c.c1_s = ctx_s + dense_c1_offset(L);
  c.csym_s = c.c1_s + dense_c1_floats(L);
  c.ctx2d = p.ctx2d;
#pragma unroll
  for (int j = 0; j < R; ++j) c.floor_l[j] = lab0 + j < L ? -INFINITY : INFINITY;
  if constexpr (KT > 0) {
#pragma unroll
    for (int k = 0; k < KT; ++k) c.c_reg[k] = p.ctx[k];
  }
  if constexpr (KT == -1) {
#pragma unroll
    for (int j = 0; j < R; ++j) c.cv0[j] = ctx_s[lab0 + j < L ? lab0 + j : L - 1];
  }

  auto main_walk = [&]() __attribute__((always_inline)) {
    float prev[R], uf[R];
#pragma unroll
    for (int j = 0; j < R; ++j) prev[j] = uf[j] = 0.f;
    auto pixel = [&](float (&out)[R], const float (&un)[R], const float w, const bool start, const auto plain)
        __attribute__((always_inline)) {
      float a[R], v[R], nmin;
      int fd_idx[R];
#pragma unroll
      for (int j = 0; j < R; ++j) a[j] = fmaf(rho, prev[j], uf[j]);
#pragma unroll
      for (int j = 0; j < R; ++j) out[j] = a[j];
      team_step<R, KT, C0, false, decltype(plain)::value>(c, a, w, v, fd_idx, nmin);
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const float m = v[j] - nmin;
        prev[j] = start ? 0.f : m;  // (the chain start has no front pixel and no message)
        uf[j] = un[j];
        if (!TRAIN) out[j] = prev[j];
      }
    };
    for (int k = 0; k < iters; ++k) {
      if (k >= 1 && k <= blocks) {
        Slot<R>* s = slots + ((k - 1) & 1) * kT;
        const Flags& f = flags[(k - 1) & 1];
        // Up to two labels per lane a group of two pixels is read and written at once: one LDS instruction takes both
        // and costs the main wavefront as much as three others.  Two over one, 256 chains of 129 / 450, no argmin labels
        // kept: 60 labels 0.94 / 0.94, 96 labels 0.93 / 0.90, 128 labels 0.93 / 0.91; kept, where the helpers do most, 0.96 to
        // 1.01.  Three and four labels fill an access of 16 bytes by themselves.
        constexpr int kGroup = R <= 2 ? 2 : 1;
        float un[kGroup][R], w[kGroup], out[kGroup][R];
#pragma unroll
        for (int u = 0; u < kGroup; ++u) get_in<R>(s[u], f, u, lane, un[u], w[u]);  // (ahead of the question, which takes as long)
        bool neg = false;
        if constexpr (KT >= 0 || KT == -2) neg = ballot(f.neg[lane < kT ? lane : 0] != 0) != 0;
        if (__builtin_expect(!neg, 1)) {
#pragma unroll
          for (int i = 0; i < kT; i += kGroup) {
            float nun[kGroup][R], nw[kGroup];
            if (i + kGroup < kT) {
#pragma unroll
              for (int u = 0; u < kGroup; ++u) get_in<R>(s[i + kGroup + u], f, i + kGroup + u, lane, nun[u], nw[u]);
            }
#pragma unroll
            for (int u = 0; u < kGroup; ++u) pixel(out[u], un[u], w[u], i + u == 0 && k == 1, std::true_type());
#pragma unroll
            for (int u = 0; u < kGroup; ++u) {
              lds_put(s[i + u].out[lane], out[u]);
              if (i + kGroup < kT) {
#pragma unroll
                for (int j = 0; j < R; ++j) un[u][j] = nun[u][j];
                w[u] = nw[u];
              }
            }
          }
        } else {
#pragma clang loop unroll(disable)
          for (int i = 0; i < kT; ++i) {
            get_in<R>(s[i], f, i, lane, un[0], w[0]);
            pixel(out[0], un[0], w[0], i == 0 && k == 1, std::false_type());
            lds_put(s[i].out[lane], out[0]);
          }
        }
      }
      lds_barrier();
    }
  };

  // even_walk: a constant; the first (even direction) or the second sweep of a pair (run_chain_fwd)
  auto helper_walk = [&](const ChainCtx& ch, const bool skip_s_in, const auto even_walk)
      __attribute__((always_inline)) {
    constexpr bool EVEN = decltype(even_walk)::value;
    const int dir = ch.dir;
    const int64_t img_p = (int64_t)ch.bv * HW;
    const int64_t img_e = img_p * L;
    const bool zfirst = p.zero_first && desc.msg_nonzero == 0;
    const bool skip_s = skip_s_in || (EVEN && zfirst);
    const bool md_zero = p.first_iter && desc.msg_nonzero == 0;
    const bool mi_zero = md_zero && EVEN;
    const int img_bytes = (int)(unsigned)(HW * L * 4);
    const int img_bytes_p = (int)(HW * 4 > 0x7fffffff ? 0x7fffffff : HW * 4);
    const float* bMd = p.msg_in + (int64_t)dir * N + img_e;
    const float* bMi = p.msg_in + (int64_t)(dir ^ 1) * N + img_e;
    const rsrc_t rS = make_rsrc((zfirst ? p.belief_zero : p.belief) + img_e, img_bytes);
    const rsrc_t rMd = make_rsrc(bMd, md_zero ? 0 : img_bytes);
    const rsrc_t rMi = make_rsrc(bMi, mi_zero ? 0 : img_bytes);
    const rsrc_t rMo = make_rsrc(p.msg_out + (int64_t)dir * N + img_e, img_bytes);
    const rsrc_t rSo = make_rsrc(p.belief_out + img_e, skip_s ? 0 : img_bytes);
    const rsrc_t rImin = make_rsrc(TRAIN ? p.idx_min + (int64_t)dir * N + img_e : nullptr, TRAIN ? (int)(HW * L) : 0);
    const rsrc_t dInorm = make_rsrc(TRAIN ? p.idx_norm + (int64_t)dir * P + img_p : nullptr, TRAIN ? (int)HW : 0);
    const rsrc_t dW = make_rsrc(p.edge + (int64_t)dir * P + img_p, img_bytes_p);

    // offsets of a lane's labels past the last one lie in the next pixel or past the image: with
    // whole lanes of labels such a lane is switched off, otherwise each label on its own
    auto vec_off = [&](bool on, unsigned so, int j) __attribute__((always_inline)) {
      return (int)((on && lab0 + j < L) ? so + (unsigned)(lab0 + j) * 4u : kDeadWide);
    };
    auto load_plane = [&](rsrc_t r, bool on, unsigned so, float (&x)[R]) __attribute__((always_inline)) {
      if constexpr (VEC) {
        buf_load<R, true, load_policy(false)>(r, vec_off(on, so, 0), 0u, x);
      } else {
#pragma unroll
        for (int j = 0; j < R; ++j)
          x[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, vec_off(on, so, j), 0, load_policy(false)));
      }
    };
    // THROUGH: where the messages fit the last-level cache (p.through, kCachedMessages) what is stored had better stay there.
    // Stores that go through the L2 at once (sc1) without the hint, over the hint, 5 iterations, 4 directions: 240x320, 60
    // labels 0.95 (8 directions 0.95), 96 labels 0.95, 128 labels 0.89; 375x450, 64 labels 0.93; argmin labels kept, the layer's
    // whole pass, 0.97 to 0.99.  Larger ones 300x400, 64 labels, 8 directions (246 MB) 1.01, 375x450, 60 labels, 8 directions
    // 1.19; three labels per lane 1.00 to 1.07.  (Neither hint nor sc1: 0.98, 0.97, 0.90, 0.96.  A branch
    // at every store in place of a kernel of its own costs more than it gives: training 96 labels 2.17 -> 3.38 ms.)
    auto store_plane = [&](rsrc_t r, bool on, unsigned so, const float (&x)[R]) __attribute__((always_inline)) {
      if constexpr (THROUGH) {
        buf_store<R, true, kStoreThrough>(r, vec_off(on, so, 0), 0u, x);
      } else if constexpr (VEC) {
        buf_store<R, true>(r, vec_off(on, so, 0), 0u, x);
      } else {
#pragma unroll
        for (int j = 0; j < R; ++j)
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x[j]), r, vec_off(on, so, j), 0, MPL_ST_AUX);
      }
    };
    // the loads of chain position t (nothing is read past the end of the chain).  The second sweep of a
    // pair reads its own old message at the chain start only.
    auto load_pix = [&](const int t) __attribute__((always_inline)) {
      PixT<R> r;
      const bool on = t < n;
      const unsigned pp = (unsigned)(ch.pix0 + t * ch.pstep);
      const unsigned so = pp * (unsigned)L * 4u;
      load_plane(rS, on, so, r.s);
      if (EVEN) load_plane(rMd, on, so, r.md);
      load_plane(rMi, on, so, r.mi);
      return r;
    };
    // the edge weights of this helper's next kWs pixels, one per lane, from chain position t on
    constexpr int kWs = kAhead * kPer;
    auto load_weights = [&](const int t) __attribute__((always_inline)) {
      const int tl = t + kHelpers * lane;
      const unsigned pp = (unsigned)(ch.pix0 + tl * ch.pstep);
      return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                           dW, (lane < kWs && tl < n) ? (int)(pp * 4u) : kDeadOffset, 0, 0));
    };
    const int first_stored = p.zero_start ? 0 : 1;
    float md0[R];  // second sweep: the old message of the chain start (helper 0)
    if (!EVEN) load_plane(rMd, role == 0, (unsigned)ch.pix0 * (unsigned)L * 4u, md0);

    float tt[2][kPer][R], ww[2][kPer];  // of the blocks in the slots

    // Whether chain position t is one of first .. n - 1, in one comparison: half of the helpers' instructions were scalar
    // ones that asked about either end.  60 and 64 labels, argmin labels kept, rows of 200 to 450, two comparisons -> one:
    // 128 and 256 chains 0.97, 320 to 512 chains 0.91 to 0.94, 700 chains 0.94; 96 and 128 labels 0.98 to 1.00; 191
    // labels 512 chains 0.95.  Without argmin labels 0.97 to 1.01.
    auto within = [&](const int t, const int first) __attribute__((always_inline)) {
      return (unsigned)(t - first) < (unsigned)(n - first);
    };
    auto prepare = [&](const PixT<R>& px, const float w, const int t, const int i, Slot<R>& s, Flags& f,
                       float (&tk)[R], float& wk)
        __attribute__((always_inline)) {
      float un[R], q[R];
#pragma unroll
      for (int j = 0; j < R; ++j) {
        tk[j] = EVEN ? px.s[j] - px.md[j] : px.s[j] + px.mi[j];
        un[j] = fmaf(tk[j], rho, -px.mi[j]);  // UpdateUnaryKernel, TRWP_forward.cu:70-78
        un[j] = KT == -1 && !c.full_table ? (lab0 + j < L ? un[j] : INFINITY) : fmaxf(un[j], c.floor_l[j]);  // (keep_nan, mp_fwd.hip)
        q[j] = tk[j] - px.mi[j];
      }
      wk = w;
      put_in<R>(s, f, i, lane, un, w);
      if (KT >= 0 || KT == -2) f.neg[i] = (within(t, 1) && !(w >= 0.f)) ? 1 : 0;
      // Q of the pixel is known already, whatever its message
      if (EVEN) store_plane(rSo, t < n, (unsigned)(ch.pix0 + t * ch.pstep) * (unsigned)L * 4u, q);
    };

    // what is left of a pixel once its message is known (nothing outside the chain)
    auto finish = [&](const int t, const Slot<R>& s, const float (&tk)[R], const float wk)
        __attribute__((always_inline)) {
      const bool on = within(t, 0);
      const unsigned pp = (unsigned)(ch.pix0 + t * ch.pstep);
      const unsigned so = pp * (unsigned)L * 4u;
      float m[R];
      get_out<R>(s, lane, m);
      if constexpr (TRAIN) {
        float a[R], v[R], nmin;
        int fd_idx[R];
#pragma unroll
        for (int j = 0; j < R; ++j) a[j] = m[j];
        team_step<R, KT, C0, true, false>(c, a, wk, v, fd_idx, nmin);
        bool pr[R];
#pragma unroll
        for (int j = 0; j < R; ++j) {
          m[j] = t == 0 ? 0.f : v[j] - nmin;
          pr[j] = lab0 + j < L && v[j] == nmin;
        }
        const int nidx = last_label<R>(pr, L - 1);
        const bool idx_on = within(t, 1);
        if constexpr (VEC) {
          buf_store_u8<R, true>(rImin, (int)((idx_on && lane_ok) ? pp * (unsigned)L + (unsigned)lab0 : kDeadWide), 0u, fd_idx);
        } else {
#pragma unroll
          for (int j = 0; j < R; ++j)
            __builtin_amdgcn_raw_buffer_store_b8((unsigned char)fd_idx[j], rImin,
                                                 (int)((idx_on && lab0 + j < L) ? pp * (unsigned)L + (unsigned)(lab0 + j) : kDeadWide),
                                                 0, MPL_ST_AUX);
        }
        // every lane stores the same byte to the same address
        __builtin_amdgcn_raw_buffer_store_b8((unsigned char)nidx, dInorm, idx_on ? (int)pp : kDeadOffset, 0, 0);
      }
      // (the reference never writes the chain start)
      store_plane(rMo, within(t, first_stored), so, m);
      if constexpr (!EVEN) {
        float sn[R];
#pragma unroll
        for (int j = 0; j < R; ++j) sn[j] = tk[j] + (t == 0 ? md0[j] : m[j]);
        store_plane(rSo, on, so, sn);
      }
    };

    PixT<R> ring[kAhead][kPer];
    float wnow = load_weights(role), wnext = 0.f;
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        ring[q][u] = load_pix(q * kT + role + kHelpers * u);
        MPL_ORDER_LOADS();
      }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        ww[q][u] = 0.f;
#pragma unroll
        for (int j = 0; j < R; ++j) tt[q][u][j] = 0.f;
      }
#pragma clang loop unroll(disable)
    for (int k0 = 0; k0 < iters; k0 += kAhead) {
      wnext = load_weights((k0 + kAhead) * kT + role);
#pragma unroll
      for (int q = 0; q < kAhead; ++q) {
        const int k = k0 + q;
        constexpr int kSets = 2;
        const int set = q % kSets;
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
          const int i = role + kHelpers * u;
          Slot<R>& s = slots[set * kT + i];
          finish((k - 2) * kT + i, s, tt[set][u], ww[set][u]);
          lds_order();
          prepare(ring[q][u], readlane_f(wnow, q * kPer + u), k * kT + i, i, s, flags[set], tt[set][u], ww[set][u]);
          ring[q][u] = load_pix((k + kAhead) * kT + i);
        }
        lds_barrier();
      }
      wnow = wnext;
    }
  };

  // the second sweep of a pair reads what the first one's helpers stored: on the same compute unit,
  // once their stores are complete
  if (role == kHelpers) {
    main_walk();
    if (!(ch0.dir & 1) && p.fused_pair) {
      __syncthreads();
      main_walk();
    }
  } else {
    if (!(ch0.dir & 1)) helper_walk(ch0, p.skip_s_store != 0, std::true_type());
    if ((ch0.dir & 1) || p.fused_pair) {
      ChainCtx ch = ch0;
      bool skip_s = p.skip_s_store != 0;
      if (!(ch0.dir & 1)) {
        ch.dir = ch0.dir ^ 1;
        ch.pix0 = ch0.pix0 + (n - 1) * ch0.pstep;
        ch.pstep = -ch0.pstep;
        skip_s = p.skip_s_store2 != 0;
        wait_vmem<0>();
        __syncthreads();
      }
      helper_walk(ch, skip_s, std::false_type());
    }
  }
}

template <int R, bool VEC, bool TRAIN, int kHelpers, bool THROUGH>
__global__ void __launch_bounds__((kHelpers + 1) * kWave) sweep_fwd_team_kernel(const SweepParams p) {
  constexpr int kTeam = (kHelpers + 1) * kWave;
  extern __shared__ __align__(16) char smem_raw[];
  Slot<R>* slots = reinterpret_cast<Slot<R>*>(smem_raw);  // two sets of kT
  float* a_s = reinterpret_cast<float*>(slots + 2 * kT);  // kMaxL floats per wavefront
  float* ctx_s = a_s + (kHelpers + 1) * kMaxL;            // as in sweep_fwd_kernel
  const int L = p.L;
  Flags* flags = reinterpret_cast<Flags*>(
      ctx_s + (p.ctx2d ? L * L : dense_c1_offset(L) + dense_c1_floats(L) + dense_sym_floats(R)));
  const int tid = threadIdx.x;
  // The last wavefront is the main one in every workgroup: the wavefronts of the workgroups that a compute
  // unit gets one after another start one SIMD further each (read from the hardware-id registers for 2, 3
  // and 4 workgroups per unit), so the main wavefronts of up to four of them are on SIMDs of their own.
  // (Of seven wavefronts the main one is the fourth, whose SIMD has only one of them.)
  const int wave = uniform_i(tid / kWave);
  const int role = wave == 3 ? kHelpers : wave - (wave > 3 ? 1 : 0);  // kHelpers: main
  const ChainCtx ch = locate_chain(p);

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
  if (p.skip_dense && is_dense(desc)) return;  // (mp_fwd_dense.hip runs such a launch)
  if (R == 1 && (p.ctx2d || (is_dense(desc) && L < kSlidingMinL))) {
    for (int i = tid; i < L * L; i += kTeam) {
      const int fd = i / L, cd = i - fd * L;
      const int lo = cd < fd ? cd : fd, hi = cd < fd ? fd : cd;
      ctx_s[i] = p.ctx[p.ctx2d ? lo * L + hi : hi - lo];
    }
  } else {
    const int n_ctx = p.ctx2d ? L * L : L;
    for (int i = tid; i < n_ctx; i += kTeam) ctx_s[i] = p.ctx[i];
    if (desc.band_k == 0) {
      float* c1_s = ctx_s + dense_c1_offset(L);
      for (int i = tid; i < dense_c1_floats(L); i += kTeam) c1_s[i] = i + 1 < L ? p.ctx[i + 1] : 0.f;
      if (TRAIN) fill_dense_sym<R>(c1_s + dense_c1_floats(L), p.ctx, L, tid, kTeam);
    }
  }
  __syncthreads();
  if (role == kHelpers) __builtin_amdgcn_s_setprio(3);

#define MPL_WALK(KT, C0) team_walk<R, VEC, TRAIN, KT, C0, kHelpers, THROUGH>(p, desc, ch, slots, flags, a_s, ctx_s, role)
  // (the choice of the step: sweep_fwd_kernel)
  if (desc.linear && !p.ctx2d && (desc.band_k == 0 || desc.band_k > 4)) {
    MPL_WALK(-2, false);
    return;
  }
  if (desc.band_k > 0 && !desc.c0_is_min) {
    MPL_WALK(0, false);
    return;
  }
  switch (desc.band_k) {
    case 0: MPL_WALK(-1, false); break;
    case 1: MPL_WALK(1, true); break;
    case 2: MPL_WALK(2, true); break;
    case 3: MPL_WALK(3, true); break;
    case 4: MPL_WALK(4, true); break;
    default:
      if constexpr (R >= 2) {
        if (desc.band_k <= 8) {
          MPL_WALK(8, true);
          break;
        }
        if (desc.band_k <= 16) {
          MPL_WALK(16, true);
          break;
        }
      }
      MPL_WALK(0, true);
      break;
  }
#undef MPL_WALK
}

inline size_t team_lds_bytes(int L, int R, bool ctx2d, size_t slot, int helpers) {
  const size_t table = ctx2d ? (size_t)L * L : dense_c1_offset(L) + dense_c1_floats(L) + dense_sym_floats(R);
  return 2 * kT * slot + sizeof(float) * ((helpers + 1) * kMaxL + table) + 2 * sizeof(Flags);
}

template <int R, bool VEC, bool TRAIN, int kHelpers>
void launch_h(const SweepParams& p, hipStream_t st) {
  const size_t lds = team_lds_bytes(p.L, R, p.ctx2d != 0, sizeof(Slot<R>), kHelpers);
  const auto launch = [&](auto kernel) { kernel<<<p.block_prefix[p.n_dirs], (kHelpers + 1) * kWave, lds, st>>>(p); };
  if constexpr (VEC && R <= 2) {
    if (p.through) {
      launch(sweep_fwd_team_kernel<R, VEC, TRAIN, kHelpers, true>);
      return;
    }
  }
  launch(sweep_fwd_team_kernel<R, VEC, TRAIN, kHelpers, false>);
}

template <int R, bool VEC, bool TRAIN>
void launch_v(const SweepParams& p, hipStream_t st) {
  // Where argmin labels are kept the helpers run every step again, and three of them bound a scan of up to two chains per
  // unit (with four labels per lane, one).  Six helpers over three, rows of 129: 60 labels, min(k, 3), 256 chains 0.78,
  // Potts 256 / 400 / 768 chains 0.84 / 0.89 / 0.97; 96 labels 256 / 512 / 768 chains 0.76 / 0.85 / 1.03; 192 labels 0.77 /
  // 0.95 / 1.07, a linear table 0.96 / 0.99; 256 labels 256 / 512 chains 0.82 / 1.03; labels one by one, 127 and 191 labels
  // 256 chains 0.73, 0.79.  Without argmin labels the main wavefront bounds it (0.99 to 1.07).
  if constexpr (TRAIN) {
    if (p.block_prefix[p.n_dirs] <= (R == 4 ? 1 : 2) * (launch_policy().n_simd / 4)) {
      launch_h<R, VEC, TRAIN, 6>(p, st);
      return;
    }
  }
  launch_h<R, VEC, TRAIN, 3>(p, st);
}

}  // namespace

template <int R, bool TRAIN>
void launch_team_fwd_t(const SweepParams& p, hipStream_t st) {
  if (p.block_prefix[p.n_dirs] <= 0) return;
  if (p.L % R == 0)
    launch_v<R, true, TRAIN>(p, st);
  else if constexpr (R > 1)
    launch_v<R, false, TRAIN>(p, st);
}

template void launch_team_fwd_t<MPL_INST_R, (MPL_INST_TRAIN != 0)>(const SweepParams&, hipStream_t);

}  // namespace mpl
