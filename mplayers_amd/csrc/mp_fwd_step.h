// The steps of the forward scans over one pixel: the minimum over front labels for every kind of
// table, with or without argmin labels, and what finds the normalisation minimum along with it.
// Included by mp_fwd.hip (one wavefront per chain) and mp_fwd_team.hip (four).
#ifndef MPLAYERS_AMD_MP_FWD_STEP_H_
#define MPLAYERS_AMD_MP_FWD_STEP_H_

#include "mp_common.h"

namespace mpl {
namespace {

// The order of this wavefront's own LDS accesses, as the steps below need it where lanes exchange values
// through LDS (the hardware keeps it; no instruction is emitted).
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}

// Comparisons that are false of what is no number, whichever way round the compiler puts the select behind them (of a
// plain one it takes the opposite, which is false of it too).
__device__ __forceinline__ bool equal(const float a, const float b) {
  return __builtin_amdgcn_inverse_ballot_w64(__builtin_amdgcn_fcmpf(a, b, 1));  // (ordered, equal)
}
__device__ __forceinline__ bool at_most(const float a, const float b) {
  return __builtin_amdgcn_inverse_ballot_w64(__builtin_amdgcn_fcmpf(a, b, 5));  // (ordered, less or equal)
}

// Dense O(L^2) step: v[cd] = min_fd( a[fd] + w * ctx(cd, fd) ), largest fd on ties.
// HorizontalKernel inner loop, TRWP_forward.cu:127-153.  a_s / ctx_s live in LDS.
template <int R, bool TRAIN>
__device__ __forceinline__ void dense_step(const float (&a)[R], const bool (&valid)[R], float w,
                                           int L, int ctx2d, int lab0, float* a_s,
                                           const float* ctx_s, float (&v)[R], int (&fd_idx)[R]) {
#pragma unroll
  for (int j = 0; j < R; ++j)
    if (valid[j]) a_s[lab0 + j] = a[j];
  lds_order();
  int labc[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    int l = lab0 + j;
    labc[j] = l < L ? l : L - 1;
    v[j] = INFINITY;
    fd_idx[j] = L - 1;
  }
  for (int fd = L - 1; fd >= 0; --fd) {
    float af = a_s[fd];
#pragma unroll
    for (int j = 0; j < R; ++j) {
      int cd = labc[j];
      int ci = ctx2d ? (cd < fd ? cd * L + fd : fd * L + cd) : (cd > fd ? cd - fd : fd - cd);
      float val = fmaf(w, ctx_s[ci], af);
      if (TRAIN) {
        bool take = (fd == L - 1) || (val < v[j]);
        v[j] = take ? val : v[j];
        fd_idx[j] = take ? fd : fd_idx[j];
      } else {
        v[j] = fminf(v[j], val);
      }
    }
  }
  lds_order();
}

// Dense O(L^2) step for 1-D contexts.  The front labels are visited
// in ascending order; the context values c[|cd - fd|] of the lane's labels are kept in registers and
// moved one label up per front label (c[|cd - (fd+1)|] of label cd is c[|(cd-1) - fd|] of label
// cd - 1; c[fd+1] enters at label 0) with one lane shift.  Both a[fd] and the entering c[fd+1] are
// the same for every lane: they are read from LDS, every lane from the same address (a_w: this
// wavefront's own copy of a[], written at the start of the step; c1_s: the table moved down by one
// entry, c1_s[i] = c[i+1]), four front labels per read, one trip of T = 4 R front labels ahead of
// their use, so the loop waits for none of them.  The shift writes into the register the read
// filled (lane 0 has no source lane and keeps c[fd+1]): no instruction sets up a fill.
// Two front labels are folded per minimum (v_min3).
// TRAIN: the argmin label is found in two steps.  The scan only notes, per label, the trip whose
// candidates last reached the running minimum (the minimum over a trip's candidates against the
// minimum so far, `<=`: one comparison and one select per trip instead of one per front label), and
// returns that trip's first front label in `trip0`; dense1d_argmin then evaluates the T candidates
// of that one trip again.  The argmin the reference keeps is the largest front label whose candidate
// equals the final minimum (its descending scan with `<`): it lies in the last trip that holds such
// a candidate, and that is the last trip whose own minimum is <= the minimum before it.
// The scan covers the front labels fd_lo .. fd_hi - 1 (fd_lo a multiple of T): all of them, or the
// share of one wavefront where several scan a pixel together (split_combine below).  cv0: the
// sliding values at fd_lo, c[|cd - fd_lo|].
// (one label per lane: two groups of four to a trip, since a group's register is still a sliding value
// when the next trip would read the same one)
template <int R>
constexpr int dense_trip() { return R == 1 ? 8 : 4 * R; }

template <int R, bool TRAIN>
__device__ __forceinline__ void dense1d_step(const float (&a)[R], const float w, const int lab0,
                                             float* a_w, const float* c1_s, const float (&cv0)[R],
                                             float (&v)[R], int (&trip0)[R], const int fd_lo,
                                             const int fd_hi) {
  constexpr int T = dense_trip<R>();
  float cv[R];
  int rel[R];  // the noted trip, counted back from the current one (0, -1, ...)
#pragma unroll
  for (int j = 0; j < R; ++j) {
    a_w[lab0 + j] = a[j];
    cv[j] = cv0[j];
    v[j] = INFINITY;
    rel[j] = 0;
  }
  auto shift = [&](const float fill) __attribute__((always_inline)) {
    const float in0 = wave_shr1(cv[R - 1], fill);
#pragma unroll
    for (int j = R - 1; j > 0; --j) cv[j] = cv[j - 1];
    cv[0] = in0;
  };
  // the end of a trip: fold its minimum into the running one and note the trip where it reaches it
  auto close_trip = [&](const float (&lm)[R]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const bool take = at_most(lm[j], v[j]);
      v[j] = fminf(v[j], lm[j]);
      rel[j] = take ? 0 : rel[j] - 1;
    }
  };
  float ba[T], bc[T];  // a[fd0 + u], c[fd0 + u + 1]
  auto read4 = [&](const float* src, float (&dst)[T], const int q) __attribute__((always_inline)) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(src + 4 * q);
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[4 * q + i] = x[i];
  };
  // The register a read of c fills becomes a sliding value and stays one for R shifts: the four of
  // group q are free again after shift 4 q + 3 + R of a trip, and that is where the group's next
  // read stands -- in the same trip for the trip after it (kNext groups), or, for the last groups,
  // at the start of the trip that uses them.
  constexpr int kNext = (T - 3 - R + 3) / 4;  // groups q with 4 q + 3 + R < T
  int fd0 = fd_lo;
#pragma unroll
  for (int q = 0; q < T / 4; ++q) read4(a_w + fd0, ba, q);
#pragma unroll
  for (int q = 0; q < kNext; ++q) read4(c1_s + fd0, bc, q);
  for (; fd0 + T <= fd_hi; fd0 += T) {
    float lm[R];  // TRAIN: the minimum over this trip's candidates
#pragma unroll
    for (int u = 0; u < T; u += 2) {
      float v0[R], v1[R];
#pragma unroll
      for (int j = 0; j < R; ++j) v0[j] = fmaf(w, cv[j], ba[u]);
      shift(bc[u]);
#pragma unroll
      for (int j = 0; j < R; ++j) v1[j] = fmaf(w, cv[j], ba[u + 1]);
      shift(bc[u + 1]);
#pragma unroll
      for (int j = 0; j < R; ++j) {
        if (TRAIN)
          lm[j] = u == 0 ? fminf(v0[j], v1[j]) : fminf(fminf(lm[j], v0[j]), v1[j]);
        else
          v[j] = fminf(fminf(v[j], v0[j]), v1[j]);
      }
      // reads that stand after the shifts u and u + 1
#pragma unroll
      for (int s = u; s < u + 2; ++s) {
        if ((s & 3) == 3) read4(a_w + fd0 + T, ba, s / 4);  // a: free once its four labels are done
        if (s >= 3 + R && ((s - 3 - R) & 3) == 0) read4(c1_s + fd0 + T, bc, (s - 3 - R) / 4);
        if (s + T >= 3 + R && s + T - 3 - R < T && ((s + T - 3 - R) & 3) == 0 &&
            (s + T - 3 - R) / 4 >= kNext)
          read4(c1_s + fd0, bc, (s + T - 3 - R) / 4);
      }
    }
    if (TRAIN) close_trip(lm);
  }
  // what is left of the share: fewer than T front labels, one at a time
  if (fd0 < fd_hi) {
#pragma unroll
    for (int q = kNext; q < T / 4; ++q) read4(c1_s + fd0, bc, q);
    float lm[R];
#pragma unroll
    for (int j = 0; j < R; ++j) lm[j] = INFINITY;
#pragma unroll
    for (int u = 0; u < T - 1; ++u) {
      if (fd0 + u < fd_hi) {  // wave-uniform
#pragma unroll
        for (int j = 0; j < R; ++j) {
          const float val = fmaf(w, cv[j], ba[u]);
          if (TRAIN)
            lm[j] = fminf(lm[j], val);
          else
            v[j] = fminf(v[j], val);
        }
        shift(bc[u]);
      }
    }
    if (TRAIN) close_trip(lm);
    fd0 += T;
  }
#pragma unroll
  for (int j = 0; j < R; ++j) trip0[j] = (fd0 - T) + rel[j] * T;
}

// The argmin labels of dense1d_step: for every label of the lane, the largest front label of the
// trip starting at trip0 whose candidate a[fd] + w * c[|cd - fd|] equals the minimum v (the same
// multiply-add on the same operands as in the scan: the same bits).  a_w: the wavefront's copy of
// a[] (front labels past the last one read as +inf or as whatever lies there: their candidates
// are not the minimum); csym_s: the table laid out around its centre, csym_s[dense_sym_centre<R>() + d]
// = c[|d|], so that a lane reads the entries of consecutive front labels at consecutive addresses.
template <int R>
constexpr int dense_sym_centre() { return R * kWave; }  // |cd - fd| < R * 64

template <int R>
__device__ __forceinline__ void fill_dense_sym(float* csym_s, const float* ctx, int L, int tid,
                                               int n_threads) {
  for (int i = tid; i < dense_sym_floats(R); i += n_threads) {
    const int d = i < dense_sym_centre<R>() ? dense_sym_centre<R>() - i : i - dense_sym_centre<R>();
    csym_s[i] = d < L ? ctx[d] : 0.f;
  }
}

template <int R>
__device__ __forceinline__ void dense1d_argmin(const float (&v)[R], const int (&trip0)[R],
                                               const float w, const int lab0, const int L,
                                               const float* a_w, const float* csym_s,
                                               int (&fd_idx)[R]) {
  constexpr int T = dense_trip<R>();
#pragma unroll
  for (int j = 0; j < R; ++j) {
    // (no trip is noted where no candidate is a number, and no label found there: the last one, as the
    // reference's scan has it)
    const int t0 = max(trip0[j], 0);
    const int l = lab0 + j < L ? lab0 + j : L - 1;
    float af[T];
#pragma unroll
    for (int q = 0; q < T / 4; ++q) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(a_w + t0 + 4 * q);
#pragma unroll
      for (int i = 0; i < 4; ++i) af[4 * q + i] = x[i];
    }
    const float* cp = csym_s + (dense_sym_centre<R>() + l - t0 - (T - 1));  // entry of front label t0 + T - 1
    int arg = kMaxL;
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const float val = fmaf(w, cp[T - 1 - u], af[u]);
      arg = equal(val, v[j]) ? u : arg;
    }
    const int fd = t0 + arg;
    fd_idx[j] = fd < L ? fd : L - 1;
  }
}

// The same scan with both broadcasts taken from the lanes that hold the values (v_readlane of a[]
// and of the lane's own table entries c[label]) instead of LDS: no staging, no reads in flight, and
// little state outside the step.  Two more issue slots per front label than dense1d_step; it is the
// step that a kernel compiled for a band or a truncated-linear table takes at a pixel with a
// negative edge weight, where the band and the label scans do not hold.
// `<=` on the ascending scan keeps the largest front label among equals, as the reference's
// descending scan with `<` does.  fd_lo a multiple of R.
template <int R, bool TRAIN, bool WHOLE>  // WHOLE: L is a multiple of R
__device__ __forceinline__ void dense1d_step_lanes(const float (&a)[R], float w, int L, int lab0,
                                             const float* ctx_s, float (&v)[R], int (&fd_idx)[R],
                                             const int fd_lo, const int fd_hi) {
  float c_own[R], cv[R];  // c[label] of the lane's labels; the sliding c[|label - fd|]
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int l = lab0 + j < L ? lab0 + j : L - 1;
    c_own[j] = ctx_s[l];
    cv[j] = fd_lo == 0 ? c_own[j] : ctx_s[l > fd_lo ? l - fd_lo : fd_lo - l];
    v[j] = INFINITY;
    fd_idx[j] = L - 1;
  }
  // the weight in a vector register: a multiply-add takes one scalar operand, and that is a[fd]
  float wv = w;
  asm volatile("" : "+v"(wv));
  // one front label: fd = fd0 + u is owned by lane src = fd0 / R, register u
  auto visit = [&](const int fd, const int u, const int src) __attribute__((always_inline)) {
    const float af = readlane_f(a[u], src);
    // c[fd + 1]: the next label's own entry (past the last label the value is never used)
    const float cn = u + 1 < R ? readlane_f(c_own[u + 1 < R ? u + 1 : 0], src)
                               : readlane_f(c_own[0], (src + 1) & 63);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const float val = fmaf(wv, cv[j], af);
      if (TRAIN) {
        // (the minimum and the comparison are independent instructions; a select of the value
        // would wait for the comparison's lane mask like the select of the label does)
        const bool take = at_most(val, v[j]);
        v[j] = fminf(v[j], val);
        fd_idx[j] = take ? fd : fd_idx[j];
      } else {
        v[j] = fminf(v[j], val);
      }
    }
    const float in0 = wave_shr1(cv[R - 1], cn);
#pragma unroll
    for (int j = R - 1; j > 0; --j) cv[j] = cv[j - 1];
    cv[0] = in0;
  };
  // Two rounds of R front labels per trip: after R one-label shifts the sliding values sit in
  // registers the shifts created, after 2 R they can be back in the ones the trip started with,
  // so the loop carries no register moves.
  int fd0 = fd_lo;
  int src0 = fd_lo / R;  // the lane that owns front label fd0 (counted along: no division per trip)
  for (; fd0 + 2 * R <= fd_hi; fd0 += 2 * R, src0 += 2) {
#pragma unroll
    for (int u = 0; u < 2 * R; ++u) visit(fd0 + u, u % R, src0 + u / R);
  }
  for (; fd0 < fd_hi; fd0 += R, ++src0) {
#pragma unroll
    for (int u = 0; u < R; ++u)
      if (WHOLE || fd0 + u < fd_hi) visit(fd0 + u, u, src0);  // wave-uniform
  }
}

// Dense step for 2-D contexts (one label per lane): a[fd] is broadcast with v_readlane and the context
// comes from a full table tab[fd * L + cd] in LDS, which consecutive lanes read without bank
// conflicts.  Same scan order as dense_step.  1-D tables of fewer than kSlidingMinL labels take it as well: dense1d_step works in trips of eight front labels and finds the argmin
// label in a second step.  Measured, TRWP 600x700, 4 directions, 2 iterations, us with this / with dense1d_step, argmin
// labels kept: 3 labels 1544 / 2762, 4 1773 / 2818, 6 2292 / 2911, 8 2768 / 2684, 16 4678 / 3287; without them:
// 3 labels 1390 / 1583, 4 1598 / 1639, 8 2459 / 1544.
constexpr int kSlidingMinL = 8;
template <bool TRAIN>
__device__ __forceinline__ void dense_step_r1(float a, int L, float w, int lane, const float* tab,
                                              float& v, int& fd_idx) {
  const float* col = tab + (lane < L ? lane : L - 1);
  float best = INFINITY;
  int arg = L - 1;
#pragma unroll 4
  for (int fd = L - 1; fd >= 0; --fd) {
    const float af = readlane_f(a, fd);
    const float val = fmaf(w, col[fd * L], af);
    if (TRAIN) {
      const bool take = (fd == L - 1) || (val < best);
      best = take ? val : best;
      arg = take ? fd : arg;
    } else {
      best = fminf(best, val);
    }
  }
  v = best;
  fd_idx = arg;
}

// For the 21 candidates of a lane's label and their minimum `best`: the largest fd with
// val[fd] == best, and in `red` (on entry: best in the lanes of the 21 labels, +inf elsewhere) the
// minimum over lanes 0..31 in lane 31.
// A comparison leaves its lane mask in scalar registers, and a select may read such a mask only two
// issue slots after it was written; a lane shift may read a vector register only two slots after
// it was written.  The compiler keeps every mask in vcc and pads each of these pairs with idle
// slots (some 50 per pixel, and a wavefront that has its SIMD to itself pays for every slot), so
// the three chains are interleaved by hand: masks rotate over three registers, every select comes
// at least two instructions after its comparison, every shift at least two after the one before,
// and the first shift three after the start (the compiler wrote `red` just before).
__device__ __forceinline__ void argmin_and_lane_min_21(const float (&val)[21], float best, float& red,
                                                       int& arg) {
  unsigned long long m1, m2;
  asm(
      "v_cmp_eq_f32_e64 vcc, %5, %4\n\t"
      "v_cmp_eq_f32_e64 %2, %6, %4\n\t"
      "v_cmp_eq_f32_e64 %3, %7, %4\n\t"
      "v_min_f32_dpp %1, %1, %1 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_e64 %0, 20, 0, vcc\n\t"
      "v_cmp_eq_f32_e64 vcc, %8, %4\n\t"
      "v_min_f32_dpp %1, %1, %1 row_shr:2 row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_e64 %0, %0, 1, %2\n\t"
      "v_cmp_eq_f32_e64 %2, %9, %4\n\t"
      "v_min_f32_dpp %1, %1, %1 row_shr:4 row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_e64 %0, %0, 2, %3\n\t"
      "v_cmp_eq_f32_e64 %3, %10, %4\n\t"
      "v_min_f32_dpp %1, %1, %1 row_shr:8 row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_e64 %0, %0, 3, vcc\n\t"
      "v_cmp_eq_f32_e64 vcc, %11, %4\n\t"
      "v_min_f32_dpp %1, %1, %1 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
      "v_cndmask_b32_e64 %0, %0, 4, %2\n\t"
      "v_cmp_eq_f32_e64 %2, %12, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 5, %3\n\t"
      "v_cmp_eq_f32_e64 %3, %13, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 6, vcc\n\t"
      "v_cmp_eq_f32_e64 vcc, %14, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 7, %2\n\t"
      "v_cmp_eq_f32_e64 %2, %15, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 8, %3\n\t"
      "v_cmp_eq_f32_e64 %3, %16, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 9, vcc\n\t"
      "v_cmp_eq_f32_e64 vcc, %17, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 10, %2\n\t"
      "v_cmp_eq_f32_e64 %2, %18, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 11, %3\n\t"
      "v_cmp_eq_f32_e64 %3, %19, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 12, vcc\n\t"
      "v_cmp_eq_f32_e64 vcc, %20, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 13, %2\n\t"
      "v_cmp_eq_f32_e64 %2, %21, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 14, %3\n\t"
      "v_cmp_eq_f32_e64 %3, %22, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 15, vcc\n\t"
      "v_cmp_eq_f32_e64 vcc, %23, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 16, %2\n\t"
      "v_cmp_eq_f32_e64 %2, %24, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 17, %3\n\t"
      "v_cmp_eq_f32_e64 %3, %25, %4\n\t"
      "v_cndmask_b32_e64 %0, %0, 18, vcc\n\t"
      "v_cndmask_b32_e64 %0, %0, 19, %2\n\t"
      "v_cndmask_b32_e64 %0, %0, 20, %3\n\t"
      : "=&v"(arg), "+v"(red), "=&s"(m1), "=&s"(m2)
      : "v"(best), "v"(val[0]), "v"(val[1]), "v"(val[2]), "v"(val[3]), "v"(val[4]), "v"(val[5]), "v"(val[6]), "v"(val[7]), "v"(val[8]), "v"(val[9]), "v"(val[10]), "v"(val[11]), "v"(val[12]), "v"(val[13]), "v"(val[14]), "v"(val[15]), "v"(val[16]), "v"(val[17]), "v"(val[18]), "v"(val[19]), "v"(val[20])
      : "vcc");
}

// Several labels per lane, no argmin labels: the wavefront minimum of the beliefs and, in the issue
// slots its six lane-shift minima leave (a lane shift may read a register two slots after it was
// written, and a wavefront that has its SIMD to itself pays for every idle slot), the centre tap and
// the first tap of the band step: on exit v[j] = min(a[j] + w c[0], min(a[label-1], a[label+1]) + w c[1]),
// up / dn hold the beliefs of the labels one up and one down, and `red` holds in lane 63 the minimum
// of a[] over the wavefront.  The same operations on the same operands as wave_min_fast and
// band_step's first tap: the same bits.  w: the edge weight in a vector register.
#define MPL_RED(CTRL) "v_min_f32_dpp %0, %0, %0 " CTRL " bank_mask:0xf\n\t"
__device__ __forceinline__ void band_head(const float (&a)[2], float w, float c0, float c1, float& red,
                                          float (&v)[2], float (&up)[2], float (&dn)[2]) {
  float tu, td, q0, q1, p0, p1;
  red = fminf(a[0], a[1]);
  asm("v_mov_b32 %1, 0x7f800000\n\t"
      "v_mov_b32 %2, 0x7f800000\n\t"
      MPL_RED("row_shr:1 row_mask:0xf")
      "v_fma_f32 %5, %9, %10, %7\n\t"
      "v_fma_f32 %6, %9, %10, %8\n\t"
      MPL_RED("row_shr:2 row_mask:0xf")
      "v_mov_b32_dpp %1, %7 wave_shl:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b32_dpp %2, %8 wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
      MPL_RED("row_shr:4 row_mask:0xf")
      "v_min_f32 %3, %8, %2\n\t"
      "v_min_f32 %4, %1, %7\n\t"
      MPL_RED("row_shr:8 row_mask:0xf")
      "v_fmac_f32 %3, %9, %11\n\t"
      "v_fmac_f32 %4, %9, %11\n\t"
      MPL_RED("row_bcast:15 row_mask:0xa")
      "v_min_f32 %5, %5, %3\n\t"
      "v_min_f32 %6, %6, %4\n\t"
      "v_min_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf"
      : "+v"(red), "=&v"(tu), "=&v"(td), "=&v"(q0), "=&v"(q1), "=&v"(p0), "=&v"(p1)
      : "v"(a[0]), "v"(a[1]), "v"(w), "v"(c0), "v"(c1));
  v[0] = p0;
  v[1] = p1;
  up[0] = a[1];
  up[1] = tu;
  dn[0] = td;
  dn[1] = a[0];
}

__device__ __forceinline__ void band_head(const float (&a)[3], float w, float c0, float c1, float& red,
                                          float (&v)[3], float (&up)[3], float (&dn)[3]) {
  float tu, td, q0, q1, q2, p0, p1, p2;
  red = fminf(fminf(a[0], a[1]), a[2]);
  // %0 red  %1 tu  %2 td  %3..%5 q  %6..%8 p  %9..%11 a  %12 w  %13 c0  %14 c1
  asm("v_mov_b32 %1, 0x7f800000\n\t"
      "v_mov_b32 %2, 0x7f800000\n\t"
      MPL_RED("row_shr:1 row_mask:0xf")
      "v_fma_f32 %6, %12, %13, %9\n\t"
      "v_fma_f32 %7, %12, %13, %10\n\t"
      MPL_RED("row_shr:2 row_mask:0xf")
      "v_mov_b32_dpp %1, %9 wave_shl:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b32_dpp %2, %11 wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
      MPL_RED("row_shr:4 row_mask:0xf")
      "v_fma_f32 %8, %12, %13, %11\n\t"
      "v_min_f32 %4, %11, %9\n\t"
      MPL_RED("row_shr:8 row_mask:0xf")
      "v_min_f32 %3, %10, %2\n\t"
      "v_min_f32 %5, %1, %10\n\t"
      MPL_RED("row_bcast:15 row_mask:0xa")
      "v_fmac_f32 %3, %12, %14\n\t"
      "v_fmac_f32 %4, %12, %14\n\t"
      MPL_RED("row_bcast:31 row_mask:0xc")
      "v_fmac_f32 %5, %12, %14\n\t"
      "v_min_f32 %6, %6, %3\n\t"
      "v_min_f32 %7, %7, %4\n\t"
      "v_min_f32 %8, %8, %5"
      : "+v"(red), "=&v"(tu), "=&v"(td), "=&v"(q0), "=&v"(q1), "=&v"(q2), "=&v"(p0), "=&v"(p1),
        "=&v"(p2)
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(w), "v"(c0), "v"(c1));
  v[0] = p0;
  v[1] = p1;
  v[2] = p2;
  up[0] = a[1];
  up[1] = a[2];
  up[2] = tu;
  dn[0] = td;
  dn[1] = a[0];
  dn[2] = a[1];
}

__device__ __forceinline__ void band_head(const float (&a)[4], float w, float c0, float c1, float& red,
                                          float (&v)[4], float (&up)[4], float (&dn)[4]) {
  float tu, td, q0, q1, q2, q3, p0, p1, p2, p3;
  red = fminf(fminf(a[0], a[1]), fminf(a[2], a[3]));
  // %0 red  %1 tu  %2 td  %3..%6 q  %7..%10 p  %11..%14 a  %15 w  %16 c0  %17 c1
  asm("v_mov_b32 %1, 0x7f800000\n\t"
      "v_mov_b32 %2, 0x7f800000\n\t"
      MPL_RED("row_shr:1 row_mask:0xf")
      "v_fma_f32 %7, %15, %16, %11\n\t"
      "v_fma_f32 %8, %15, %16, %12\n\t"
      MPL_RED("row_shr:2 row_mask:0xf")
      "v_mov_b32_dpp %1, %11 wave_shl:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b32_dpp %2, %14 wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
      MPL_RED("row_shr:4 row_mask:0xf")
      "v_fma_f32 %9, %15, %16, %13\n\t"
      "v_fma_f32 %10, %15, %16, %14\n\t"
      MPL_RED("row_shr:8 row_mask:0xf")
      "v_min_f32 %4, %13, %11\n\t"
      "v_min_f32 %5, %14, %12\n\t"
      MPL_RED("row_bcast:15 row_mask:0xa")
      "v_min_f32 %3, %12, %2\n\t"
      "v_min_f32 %6, %1, %13\n\t"
      MPL_RED("row_bcast:31 row_mask:0xc")
      "v_fmac_f32 %3, %15, %17\n\t"
      "v_fmac_f32 %4, %15, %17\n\t"
      "v_fmac_f32 %5, %15, %17\n\t"
      "v_fmac_f32 %6, %15, %17\n\t"
      "v_min_f32 %7, %7, %3\n\t"
      "v_min_f32 %8, %8, %4\n\t"
      "v_min_f32 %9, %9, %5\n\t"
      "v_min_f32 %10, %10, %6"
      : "+v"(red), "=&v"(tu), "=&v"(td), "=&v"(q0), "=&v"(q1), "=&v"(q2), "=&v"(q3), "=&v"(p0),
        "=&v"(p1), "=&v"(p2), "=&v"(p3)
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(w), "v"(c0), "v"(c1));
  v[0] = p0;
  v[1] = p1;
  v[2] = p2;
  v[3] = p3;
  up[0] = a[1];
  up[1] = a[2];
  up[2] = a[3];
  up[3] = tu;
  dn[0] = td;
  dn[1] = a[0];
  dn[2] = a[1];
  dn[3] = a[2];
}
// One label per lane, the same.  KT == 1 (a Potts table): the centre tap alone.  The minimum goes round each row of
// lanes first: a rotation reaches every lane, so it needs no copy of the beliefs to fall back on.
template <int KT>
__device__ __forceinline__ void band_head(const float (&a)[1], float w, float c0, float c1, float& red,
                                          float (&v)[1], float (&up)[1], float (&dn)[1]) {
  if constexpr (KT == 1) {
    asm("v_fma_f32 %1, %3, %4, %2\n\ts_nop 0\n\t"
        "v_min_f32_dpp %0, %2, %2 row_ror:8 row_mask:0xf bank_mask:0xf\n\ts_nop 1\n\t"
        MPL_RED("row_ror:4 row_mask:0xf") "s_nop 1\n\t"
        MPL_RED("row_ror:2 row_mask:0xf") "s_nop 1\n\t"
        MPL_RED("row_ror:1 row_mask:0xf") "s_nop 1\n\t"
        MPL_RED("row_bcast:15 row_mask:0xa") "s_nop 1\n\t"
        "v_min_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf"
        : "=&v"(red), "=&v"(v[0])
        : "v"(a[0]), "v"(w), "v"(c0));
    up[0] = dn[0] = a[0];
  } else {
    float tu, td, q, p;
    asm("v_mov_b32 %1, 0x7f800000\n\t"
        "v_mov_b32 %2, 0x7f800000\n\t"
        "v_min_f32_dpp %0, %5, %5 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_mov_b32_dpp %1, %5 wave_shl:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_mov_b32_dpp %2, %5 wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
        MPL_RED("row_ror:4 row_mask:0xf")
        "v_fma_f32 %4, %6, %7, %5\n\t"
        "v_min_f32 %3, %1, %2\n\t"
        MPL_RED("row_ror:2 row_mask:0xf")
        "v_fmac_f32 %3, %6, %8\n\t"
        "s_nop 0\n\t"
        MPL_RED("row_ror:1 row_mask:0xf")
        "v_min_f32 %4, %4, %3\n\t"
        "s_nop 0\n\t"
        MPL_RED("row_bcast:15 row_mask:0xa")
        "s_nop 1\n\t"
        "v_min_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf"
        : "=&v"(red), "=&v"(tu), "=&v"(td), "=&v"(q), "=&v"(p)
        : "v"(a[0]), "v"(w), "v"(c0), "v"(c1));
    v[0] = p;
    up[0] = tu;
    dn[0] = td;
  }
}
#undef MPL_RED
// Band O(L*K) step for 1-D contexts with a constant tail (c[k] == cmax for k >= K, c[k] <= cmax
// below), exact for w >= 0:
//   v[cd] = min( min_{|k|<K} a[cd+k] + w*c[|k|],  min_fd a[fd] + w*cmax )
// The second term is an upper bound for every label and is attained by all labels farther than the
// band from argmin(a); fp32 addition is monotone, so the values are bit-identical to the dense scan.
// KT > 0: KT - 1 taps with c[] in registers (KT >= K).  KT == 0: K at run time, taps in LDS.
// HEAD (band_head ran: KT >= 2 in registers, several labels per lane, no argmin labels): v, up and dn come in as the
// first tap left them, and the taps go on from the second.
template <int R, bool TRAIN, int KT, bool HEAD = false>
__device__ __forceinline__ void band_step(const float (&a)[R], float w, int K, const float* c_reg,
                                          const float* ctx_s, float cmax, float amin, int fstar,
                                          int lab0, float (&v)[R], int (&fd_idx)[R],
                                          const float* up_in = nullptr, const float* dn_in = nullptr) {
  static_assert(!HEAD || (KT >= 2 && !TRAIN), "the head covers the first tap of a band in registers");
  const float inf = INFINITY;
  float up[R], dn[R];
  int off[R];
  const float c0 = KT > 0 ? c_reg[0] : ctx_s[0];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    up[j] = HEAD ? up_in[j] : a[j];
    dn[j] = HEAD ? dn_in[j] : a[j];
    if (!HEAD) v[j] = fmaf(w, c0, a[j]);
    off[j] = 0;
  }
  // `refill`: up[0] / dn[R-1] still hold unshifted beliefs, so the vacated lane is set to +inf;
  // from tap R+1 on every vector has been through one such shift and the lane keeps its +inf
  auto tap = [&](int k, float ck, bool refill) {
    // one-label shifts: up[j] <- a[label + k], dn[j] <- a[label - k]
    float tu = refill ? wave_shl1(up[0], inf) : wave_shl1_keep(up[0]);
    float td = refill ? wave_shr1(dn[R - 1], inf) : wave_shr1_keep(dn[R - 1]);
#pragma unroll
    for (int j = 0; j < R - 1; ++j) up[j] = up[j + 1];
    up[R - 1] = tu;
#pragma unroll
    for (int j = R - 1; j > 0; --j) dn[j] = dn[j - 1];
    dn[0] = td;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      if (TRAIN) {
        float cu = fmaf(w, ck, up[j]);
        float cd = fmaf(w, ck, dn[j]);
        bool tk = cu <= v[j];  // larger front label wins ties
        v[j] = tk ? cu : v[j];
        off[j] = tk ? k : off[j];
        bool tk2 = cd < v[j];  // smaller front label loses ties
        v[j] = tk2 ? cd : v[j];
        off[j] = tk2 ? -k : off[j];
      } else {
        // x -> fma(w, ck, x) is monotone, so the smaller belief of the two gives the smaller
        // candidate: one multiply-add per tap and label, the same bits
        v[j] = fminf(v[j], fmaf(w, ck, fminf(up[j], dn[j])));
      }
    }
  };
  if (KT > 0) {
#pragma unroll
    for (int k = HEAD ? 2 : 1; k < KT; ++k) tap(k, c_reg[k], k <= R);
  } else {
    // R taps per trip: the R one-label rotations of up[] / dn[] then cancel, so the loop carries
    // no register moves, and the R coefficients are fetched from LDS together
    int k = 1;
    if (K > R) {
      float cc[R];
#pragma unroll
      for (int u = 0; u < R; ++u) cc[u] = ctx_s[1 + u];
#pragma unroll
      for (int u = 0; u < R; ++u) tap(1 + u, cc[u], true);
      k = 1 + R;
      for (; k + R <= K; k += R) {
#pragma unroll
        for (int u = 0; u < R; ++u) cc[u] = ctx_s[k + u];
#pragma unroll
        for (int u = 0; u < R; ++u) tap(k + u, cc[u], false);
      }
#pragma unroll
      for (int u = 0; u < R - 1; ++u)
        if (k + u < K) tap(k + u, ctx_s[k + u], false);
    } else {
#pragma unroll
      for (int u = 0; u < R - 1; ++u)
        if (1 + u < K) tap(1 + u, ctx_s[1 + u], true);
    }
  }
  const float far = fmaf(w, cmax, amin);
#pragma unroll
  for (int j = 0; j < R; ++j) {
    if (TRAIN) {
      int fb = lab0 + j + off[j];
      bool lt = far < v[j];
      bool eq = far == v[j];
      int fe = fb > fstar ? fb : fstar;
      fd_idx[j] = lt ? fstar : (eq ? fe : fb);
      v[j] = lt ? far : v[j];
    } else {
      v[j] = fminf(v[j], far);
    }
  }
}

// O(L log L / 64) step for truncated linear contexts c[k] = min(s*k, cmax) of any width, w >= 0.
// With t = w*s,
//   min_{fd <= cd} a[fd] + t*(cd - fd) =  t*cd + prefixmin_{fd <= cd} (a[fd] - t*fd)
//   min_{fd >= cd} a[fd] + t*(fd - cd) = -t*cd + suffixmin_{fd >= cd} (a[fd] + t*fd)
// so two scans over the labels find, for every cd, the best front label on either side; a label
// beyond the truncation can only win where the far candidate min(a) + w*cmax is at least as good.
// The scans run on rounded differences, so they only *select* the candidates (the largest label
// among equals on each side, as the reference's scan order does); the values are then evaluated
// from the table exactly as the dense scan does, a[fd] + w*c[|cd - fd|], and compared with the far
// candidate.  A selection off by the rounding of t*L picks a value within a few ulp of the largest
// belief of the true minimum.
template <int R, bool TRAIN>
__device__ __forceinline__ void linear_step(const float (&a)[R], float w, float slope, float cmax,
                                            float amin, int fstar, int lab0, int lane, int L,
                                            float* a_s, const float* ctx_s, float (&v)[R],
                                            int (&fd_idx)[R]) {
  const float inf = INFINITY;
  constexpr int big = 0x7fffffff;
  const float t = w * slope;
  float gm[R], gp[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const float l = (float)(lab0 + j);
    gm[j] = fmaf(-t, l, a[j]);
    gp[j] = fmaf(t, l, a[j]);
    a_s[lab0 + j] = a[j];  // staged for the gathers below
  }
  // left side: prefix minimum and its largest achiever (the largest label up to cd whose own
  // prefix minimum it is)
  float q[R], pl[R];
  q[0] = gm[0];
#pragma unroll
  for (int j = 1; j < R; ++j) q[j] = fminf(q[j - 1], gm[j]);
  const float before = wave_shr1(lane_prefix_min(q[R - 1]), inf);
  int qi[R], il[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    pl[j] = fminf(before, q[j]);
    const int f = (gm[j] == pl[j]) ? lab0 + j : -1;
    qi[j] = j == 0 ? f : max(qi[j > 0 ? j - 1 : 0], f);
  }
  const int before_i = dpp_i<0x138>(-1, lane_prefix_max(qi[R - 1]));  // lane i <- lane i-1
#pragma unroll
  for (int j = 0; j < R; ++j) il[j] = max(max(before_i, qi[j]), 0);
  // right side: suffix minimum; its largest achiever is where the plateau of that minimum ends
  float sfx[R], pr[R], nx[R];
  sfx[R - 1] = gp[R - 1];
#pragma unroll
  for (int j = R - 2; j >= 0; --j) sfx[j] = fminf(sfx[j + 1], gp[j]);
  const float after = wave_shl1(lane_suffix_min(sfx[0], lane), inf);
#pragma unroll
  for (int j = 0; j < R; ++j) pr[j] = fminf(after, sfx[j]);
#pragma unroll
  for (int j = 0; j < R - 1; ++j) nx[j] = pr[j + 1];
  nx[R - 1] = wave_shl1(pr[0], inf);
  int si[R], ir[R];
#pragma unroll
  for (int j = R - 1; j >= 0; --j) {
    const int b = (pr[j] < nx[j]) ? lab0 + j : big;
    si[j] = j == R - 1 ? b : min(si[j < R - 1 ? j + 1 : j], b);
  }
  const int after_i = dpp_i<0x130>(big, lane_suffix_min(si[0], lane));  // lane i <- lane i+1
#pragma unroll
  for (int j = 0; j < R; ++j) ir[j] = min(min(after_i, si[j]), L - 1);
  lds_order();  // a_s
  const float far = fmaf(w, cmax, amin);
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int cd = lab0 + j;
    const int kl = cd - il[j], kr = ir[j] - cd;
    const float vl = fmaf(w, ctx_s[kl < 0 ? 0 : (kl < L ? kl : L - 1)], a_s[il[j]]);
    const float vr = fmaf(w, ctx_s[kr < 0 ? 0 : kr], a_s[ir[j]]);
    const bool tr = vr <= vl;  // the larger front label wins ties
    float best = tr ? vr : vl;
    int arg = tr ? ir[j] : il[j];
    const bool lt = far < best, eq = far == best;
    if (TRAIN) fd_idx[j] = lt ? fstar : (eq ? (arg > fstar ? arg : fstar) : arg);
    v[j] = lt ? far : best;
  }
  lds_order();  // the next step overwrites a_s
}

}  // namespace
}  // namespace mpl

#endif  // MPLAYERS_AMD_MP_FWD_STEP_H_
