// TRWP scans for 21 labels with a 2-D table (the segmentation layers), four wavefronts per chain.  The
// recurrences and what each plane holds: mp_fwd.hip, mp_bwd.hip.
//
// Such a launch is bound by the length of one pixel's step: planes of a few megabytes, chains of some
// hundred pixels that a wavefront walks alone, and 21 of its 64 lanes at work.  As in mp_fwd_team.hip
// three helper wavefronts load the planes, put what the recurrence needs of a pixel into an LDS slot
// and, two blocks of pixels later, finish and store it; the main wavefront runs the recurrence out of
// LDS.  Here every wavefront uses both its halves (32 lanes each, label l in lane l and 32 + l):
//   * a helper has one pixel in each half, so that an instruction serves two pixels,
//   * the main wavefront holds the recurrence twice and splits what a label sums or searches over: the
//     lower half takes the source labels 0 .. 10, the upper one 11 .. 20, and one exchange of halves
//     joins them.  The 11 values reach the lanes as row broadcasts, a lane operand each, from a half's
//     source labels in lanes 0 .. 10 of both its rows.
// The forward step is then 11 multiply-adds and 5 minima in place of 21 and 10, and the argmin labels
// are left to the helpers, who compare the same 21 candidates with the minimum the main wavefront found.
// The reverse step adds up 11 gradients under masks (1 or 0 per pair of labels, from the helpers).
//
// A lone wavefront issues a 32-bit instruction every 4.2 clocks, one in the 64-bit encoding (lane operands
// among them) every 5.2, an exchange of rows or halves takes 8.2, an LDS access 10 to 14 (measured); by
// that count the forward step is 290 clocks and the reverse step 250.  Measured, ns per pixel of rows of 256 /
// 512 chains, one wavefront per chain -> this: 215 / 223 -> 143 / 145 without argmin labels, 340 / 347 -> 171 / 175
// with them.  4x129x129, 4 directions, 5 iterations, both other gradients wanted: backward 0.96 -> 0.65 ms, 0.59
// with a table of dcontext per die (dctx_table).
//
// Errors of the reverse scan against 64 bits, one wavefront -> four, geometric means of the relative 2-norm
// over 40 problems (images up to 130x130, 4 and 8 directions, 1 to 5 iterations; normal, positive and cross
// entropy gradients): dunary 1.52e-7 -> 1.35e-7, dcontext 5.0e-7 both, dedge_weights 1.79e-7 -> 1.63e-7.
// With longer chains, 36 problems of up to 2000 pixels a chain, by kind of gradient (normal / positive / cross
// entropy): dunary 1.23 / 1.07 / 1.07e-7 -> 1.17 / 0.96 / 1.10e-7, dcontext 6.1 / 4.7 / 5.7e-7 -> 5.4 / 4.7 / 4.9e-7,
// dedge_weights 1.28 / 1.19 / 1.32e-7 -> 1.24 / 1.09 / 1.34e-7; soft-weighted dunary 8.1 / 12.1 / 6.4e-8 -> 7.3 / 8.8 /
// 6.0e-8, dcontext 7.4 / 5.4 / 6.7e-7 -> 7.2 / 5.2 / 6.4e-7, dedge_weights 4.5 / 3.0 / 7.2e-7 -> 3.4 / 2.3 / 5.3e-7.
// Soft-weighted, 30 problems up to 100x100, 4 directions: 9.6e-8 -> 8.8e-8, 2.7e-7 both, 2.55e-7 -> 2.44e-7
// (dedge_weights 2.9e-7 to 3.6e-7 while the expected dual's own rounding was left in).  Its scans,
// 2x129x129, five iterations, duals kept: forward 1.44 -> 0.87 ms, bound by the main wavefront (11 exponentials and
// three exchanges of halves a pixel), reverse 2.03 -> 1.10 ms, by the helpers' softmin weights, 540 instructions for two
// pixels (650 while every weight was stored under a mask of its own, and the loads were waited for: keep).  Forward errors
// over 24 problems: messages 5.0e-7 -> 4.7e-7, costs 1.11e-7 -> 1.06e-7, duals 7.7e-8 ->
// 7.5e-8.

#include <type_traits>

#include "mp_fwd_step.h"

namespace mpl {
namespace {

constexpr int kL = 21;
constexpr int kHalf = 32;
constexpr int kSrc = 11;             // source labels per half (the upper half has one that does not exist)
constexpr int kHelpers = 3;          // one SIMD of the compute unit each, the main one the fourth
constexpr int kT = 2 * kHelpers;     // pixels per block
constexpr int kTeam = (kHelpers + 1) * kWave;
constexpr int kAhead = 2;            // blocks whose loads are in flight (four measure the same)
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kRow = 36;             // words between the pixels of a slot read by both halves at once

// workgroup barrier over LDS contents only: global loads in flight stay in flight
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// f(0) .. f(N - 1) with constant arguments
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(const F& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>());
    static_for<N, I + 1>(f);
  }
}

// A loaded value in a register of its own, moved there where it is first used.  The helpers keep some of what they
// load for a pixel until the pixel is finished; left to the compiler the two share a register and change places
// once per two blocks, with moves right behind the loads of the block after next that wait for all of them: the
// whole latency of memory, every twelve pixels.
template <typename T>
__device__ __forceinline__ T keep(T x) {
  T y;
  asm volatile("v_mov_b32 %0, %1" : "=v"(y) : "v"(x));
  return y;
}

__device__ __forceinline__ int bits(float x) { return __builtin_bit_cast(int, x); }
__device__ __forceinline__ float flt(int x) { return __builtin_bit_cast(float, x); }

// The scans want the labels of a half's sources in lanes 0 .. 10 of both its rows: the label a lane holds
// in that order, `source_label`, is an address to what comes from LDS; what is in registers by label (label
// l in lanes l and 32 + l) gets there by an exchange of rows and two shifts.
__device__ __forceinline__ int source_label(int lane) { return (lane / kHalf) * kSrc + (lane & 15); }

// Joins the two halves' minima over their source labels (best), and takes the minimum over all labels
// (nmin, in every lane).  v: the joint minima by label, src: the same by source label.  pad: +inf in the
// lanes of a row that hold no label 16 .. 20, -inf in the others.  The issue slots that a lane operand
// needs between its writing and its reading (two) hold the other chain's instructions.
__device__ __forceinline__ void join_min(float best, float pad, float& v, float& src, float& nmin) {
  float t, y;
  asm("v_mov_b32 %3, %0\n\t"
      "s_nop 1\n\t"
      "v_permlane32_swap_b32 %0, %3\n\t"
      "v_min_f32 %0, %0, %3\n\t"
      "v_mov_b32 %1, %0\n\t"
      "v_mov_b32 %4, %0\n\t"
      "s_nop 1\n\t"
      "v_permlane16_swap_b32 %1, %4\n\t"
      "v_max_f32 %3, %4, %5\n\t"
      "v_min_f32 %2, %1, %3\n\t"
      "v_mov_b32_dpp %1, %1 row_shl:11 row_mask:0xc bank_mask:0xf\n\t"
      "s_nop 0\n\t"
      "v_min_f32_dpp %2, %2, %2 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b32_dpp %1, %4 row_shr:5 row_mask:0xc bank_mask:0xf\n\t"
      "s_nop 0\n\t"
      "v_min_f32_dpp %2, %2, %2 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_min_f32_dpp %2, %2, %2 row_ror:2 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_min_f32_dpp %2, %2, %2 row_ror:1 row_mask:0xf bank_mask:0xf"
      : "+&v"(best), "=&v"(src), "=&v"(nmin), "=&v"(t), "=&v"(y)
      : "v"(pad));
  v = best;
}

// The same from the softmin messages by label, which are +inf in the lanes without one.
__device__ __forceinline__ void spread_min(float v, float& src, float& nmin) {
  float y;
  asm("v_mov_b32 %0, %3\n\t"
      "v_mov_b32 %2, %3\n\t"
      "s_nop 1\n\t"
      "v_permlane16_swap_b32 %0, %2\n\t"
      "v_min_f32 %1, %0, %2\n\t"
      "s_nop 0\n\t"
      "v_mov_b32_dpp %0, %0 row_shl:11 row_mask:0xc bank_mask:0xf\n\t"
      "s_nop 0\n\t"
      "v_min_f32_dpp %1, %1, %1 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b32_dpp %0, %2 row_shr:5 row_mask:0xc bank_mask:0xf\n\t"
      "s_nop 0\n\t"
      "v_min_f32_dpp %1, %1, %1 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_min_f32_dpp %1, %1, %1 row_ror:2 row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1\n\t"
      "v_min_f32_dpp %1, %1, %1 row_ror:1 row_mask:0xf bank_mask:0xf"
      : "=&v"(src), "=&v"(nmin), "=&v"(y)
      : "v"(v));
}

// The reverse step.  m[0 .. 10] are the masks of a lane's label, m[11] is 1 where it is the argmin label of
// the normalisation's label.  With DC the sums of dcontext by pair of source label and label (pairs: source
// label q of the half, the lane's label) are kept by the main wavefront: gw, the gradient times the edge
// weight, under the same masks.  Those multiply-adds stand in the issue slots that the exchanges and lane
// shifts of the recurrence leave idle, the first four of them a pixel late.

// x by label -> by source label.  zero: becomes NaN where gw is not finite
template <bool DC>
__device__ __forceinline__ float to_sources(float x, float gw, const f32x4& m0, float (&pairs)[kSrc], float& zero) {
  float y;
  if constexpr (DC) {
    // (a lane operand may be read two issue slots after it was written, and the compiler does not look into
    // the block for it: the first two instructions leave that of gw alone)
    asm("v_mov_b32 %1, %0\n\t"
        "v_fmac_f32 %6, 0, %7\n\t"
        "v_fmac_f32_dpp %2, %7, %8 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %3, %7, %9 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_permlane16_swap_b32 %0, %1\n\t"
        "v_fmac_f32_dpp %4, %7, %10 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %5, %7, %11 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
        "v_mov_b32_dpp %0, %0 row_shl:11 row_mask:0xc bank_mask:0xf\n\t"
        "v_mov_b32_dpp %0, %1 row_shr:5 row_mask:0xc bank_mask:0xf"
        : "+&v"(x), "=&v"(y), "+&v"(pairs[0]), "+&v"(pairs[1]), "+&v"(pairs[2]), "+&v"(pairs[3]), "+&v"(zero)
        : "v"(gw), "v"(m0[0]), "v"(m0[1]), "v"(m0[2]), "v"(m0[3]));
  } else {
    asm("v_mov_b32 %1, %0\n\t"
        "s_nop 1\n\t"
        "v_permlane16_swap_b32 %0, %1\n\t"
        "s_nop 1\n\t"
        "v_mov_b32_dpp %0, %0 row_shl:11 row_mask:0xc bank_mask:0xf\n\t"
        "v_mov_b32_dpp %0, %1 row_shr:5 row_mask:0xc bank_mask:0xf"
        : "+&v"(x), "=&v"(y));
  }
  return x;
}

// Sums the gradients g (by source label) under the masks, less the sum of all of them (tot: of the half's
// sources) where m[11] says so, over both halves.  src_mask: all ones in the lanes of source labels, zero
// in the others.
template <bool DC>
__device__ __forceinline__ float masked_sums(float g, float gw, const f32x4 (&m)[3], int src_mask, float& tot,
                                             float (&pairs)[kSrc]) {
  float x, y;
#define MPL_SUMS_HEAD \
  "v_and_b32 %[t], %[k], %[g]\n\ts_nop 0\n\t" \
  "v_mul_f32_dpp %[x], %[g], %[m0] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t" \
  "v_mul_f32_dpp %[y], %[g], %[m1] row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t" \
  "v_add_f32_dpp %[t], %[t], %[t] row_ror:8 row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %[x], %[g], %[m2] row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %[y], %[g], %[m3] row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t" \
  "v_add_f32_dpp %[t], %[t], %[t] row_ror:4 row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %[x], %[g], %[m4] row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %[y], %[g], %[m5] row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t" \
  "v_add_f32_dpp %[t], %[t], %[t] row_ror:2 row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %[x], %[g], %[m6] row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %[y], %[g], %[m7] row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t" \
  "v_add_f32_dpp %[t], %[t], %[t] row_ror:1 row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %[x], %[g], %[m8] row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %[y], %[g], %[m9] row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %[x], %[g], %[m10] row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t" \
  "v_fma_f32 %[y], -%[n], %[t], %[y]\n\t" \
  "v_add_f32 %[x], %[x], %[y]\n\t" \
  "v_mov_b32 %[y], %[x]\n\t"
#define MPL_SUMS_IN                                                                                                  \
  [g] "v"(g), [k] "v"(src_mask), [m0] "v"(m[0][0]), [m1] "v"(m[0][1]), [m2] "v"(m[0][2]), [m3] "v"(m[0][3]),           \
      [m4] "v"(m[1][0]), [m5] "v"(m[1][1]), [m6] "v"(m[1][2]), [m7] "v"(m[1][3]), [m8] "v"(m[2][0]), [m9] "v"(m[2][1]), \
      [m10] "v"(m[2][2]), [n] "v"(m[2][3])
#define MPL_PAIR(N) "v_fmac_f32_dpp %[p" #N "], %[w], %[m" #N "] row_newbcast:" #N " row_mask:0xf bank_mask:0xf\n\t"
  if constexpr (DC) {
    asm(MPL_SUMS_HEAD MPL_PAIR(4) MPL_PAIR(5)
        "v_permlane32_swap_b32 %[x], %[y]\n\t"
        MPL_PAIR(6) MPL_PAIR(7) MPL_PAIR(8) MPL_PAIR(9) MPL_PAIR(10)
        "v_add_f32 %[x], %[x], %[y]"
        : [x] "=&v"(x), [y] "=&v"(y), [t] "=&v"(tot), [p4] "+&v"(pairs[4]), [p5] "+&v"(pairs[5]), [p6] "+&v"(pairs[6]),
          [p7] "+&v"(pairs[7]), [p8] "+&v"(pairs[8]), [p9] "+&v"(pairs[9]), [p10] "+&v"(pairs[10])
        : MPL_SUMS_IN, [w] "v"(gw));
  } else {
    asm(MPL_SUMS_HEAD "s_nop 1\n\t"
        "v_permlane32_swap_b32 %[x], %[y]\n\t"
        "v_add_f32 %[x], %[x], %[y]"
        : [x] "=&v"(x), [y] "=&v"(y), [t] "=&v"(tot)
        : MPL_SUMS_IN);
  }
#undef MPL_PAIR
#undef MPL_SUMS_IN
#undef MPL_SUMS_HEAD
  return x;
}

// lane N of every row, in all its lanes
template <int N>
__device__ __forceinline__ float row_bcast(float x) {
  return flt(__builtin_amdgcn_mov_dpp(bits(x), 0x150 + N, 0xf, 0xf, true));
}
// lower half of x in both halves, upper half of x in both halves
__device__ __forceinline__ void halves(float x, float& lower, float& upper) {
  const auto r = __builtin_amdgcn_permlane32_swap((unsigned)bits(x), (unsigned)bits(x), false, false);
  lower = flt((int)r[0]);
  upper = flt((int)r[1]);
}

// sums over the lanes of each half, in its last lane
__device__ __forceinline__ float half_sum(float x) {
#define MPL_ADD_DPP(CTRL) "s_nop 1\n\tv_add_f32_dpp %0, %0, %0 " CTRL " bank_mask:0xf\n\t"
  asm(MPL_ADD_DPP("row_shr:1 row_mask:0xf") MPL_ADD_DPP("row_shr:2 row_mask:0xf")
      MPL_ADD_DPP("row_shr:4 row_mask:0xf") MPL_ADD_DPP("row_shr:8 row_mask:0xf")
      MPL_ADD_DPP("row_bcast:15 row_mask:0xa") "s_nop 0"
      : "+v"(x));
#undef MPL_ADD_DPP
  return x;
}

// ---- forward ---------------------------------------------------------------------------------------
struct alignas(16) FwdSlots {   // one set
  float in[kT][kHalf][2];       // U, edge weight
  float a[kT][kRow];            // beliefs the pixel's message comes from (argmin labels kept)
  float out[kT][kHalf][2];      // v and the normalisation minimum; without argmin labels the message
};

// SOFT: the soft-weighted operator.  The main wavefront takes each half's softmin sums around the joint
// minimum; where the duals are kept (TRAIN) the helpers form a pixel's block again from its beliefs, 64
// entries to a store.
template <bool TRAIN, bool SOFT>
__global__ void __launch_bounds__(kTeam) fwd_team21_kernel(const SweepParams p) {
  extern __shared__ __align__(16) char smem_raw[];
  FwdSlots* sets = reinterpret_cast<FwdSlots*>(smem_raw);  // two
  const int tid = threadIdx.x;
  // (the last wavefront: mp_fwd_team.hip)
  const int role = uniform_i(tid / kWave);  // kHelpers: main
  const int lane = tid & (kWave - 1);
  const int l = lane & (kHalf - 1);
  const int half = lane / kHalf;
  const bool ok = l < kL;
  const ChainCtx ch0 = locate_chain(p);
  const int n = ch0.n;
  const float rho = p.rho;
  const int blocks = (n + kT - 1) / kT;
  const int iters = (blocks + 2 + kAhead - 1) / kAhead * kAhead;
  const float floor_l = ok ? -INFINITY : INFINITY;
  auto table = [&](int fd) __attribute__((always_inline)) {  // ctx(l, fd), TRWP_forward.cu:101-113
    const int cd = ok ? l : kL - 1, f = fd < kL ? fd : kL - 1;
    return p.ctx[cd < f ? cd * kL + f : f * kL + cd];
  };

  auto main_walk = [&]() __attribute__((always_inline)) {
    float tc[kSrc];
#pragma unroll
    for (int i = 0; i < kSrc; ++i) tc[i] = table(half * kSrc + i);
    const int sl = source_label(lane);
    const float pad = (lane & 15) < kL - 16 ? -INFINITY : INFINITY;
    float prev = 0.f, uf = 0.f;  // message and U of the front pixel, by source label
    for (int k = 0; k < iters; ++k) {
      if (k >= 1 && k <= blocks) {
        FwdSlots& s = sets[(k - 1) & 1];
        // (two pixels to an LDS instruction, as in mp_fwd_team.hip: 1 to 2 % of a scan of rows of 129; the reverse scan,
        // whose masks are most of what it reads, has nothing from it)
        f32x2 two[2], nxt[2], out[2];
        float as[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) two[u] = *reinterpret_cast<const f32x2*>(s.in[u][sl]);
#pragma unroll
        for (int i = 0; i < kT; ++i) {
          const int u = i & 1;
          if (u == 0 && i + 2 < kT) {
#pragma unroll
            for (int j = 0; j < 2; ++j) nxt[j] = *reinterpret_cast<const f32x2*>(s.in[i + 2 + j][sl]);
          }
          const f32x2 cur = two[u];
          const float a = fmaf(rho, prev, uf);
          as[u] = a;
          float c[kSrc];
          static_for<kSrc>([&](auto ii) __attribute__((always_inline)) {
            constexpr int q = decltype(ii)::value;
            c[q] = fmaf(cur[1], tc[q], row_bcast<q>(a));
          });
          float v, vs, nmin;
          if (SOFT) c[kSrc - 1] = half ? c[0] : c[kSrc - 1];  // (the upper half's last source does not exist)
          const float best = fminf(fminf(fminf(fminf(c[0], c[1]), c[2]), fminf(fminf(c[3], c[4]), c[5])),
                                   fminf(fminf(fminf(c[6], c[7]), c[8]), fminf(c[9], c[10])));
          if constexpr (SOFT) {
            // TRWP_forward_soft.cu:81-97, the duals relative to the least one
            float lower, upper;
            halves(best, lower, upper);
            const float mn = fminf(lower, upper);
            float se[2] = {0.f, 0.f}, sd[2] = {0.f, 0.f};
#pragma unroll
            for (int q = 0; q < kSrc; ++q) {
              const float d = c[q] - mn;
              float e = __builtin_amdgcn_exp2f(d * -kLog2e);
              if (q == kSrc - 1) e = half ? 0.f : e;
              se[q & 1] += e;
              sd[q & 1] = fmaf(e, d, sd[q & 1]);
            }
            float se_l, se_u;
            halves(se[0] + se[1], se_l, se_u);
            halves(sd[0] + sd[1], lower, upper);
            v = fmaf(lower + upper, __builtin_amdgcn_rcpf(se_l + se_u), mn);
            v = ok ? v : INFINITY;
            spread_min(v, vs, nmin);
          } else {
            join_min(best, pad, v, vs, nmin);
          }
          prev = (i == 0 && k == 1) ? 0.f : vs - nmin;  // (the chain start has no front pixel and no message)
          out[u] = (TRAIN || SOFT) ? f32x2{v, nmin} : f32x2{prev, 0.f};
          uf = cur[0];
          if (u == 1) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              if (TRAIN) s.a[i - 1 + j][sl] = as[j];
              if (TRAIN || SOFT)
                *reinterpret_cast<f32x2*>(s.out[i - 1 + j][l]) = out[j];
              else
                s.out[i - 1 + j][sl][0] = out[j][0];
              two[j] = nxt[j];
            }
          }
        }
      }
      lds_barrier();
    }
  };

  const int64_t HW = (int64_t)p.H * p.W;
  const int64_t P = (int64_t)p.B * HW;
  const int64_t N = P * kL;

  // even_walk: a constant; the first (even direction) or the second sweep of a pair (run_chain_fwd)
  auto helper_walk = [&](const ChainCtx& ch, const bool skip_s_in, const auto even_walk)
      __attribute__((always_inline)) {
    constexpr bool EVEN = SOFT || decltype(even_walk)::value;  // (soft-weighted: every sweep stores S)
    const int dir = ch.dir;
    const int64_t img_p = (int64_t)ch.bv * HW;
    const int64_t img_e = img_p * kL;
    const bool known = p.desc != nullptr && p.desc->msg_nonzero == 0;  // the initial messages are zero
    const bool zfirst = p.zero_first && known;
    const bool skip_s = skip_s_in || (EVEN && zfirst);
    const bool md_zero = p.first_iter && known;
    const bool mi_zero = md_zero && EVEN;
    const int img_bytes = (int)(unsigned)(HW * kL * 4);
    const rsrc_t rS = make_rsrc((zfirst ? p.belief_zero : p.belief) + img_e, img_bytes);
    const rsrc_t rMd = make_rsrc(p.msg_in + (int64_t)dir * N + img_e, md_zero ? 0 : img_bytes);
    const rsrc_t rMi = make_rsrc(p.msg_in + (int64_t)(dir ^ 1) * N + img_e, mi_zero ? 0 : img_bytes);
    const rsrc_t rMo = make_rsrc(p.msg_out + (int64_t)dir * N + img_e, img_bytes);
    const rsrc_t rSo = make_rsrc(p.belief_out + img_e, skip_s ? 0 : img_bytes);
    constexpr bool ARGMIN = TRAIN && !SOFT;
    const rsrc_t rImin = make_rsrc(ARGMIN ? p.idx_min + (int64_t)dir * N + img_e : nullptr, ARGMIN ? (int)(HW * kL) : 0);
    const rsrc_t rInorm = make_rsrc(TRAIN ? p.idx_norm + (int64_t)dir * P + img_p : nullptr, TRAIN ? (int)HW : 0);
    const rsrc_t rW = make_rsrc(p.edge + (int64_t)dir * P + img_p, (int)(HW * 4));
    // the entries lane + 64 j of a block of duals, [front label][label] in even directions, [label][front label] in
    // odd ones (TRWP_forward_soft.cu:64): the table is symmetric, so they differ in whose belief they add
    constexpr int kEntries = (kL * kL + kWave - 1) / kWave;
    float tblk[SOFT && TRAIN ? kEntries : 1];
    int ablk[SOFT && TRAIN ? kEntries : 1];
    float* const duals = SOFT && TRAIN ? p.edge_label + ((int64_t)dir * P + img_p) * (kL * kL) : nullptr;
    if constexpr (SOFT && TRAIN) {
#pragma unroll
      for (int j = 0; j < kEntries; ++j) {
        const int e = lane + kWave * j < kL * kL ? lane + kWave * j : kL * kL - 1;
        const int row = e / kL, col = e - row * kL;
        tblk[j] = keep(p.ctx[row < col ? row * kL + col : col * kL + row]);  // (waited for here, not in the loop)
        ablk[j] = (dir & 1) ? col : row;
      }
    }
    float tcol[ARGMIN ? kL : 1];
    if constexpr (ARGMIN) {
#pragma unroll
      for (int fd = 0; fd < kL; ++fd) tcol[fd] = table(fd);
    }
    const int i = 2 * role + half;  // the pixel of a block in this half
    struct Pix {
      float s, md, mi, w;
    };
    auto pixel_off = [&](const int t) __attribute__((always_inline)) { return (unsigned)(ch.pix0 + t * ch.pstep); };
    auto label_off = [&](const bool on, const unsigned pp) __attribute__((always_inline)) {
      return (int)((on && ok) ? (pp * (unsigned)kL + (unsigned)l) * 4u : kDeadWide);
    };
    auto load = [&](rsrc_t r, int off) __attribute__((always_inline)) {
      return flt((int)__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
    };
    auto store = [&](rsrc_t r, int off, float x) __attribute__((always_inline)) {
      __builtin_amdgcn_raw_buffer_store_b32((unsigned)bits(x), r, off, 0, 0);
    };
    // the loads of chain position t (nothing is read past the end of the chain)
    auto load_pix = [&](const int t) __attribute__((always_inline)) {
      Pix r;
      const bool on = t < n;
      const unsigned pp = pixel_off(t);
      const int off = label_off(on, pp);
      r.s = load(rS, off);
      r.md = 0.f;
      if (EVEN) r.md = load(rMd, off);
      r.mi = load(rMi, off);
      r.w = load(rW, (int)(on ? pp * 4u : kDeadWide));
      return r;
    };
    // second sweep: the old message of the chain start
    float md0 = 0.f;
    if (!EVEN) md0 = load(rMd, label_off(i == 0, pixel_off(0)));

    float tt[2] = {0.f, 0.f}, ww[2] = {0.f, 0.f};
    auto prepare = [&](const Pix& px, const int t, FwdSlots& s, float& tk, float& wk) __attribute__((always_inline)) {
      tk = EVEN ? px.s - px.md : px.s + px.mi;
      float un = fmaf(tk, rho, -px.mi);  // UpdateUnaryKernel, TRWP_forward.cu:70-78
      if (!SOFT) un = fmaxf(un, floor_l);
      wk = SOFT && TRAIN ? keep(px.w) : px.w;
      *reinterpret_cast<f32x2*>(s.in[i][l]) = f32x2{un, px.w};
      // Q of the pixel is known already, whatever its message
      if (EVEN && !SOFT) store(rSo, label_off(t < n, pixel_off(t)), tk - px.mi);
    };
    // what is left of a pixel once its message is known (nothing outside the chain)
    auto finish = [&](const int t, const FwdSlots& s, const float tk, const float wk) __attribute__((always_inline)) {
      const bool on = t >= 0 && t < n;
      const bool step = t > 0 && t < n;
      const unsigned pp = pixel_off(t);
      const int off = label_off(on, pp);
      float m;
      if constexpr (SOFT) {
        const f32x2 o = *reinterpret_cast<const f32x2*>(s.out[i][l]);
        m = o[0] - o[1];
        if constexpr (TRAIN) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {  // the pixel of either half
            const int th = uniform_i(t - half) + h;
            const bool live = th > 0 && th < n;
            const float w = flt(__builtin_amdgcn_readlane(bits(wk), h * kHalf));
            const rsrc_t rBlk = make_rsrc(duals + (live ? (int64_t)pixel_off(th) * (kL * kL) : 0), live ? kL * kL * 4 : 0);
#pragma unroll
            for (int j = 0; j < kEntries; ++j)
              store(rBlk, (lane + kWave * j) * 4, fmaf(w, tblk[j], s.a[2 * role + h][ablk[j]]));
          }
          const uint64_t at = ballot(ok && o[0] == o[1]);
          const unsigned lo = (unsigned)at, hi = (unsigned)(at >> 32);
          const int n0 = lo ? 31 - __builtin_clz(lo) : kL - 1, n1 = hi ? 31 - __builtin_clz(hi) : kL - 1;
          __builtin_amdgcn_raw_buffer_store_b8((unsigned char)(half ? n1 : n0), rInorm,
                                               (int)((step && l == 0) ? pp : kDeadWide), 0, 0);
        }
      } else if constexpr (TRAIN) {
        const f32x2 o = *reinterpret_cast<const f32x2*>(s.out[i][l]);
        float val[kL];
#pragma unroll
        for (int q = 0; q < 5; ++q) {
          const f32x4 x = *reinterpret_cast<const f32x4*>(&s.a[i][4 * q]);
#pragma unroll
          for (int z = 0; z < 4; ++z) val[4 * q + z] = fmaf(wk, tcol[4 * q + z], x[z]);
        }
        val[20] = fmaf(wk, tcol[20], s.a[i][20]);
        int arg;
        float unused = 0.f;
        argmin_and_lane_min_21(val, o[0], unused, arg);
        const uint64_t at = ballot(ok && o[0] == o[1]);
        const unsigned lo = (unsigned)at, hi = (unsigned)(at >> 32);
        const int n0 = lo ? 31 - __builtin_clz(lo) : kL - 1, n1 = hi ? 31 - __builtin_clz(hi) : kL - 1;
        m = t == 0 ? 0.f : o[0] - o[1];
        __builtin_amdgcn_raw_buffer_store_b8((unsigned char)arg, rImin,
                                             (int)((step && ok) ? pp * (unsigned)kL + (unsigned)l : kDeadWide), 0, 0);
        __builtin_amdgcn_raw_buffer_store_b8((unsigned char)(half ? n1 : n0), rInorm,
                                             (int)((step && l == 0) ? pp : kDeadWide), 0, 0);
      } else {
        m = s.out[i][l][0];
      }
      // (the reference never writes the chain start)
      store(rMo, (step || (!SOFT && p.zero_start)) ? off : (int)kDeadWide, m);
      if constexpr (SOFT) store(rSo, step ? off : (int)kDeadWide, tk + m);
      if constexpr (!EVEN) store(rSo, off, tk + (t == 0 ? md0 : m));
    };

    Pix ring[kAhead];
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
      ring[q] = load_pix(q * kT + i);
      MPL_ORDER_LOADS();
    }
#pragma clang loop unroll(disable)
    for (int k0 = 0; k0 < iters; k0 += kAhead) {
#pragma unroll
      for (int q = 0; q < kAhead; ++q) {
        const int k = k0 + q;
        FwdSlots& s = sets[q & 1];
        finish((k - 2) * kT + i, s, tt[q & 1], ww[q & 1]);
        lds_order();
        prepare(ring[q], k * kT + i, s, tt[q & 1], ww[q & 1]);
        ring[q] = load_pix((k + kAhead) * kT + i);
        lds_barrier();
      }
    }
  };

  // the second sweep of a pair reads what the first one's helpers stored: on the same compute unit,
  // once their stores are complete
  if (role == kHelpers) {
    __builtin_amdgcn_s_setprio(3);
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

// ---- backward --------------------------------------------------------------------------------------
template <int kT>
struct alignas(16) BwdSlots {   // one set
  float mask[kT][2][kL][12];    // per half's sources and label: 1 where the source label points at the
                                // label, else 0; last: 1 where the normalisation's argmin label is the label
  float base[kT][kHalf][2];     // gradient of the message without what the recurrence adds; the edge weight,
                                // 0 where the pixel has no incoming edge
  float sc[kT][kHalf];          // dU of the pixel (main wavefront)
  float tot[kT][2];             // sums of the message's gradient over a half's sources (main wavefront)
  int fd[kT][kHalf];            // argmin labels
};
constexpr int kPairs = kL * kL;

// Helpers of the soft-weighted scan where every chain has a compute unit to itself: the fourth SIMD, the main
// wavefront's in the other launches, takes two of them.  More chains fill the SIMDs with three each.  Rows of 129 pixels,
// all gradients, us per pair of walks with three / six: 128 chains 90 / 76, 256 chains 95 / 81, 258 chains 111 / 145, 512 chains 117 / 153.
// The hard scan gains where dcontext is wanted and the LDS holds every chain of a unit: 128 chains 47.5 / 43.7, 256 chains
// 46.5 / 42.7, 400 chains 50 / 47, 512 chains 51 / 47, 516 chains 59 / 82; without dcontext 0.97 to 1.05 of the time.
constexpr int kManyHelpers = 6;

// GR: dedge_weights and / or dcontext are wanted; DC: dcontext is.  SOFT: the soft-weighted operator, whose
// step has the same form with J[cd][fd] = d message(cd) / d belief(fd) in place of the masks: the helpers
// read a pixel's duals, take the softmin weights of a label over its front labels and put J into the slot.
template <bool GR, bool DC, bool SOFT, int kHelpers>
__global__ void __launch_bounds__((kHelpers + 1) * kWave) bwd_team21_kernel(const BackParams p) {
  constexpr int kT = 2 * kHelpers, kTeam = (kHelpers + 1) * kWave;
  using Slots = BwdSlots<kT>;
  extern __shared__ __align__(16) char smem_raw[];
  Slots* sets = reinterpret_cast<Slots*>(smem_raw);  // two
  float* acc = reinterpret_cast<float*>(sets + 2);         // kMaxL
  float* ctx_s = acc + kMaxL;                              // the table, then dcontext of the chain
  float* hist_s = ctx_s + kPairs;
  const int tid = threadIdx.x;
  // kHelpers: main, the fourth wavefront (the last of four: mp_fwd_team.hip; of seven the one whose SIMD has no other)
  const int wave = uniform_i(tid / kWave);
  const int role = wave == 3 ? kHelpers : wave - (wave > 3 ? 1 : 0);
  const int lane = tid & (kWave - 1);
  const int l = lane & (kHalf - 1);
  const int half = lane / kHalf;
  const bool ok = l < kL;
  const ChainCtx ch0 = locate_chain<false>(p);
  const int n = ch0.n;
  const float rho = p.rho;
  const int blocks = (n + kT - 1) / kT;
  const int iters = (blocks + 2 + kAhead - 1) / kAhead * kAhead;
  const bool want_de = GR && p.dedge != nullptr;
  const bool same = SOFT || p.same_label != 0;
  if (tid < kMaxL) acc[tid] = 0.f;
  if (GR) {
    for (int i = tid; i < kPairs; i += kTeam) ctx_s[i] = p.ctx[i];
    for (int i = tid; i < kPairs; i += kTeam) hist_s[i] = 0.f;
  }
  __syncthreads();

  float pairs[kSrc];  // (main wavefront) dcontext: source label half * kSrc + q, label l
#pragma unroll
  for (int q = 0; q < kSrc; ++q) pairs[q] = 0.f;
  auto main_walk = [&]() __attribute__((always_inline)) {
    const int sl = source_label(lane);
    const int src_mask = (lane & 15) < kSrc && sl < kL ? -1 : 0;
    const int ok_mask = ok ? -1 : 0;
    const int lm = ok ? l : kL - 1;  // (a lane without a label repeats the last one's sums: nothing reads them)
    float sc = 0.f;
    struct In {
      f32x4 m[3];
      f32x2 b;
    };
    auto get = [&](const Slots& s, const int i) __attribute__((always_inline)) {
      In x;
#pragma unroll
      for (int q = 0; q < 3; ++q) x.m[q] = *reinterpret_cast<const f32x4*>(&s.mask[i][half][lm][4 * q]);
      x.b = *reinterpret_cast<const f32x2*>(s.base[i][sl]);
      return x;
    };
    // A block of pixels whose gradients, or their products with the edge weight, are not all finite, one after
    // another: a zero mask does not switch such a term off, so the gradients go to their labels through LDS.
    // (What the normalisation takes off stays a term of its own: where the weight is not finite, that entry of
    // dcontext can be NaN here and infinite with one wavefront per chain.)
    auto careful_block = [&](Slots& s, const int k) __attribute__((always_inline)) {
#pragma clang loop unroll(disable)
      for (int i = 0; i < kT; ++i) {
        const In cur = get(s, i);
        s.sc[i][l] = sc;
        float none[kSrc], nothing;
        const float g = fmaf(rho, to_sources<false>(sc, 0.f, cur.m[0], none, nothing), cur.b[0]);
        if (src_mask != 0 && (lane & 16) == 0) atomicAdd(&acc[s.fd[i][sl]], g);
        lds_order();
        sc = acc[l];
        lds_order();
        acc[lane] = 0.f;
        lds_order();
        float tot = src_mask != 0 ? g : 0.f, lower, upper;
        tot += dpp_f<0x128>(0.f, tot);  // row_ror: 8, 4, 2, 1
        tot += dpp_f<0x124>(0.f, tot);
        tot += dpp_f<0x122>(0.f, tot);
        tot += dpp_f<0x121>(0.f, tot);
        halves(tot, lower, upper);
        if (cur.m[2][3] != 0.f) sc -= lower + upper;
        if (GR) s.tot[i][half] = tot;
        if (DC && n - 1 - ((k - 1) * kT + i) >= 1) {
          const float gwi = cur.b[1] * g;
          static_for<kSrc>([&](auto ii) __attribute__((always_inline)) {
            constexpr int q = decltype(ii)::value;
            const float x = row_bcast<q>(gwi);
            pairs[q] += bits(cur.m[q / 4][q % 4]) != 0 ? x : 0.f;
          });
        }
      }
    };
    float gw = 0.f;  // of the pixel before, whose first four pairs are still to be added
    f32x4 m0 = {0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < iters; ++k) {
      if (k >= 1 && k <= blocks) {
        Slots& s = sets[(k - 1) & 1];
        In cur = get(s, 0);
        const float sc_was = sc;
        float pairs_were[kSrc], zero = 0.f;
        if (DC) {
          static_for<4>([&](auto ii) __attribute__((always_inline)) {
            constexpr int q = decltype(ii)::value;
            pairs[q] = fmaf(row_bcast<q>(gw), m0[q], pairs[q]);
          });
          gw = 0.f;
#pragma unroll
          for (int q = 0; q < kSrc; ++q) pairs_were[q] = pairs[q];
        }
#pragma unroll
        for (int i = 0; i < kT; ++i) {
          In nxt = cur;
          if (i + 1 < kT) nxt = get(s, i + 1);
          s.sc[i][l] = sc;
          // gradient w.r.t. the normalised message of this pixel, including what the previous step
          // added through the recurrence (dmsg[front] += rho * value, TRWP_backward.cu:108)
          float g = fmaf(rho, to_sources<DC>(sc, gw, m0, pairs, zero), cur.b[0]);
          // The chain start has no message, and neither have the places of the block past it: without a gradient
          // there, the sums and dcontext stay what they are (a zero weight would not do: zero times what is
          // not finite)
          if (SOFT) g = flt(bits(g) & ((k - 1) * kT + i < n - 1 ? -1 : 0));
          if (DC) {
            gw = cur.b[1] * g;
            m0 = cur.m[0];
          }
          float tot;
          // MsgNormNaiveBack (commonCUDA.cuh:131-145) through the argmin label of its label
          sc = masked_sums<DC>(g, gw, cur.m, src_mask, tot, pairs);
          // (weights are not masks: what is not finite reaches every label by itself, but not from the
          // lanes without one)
          if (SOFT) sc = flt(bits(sc) & ok_mask);
          if (GR) s.tot[i][half] = tot;
          cur = nxt;
        }
        // an infinity or a NaN in any gradient makes NaN of every sum of its pixel and of all after it
        // (tested as an integer: the compiler may take NaN for anything)
        int probe = SOFT ? 0 : uniform_i(bits(sc));
        asm("" : "+s"(probe));
        bool odd_sums = !SOFT && (probe & 0x7f800000) == 0x7f800000;
        if constexpr (!SOFT && DC) {
          // ... and so does one in a gradient times the edge weight with the pairs' sums (an integer, again)
          int z = bits(zero);
          asm("v_fmac_f32 %0, 0, %1" : "+v"(z) : "v"(gw));
          odd_sums |= ballot(z != 0) != 0;
        }
        if (!SOFT && __builtin_expect(odd_sums, 0)) {
          sc = sc_was;
          if (DC) {
            gw = 0.f;
#pragma unroll
            for (int q = 0; q < kSrc; ++q) pairs[q] = pairs_were[q];
          }
          careful_block(s, k);
        }
      }
      lds_barrier();
    }
    if (DC) {
      static_for<4>([&](auto ii) __attribute__((always_inline)) {
        constexpr int q = decltype(ii)::value;
        pairs[q] = fmaf(row_bcast<q>(gw), m0[q], pairs[q]);
      });
    }
  };

  // even_walk: a constant; which of the two walks of a pair this is (mp_bwd.hip)
  auto helper_walk = [&](const ChainCtx& ch, const auto even_walk, const float* a_in, const bool first_touch)
      __attribute__((always_inline)) {
    constexpr bool EVEN = !SOFT && decltype(even_walk)::value;
    const int dir = ch.dir;
    const int64_t HW = (int64_t)p.H * p.W;
    const int64_t P = (int64_t)p.B * HW;
    const int64_t N = P * kL;
    const int64_t img_p = (int64_t)ch.bv * HW;
    const int64_t img_e = img_p * kL;
    float* bHd = p.h + (int64_t)dir * N + img_e;
    float* bHi = p.h + (int64_t)(dir ^ 1) * N + img_e;
    const int img_bytes = (int)(unsigned)(HW * kL * 4);
    const rsrc_t rA = make_rsrc(a_in + img_e, img_bytes);
    const rsrc_t rAo = make_rsrc(EVEN || SOFT ? p.a_out + img_e : bHd, img_bytes);
    const rsrc_t rHdIn = make_rsrc(bHd, !first_touch ? img_bytes : 0);
    const rsrc_t rHiIn = make_rsrc(bHi, EVEN || (SOFT && !first_touch) ? img_bytes : 0);
    const rsrc_t rHdOut = make_rsrc(bHd, SOFT ? img_bytes : 0);
    const rsrc_t rHiOut = make_rsrc(bHi, SOFT || (EVEN && !p.skip_h_store) ? img_bytes : 0);
    // the duals of a pixel: even directions [fd][cd], odd ones [cd][fd] (TRWP_forward_soft.cu:64); a lane takes
    // those of its label and its half's front labels
    const float* duals = SOFT ? p.edge_label + ((int64_t)dir * P + img_p) * kPairs : nullptr;
    const bool front_first = (dir & 1) == 0;
    const rsrc_t rImin = make_rsrc(SOFT ? nullptr : p.idx_min + (int64_t)dir * N + img_e, SOFT ? 0 : (int)(HW * kL));
    const rsrc_t rInorm = make_rsrc(p.idx_norm + (int64_t)dir * P + img_p, (int)HW);
    const rsrc_t rW = make_rsrc(p.edge + (int64_t)dir * P + img_p, (int)(HW * 4));
    const rsrc_t rDe = make_rsrc(want_de ? p.dedge + (int64_t)dir * P + img_p : nullptr, want_de ? (int)(HW * 4) : 0);
    const int p_last = ch.pix0 + (n - 1) * ch.pstep;
    const int i = 2 * role + half;  // the pixel of a block in this half
    const int sl = source_label(lane);
    struct Pix {
      float a, hd, hi, w, de;
      float dual[SOFT ? 2 : 1][kSrc];  // of both halves' pixels
      int fd, nidx;
    };
    auto label_off = [&](const bool on, const unsigned pp) __attribute__((always_inline)) {
      return (int)((on && ok) ? (pp * (unsigned)kL + (unsigned)l) * 4u : kDeadWide);
    };
    auto load = [&](rsrc_t r, int off) __attribute__((always_inline)) {
      return flt((int)__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
    };
    auto store = [&](rsrc_t r, int off, float x) __attribute__((always_inline)) {
      __builtin_amdgcn_raw_buffer_store_b32((unsigned)bits(x), r, off, 0, 0);
    };
    // the loads of walk position s (nothing is read past the end of the chain)
    auto load_pix = [&](const int s0) __attribute__((always_inline)) {  // (of the lower half's pixel)
      Pix r;
      const int s = s0 + half;
      const bool on = s < n;
      const unsigned pp = (unsigned)(p_last - s * ch.pstep);
      const int off = label_off(on, pp);
      r.a = load(rA, off);
      r.hd = load(rHdIn, off);
      r.hi = 0.f;
      if (EVEN || SOFT) r.hi = load(rHiIn, off);
      if constexpr (SOFT) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int sh = s0 + h;
          const unsigned ph = (unsigned)(p_last - sh * ch.pstep);
          const bool edge = sh < n - 1;  // (nobody writes the duals of a chain start)
          const rsrc_t rD = make_rsrc(duals + (edge ? (int64_t)ph * kPairs : 0), edge ? kPairs * 4 : 0);
#pragma unroll
          for (int q = 0; q < kSrc; ++q) {
            const int fd = half * kSrc + q;
            r.dual[h][q] = load(rD, (int)(ok && fd < kL ? (front_first ? fd * kL + l : l * kL + fd) * 4 : (int)kDeadOffset));
          }
        }
      }
      r.fd = SOFT ? 0 : __builtin_amdgcn_raw_buffer_load_b8(rImin, (int)((on && ok) ? pp * (unsigned)kL + (unsigned)l : kDeadWide), 0, 0);
      r.nidx = __builtin_amdgcn_raw_buffer_load_b8(rInorm, (int)(on ? pp : kDeadWide), 0, 0);
      r.w = r.de = 0.f;
      if (GR) {
        r.w = load(rW, (int)(on ? pp * 4u : kDeadWide));
        r.de = load(rDe, (int)(on ? pp * 4u : kDeadWide));
      }
      return r;
    };
    float tcol[SOFT ? kSrc : 1];  // ctx(l, front label) of the lane's front labels
    if constexpr (SOFT && GR) {
#pragma unroll
      for (int q = 0; q < kSrc; ++q) {
        const int fd = half * kSrc + q < kL ? half * kSrc + q : kL - 1, cd = ok ? l : kL - 1;
        const float x = ctx_s[cd < fd ? cd * kL + fd : fd * kL + cd];
        tcol[q] = ok && half * kSrc + q < kL ? x : 0.f;
      }
    }
    struct Kept {  // of a pixel whose dU is not known yet
      float ap, base, w, de, cv, hi;
      int nidx, fn;
    };
    // walk position u
    auto prepare = [&](const Pix& px, const int u, Slots& s, Kept& kp) __attribute__((always_inline)) {
      kp.ap = EVEN ? fmaf(rho, px.hi, px.a) : SOFT ? keep(px.a) : px.a;
      kp.base = ok ? kp.ap + (EVEN ? -px.hd - px.hi : px.hd) : 0.f;
      if (GR) {
        kp.w = keep(px.w);
        kp.de = keep(px.de);
        kp.nidx = keep(px.nidx);
      }
      *reinterpret_cast<f32x2*>(s.base[i][l]) = f32x2{kp.base, u < n - 1 ? px.w : 0.f};
      if (GR && !SOFT) {
        const int lo = l < px.fd ? l : px.fd, hi = l < px.fd ? px.fd : l;
        kp.cv = ok && px.fd < kL ? ctx_s[lo * kL + hi] : 0.f;
      }
      if (SOFT) kp.hi = keep(px.hi);
      if constexpr (SOFT) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          // softmin over the front labels of this lane's label (TRWP_backward_soft.cu:83-105), both halves
          const bool two = half * kSrc + kSrc - 1 < kL;  // (the last of the upper half does not exist)
          float d[kSrc], ex[kSrc], lower, upper;
#pragma unroll
          for (int q = 0; q < kSrc; ++q) d[q] = px.dual[h][q];
          float mn = two ? d[kSrc - 1] : INFINITY;
#pragma unroll
          for (int q = 0; q + 1 < kSrc; q += 2) mn = fminf(fminf(mn, d[q]), d[q + 1]);
          halves(mn, lower, upper);
          mn = fminf(lower, upper);
          // relative to the least dual: the sums keep the bits that its size would cost them
          float se2[2] = {0.f, 0.f}, sd2[2] = {0.f, 0.f};
#pragma unroll
          for (int q = 0; q < kSrc; ++q) {
            d[q] -= mn;
            ex[q] = q + 1 < kSrc || two ? __builtin_amdgcn_exp2f(d[q] * -kLog2e) : 0.f;
            se2[q & 1] += ex[q];
            sd2[q & 1] = fmaf(ex[q], d[q], sd2[q & 1]);
          }
          halves(se2[0] + se2[1], lower, upper);
          const float se = lower + upper;
          halves(sd2[0] + sd2[1], lower, upper);
          const float sd = lower + upper;
          // (one Newton step: the instruction's own last bit is a factor of the whole block, and shows in the
          // sums over it; se is 1 to 21, or NaN)
          float inv = __builtin_amdgcn_rcpf(se);
          inv = fmaf(inv, fmaf(-se, inv, 1.f), inv);
          // an error of the expected dual is one of every entry in the same direction: what the weighted
          // differences from it leave, which should be nothing, is taken off again
          const float soft = sd * inv;
          float left2[2] = {0.f, 0.f};
#pragma unroll
          for (int q = 0; q < kSrc; ++q) {
            d[q] = soft - d[q];
            left2[q & 1] = fmaf(ex[q], d[q], left2[q & 1]);
          }
          halves(left2[0] + left2[1], lower, upper);
          const float left = (lower + upper) * inv;
          float jv[kSrc], ev2[2] = {0.f, 0.f};
#pragma unroll
          for (int q = 0; q < kSrc; ++q) {
            const float w = inv * ex[q];
            jv[q] = fmaf(w, d[q] - left, w);  // :110-113
            if (GR) ev2[q & 1] = fmaf(tcol[q], jv[q], ev2[q & 1]);  // (tcol: zero where there is no entry)
          }
          if (ok) {
            float* const row = &s.mask[2 * role + h][l / kSrc][half * kSrc][l % kSrc];
#pragma unroll
            for (int q = 0; q + 1 < kSrc; ++q) row[q * 12] = jv[q];
            // (the upper half's last source does not exist: a zero where it would be read)
            float* const last = two ? row + (kSrc - 1) * 12 : &s.mask[2 * role + h][1][l][kSrc - 1];
            *last = two ? jv[kSrc - 1] : 0.f;
          }
          if (GR) {
            halves(ev2[0] + ev2[1], lower, upper);
            if (half == h) kp.cv = lower + upper;
          }
          lds_order();
          const int nidx = __builtin_amdgcn_readlane(px.nidx, h * kHalf) & (kHalf - 1);
          const int nn = nidx < kL ? nidx : kL - 1;
          if (ok) {
            const int upper_src = nn >= kSrc ? 1 : 0;
            const float jn = s.mask[2 * role + h][upper_src][l][nn - upper_src * kSrc];
            s.mask[2 * role + h][half][l][kSrc] = nidx < kL ? jn : 0.f;
          }
        }
        return;
      }
      s.fd[i][l] = px.fd;
      lds_order();
      const float fl = (float)l;
#pragma unroll
      for (int h = 0; h < 2; ++h) {  // the pixel of either half
        const int nidx = __builtin_amdgcn_readlane(px.nidx, h * kHalf);
        const int fn = __builtin_amdgcn_readlane(px.fd, h * kHalf + (nidx & (kHalf - 1)));
        // (no label points from a lane without one)
        const float src = sl < kL ? (float)s.fd[2 * role + h][sl] : -1.f;
        float m[12];
        static_for<kSrc>([&](auto ii) __attribute__((always_inline)) {
          constexpr int q = decltype(ii)::value;
          const float d = row_bcast<q>(src) - fl;
          m[q] = __builtin_amdgcn_fmed3f(1.f - __builtin_fabsf(d), 0.f, 1.f);
        });
        m[11] = l == fn ? 1.f : 0.f;
        if (half == h) kp.fn = fn;
        if (ok) {
#pragma unroll
          for (int q = 0; q < 3; ++q)
            *reinterpret_cast<f32x4*>(&s.mask[2 * role + h][half][l][4 * q]) = f32x4{m[4 * q], m[4 * q + 1], m[4 * q + 2], m[4 * q + 3]};
        }
      }
    };
    // what is left of a pixel once its dU is known (chain position t; nothing outside the chain)
    auto finish = [&](const int t, const Slots& s, const Kept& kp) __attribute__((always_inline)) {
      const bool on = t >= 0 && t < n;
      const unsigned pp = (unsigned)(ch.pix0 + t * ch.pstep);
      const int off = label_off(on, pp);
      const float sc = s.sc[i][l];
      if constexpr (SOFT) {
        const float an = fmaf(rho, sc, kp.ap);
        store(rAo, off, an);
        store(rHdOut, off, -an);
        store(rHiOut, off, kp.hi - sc);
      } else if constexpr (!EVEN) {
        store(rAo, off, sc);
      } else {
        store(rAo, off, fmaf(rho, sc, kp.ap));  // g_k += rho*dU for every k, dunary too
        store(rHiOut, off, -kp.ap - sc);        // g_o was 0 after its own walk (h_o = -A'), then g_o -= dU
      }
      if constexpr (GR) {
        const bool edge = t >= 1 && t < n;  // the chain start has no incoming edge
        const float tot = s.tot[i][0] + s.tot[i][1];
        float g = fmaf(rho, sc, kp.base);
        if (l == kp.nidx) g -= tot;
        float det = ok && edge ? kp.cv * g : 0.f;
        if (want_de) det = half_sum(det);
        // what the normalisation adds to dcontext; the gradients themselves are the main wavefront's
        if (SOFT && DC && ok && edge && kp.nidx < kL) {
          const int lo = l < kp.nidx ? l : kp.nidx, hi = l < kp.nidx ? kp.nidx : l;
          atomicAdd(&hist_s[lo * kL + hi], -kp.w * tot * s.mask[i][half][l][kSrc]);
        }
        if (!SOFT && DC && l == 0 && edge && kp.nidx < kL && kp.fn < kL && (same || kp.nidx != kp.fn)) {
          const int lo = kp.nidx < kp.fn ? kp.nidx : kp.fn, hi = kp.nidx < kp.fn ? kp.fn : kp.nidx;
          atomicAdd(&hist_s[lo * kL + hi], -kp.w * tot);
        }
        // each pixel receives over exactly one edge per direction: plain read-modify-write
        store(rDe, (int)((edge && l == kHalf - 1) ? pp * 4u : kDeadWide), kp.de + det);
      }
    };

    Pix ring[kAhead];
    Kept kept[2] = {};
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
      ring[q] = load_pix(q * kT + 2 * role);
      MPL_ORDER_LOADS();
    }
#pragma clang loop unroll(disable)
    for (int k0 = 0; k0 < iters; k0 += kAhead) {
#pragma unroll
      for (int q = 0; q < kAhead; ++q) {
        const int k = k0 + q;
        Slots& s = sets[q & 1];
        finish(n - 1 - ((k - 2) * kT + i), s, kept[q & 1]);
        lds_order();
        prepare(ring[q], k * kT + i, s, kept[q & 1]);
        ring[q] = load_pix((k + kAhead) * kT + 2 * role);
        lds_barrier();
      }
    }
  };

  if (role == kHelpers) {
    __builtin_amdgcn_s_setprio(3);
    main_walk();
    if ((ch0.dir & 1) && p.fused_pair) {
      __syncthreads();
      main_walk();
    }
  } else {
    if (ch0.dir & 1) helper_walk(ch0, std::false_type(), p.a_in, p.first_touch != 0);
    if (!(ch0.dir & 1) || p.fused_pair) {
      ChainCtx ch = ch0;
      if (ch0.dir & 1) {
        ch.dir = ch0.dir ^ 1;
        ch.pix0 = ch0.pix0 + (n - 1) * ch0.pstep;
        ch.pstep = -ch0.pstep;
        wait_vmem<0>();
        __syncthreads();
      }
      const bool second = (ch0.dir & 1) != 0;
      helper_walk(ch, std::true_type(), SOFT && second ? p.a_out : p.a_in, (SOFT && second) ? false : p.first_touch != 0);
    }
  }
  if (!DC) return;
  if (role == kHelpers) {
#pragma unroll
    for (int q = 0; q < kSrc; ++q) {
      const int cd = half * kSrc + q;  // the label that points, at fd = l
      if (ok && cd < kL && (same || cd != l)) {
        const int ci = cd < l ? cd * kL + l : l * kL + cd;
        if (has_value(pairs[q])) atomicAdd(&hist_s[ci], pairs[q]);
      }
    }
  }
  __syncthreads();
  float* const dctx = dctx_table(p);
  for (int i = tid; i < kPairs; i += kTeam)
    if (has_value(hist_s[i])) atomicAdd(&dctx[i], hist_s[i]);
}

}  // namespace

void launch_team21_fwd(const SweepParams& p, bool train, hipStream_t st) {
  const int blocks = p.block_prefix[p.n_dirs];
  if (blocks <= 0) return;
  const size_t lds = 2 * sizeof(FwdSlots);
  if (train)
    fwd_team21_kernel<true, false><<<blocks, kTeam, lds, st>>>(p);
  else
    fwd_team21_kernel<false, false><<<blocks, kTeam, lds, st>>>(p);
}

void launch_team21_soft_fwd(const SweepParams& p, hipStream_t st) {
  const int blocks = p.block_prefix[p.n_dirs];
  if (blocks <= 0) return;
  const size_t lds = 2 * sizeof(FwdSlots);
  if (p.edge_label != nullptr)
    fwd_team21_kernel<true, true><<<blocks, kTeam, lds, st>>>(p);
  else
    fwd_team21_kernel<false, true><<<blocks, kTeam, lds, st>>>(p);
}

void launch_team21_bwd(const BackParams& p, hipStream_t st) {
  const int blocks = p.block_prefix[p.n_dirs];
  if (blocks <= 0) return;
  const bool gr = p.dedge != nullptr || p.dctx != nullptr;
  const auto launch = [&](auto kernel, int helpers, size_t set) {
    const size_t lds = 2 * set + sizeof(float) * (kMaxL + (gr ? 2 * kPairs : 0));
    kernel<<<blocks, (helpers + 1) * kWave, lds, st>>>(p);
  };
#define MPL_BWD21(SOFT, N)                                                                                       \
  launch(p.dctx != nullptr ? bwd_team21_kernel<true, true, SOFT, N>                                              \
         : gr              ? bwd_team21_kernel<true, false, SOFT, N>                                             \
                           : bwd_team21_kernel<false, false, SOFT, N>,                                           \
         N, sizeof(BwdSlots<2 * N>))
  const int cus = launch_policy().n_simd / 4;
  // (dynamic LDS beyond 64 KB would have to be asked for)
  constexpr size_t kManyLds = 2 * sizeof(BwdSlots<2 * kManyHelpers>) + sizeof(float) * (kMaxL + 2 * kPairs);
  static_assert(kManyLds <= (64 << 10), "LDS of the reverse scans with many helpers");
  constexpr int kManyPerCu = (160 << 10) / ((kManyLds + 1279) / 1280 * 1280);  // (given out in 1280 bytes)
  if (p.edge_label == nullptr && p.dctx != nullptr && blocks <= kManyPerCu * cus)
    launch(bwd_team21_kernel<true, true, false, kManyHelpers>, kManyHelpers, sizeof(BwdSlots<2 * kManyHelpers>));
  else if (p.edge_label == nullptr)
    MPL_BWD21(false, kHelpers);
  else if (blocks <= cus)
    MPL_BWD21(true, kManyHelpers);
  else
    MPL_BWD21(true, kHelpers);
#undef MPL_BWD21
}

}  // namespace mpl
