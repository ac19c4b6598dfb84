// Reverse scan of TRWP / ISGMR with four wavefronts per chain, for more than 64 labels with a 1-D table
// in launches with fewer chains than the chip has SIMDs.  The recurrence and what each plane holds: mp_bwd.hip.
//
// What bounds such a launch is the length of one pixel's step, not memory: a wavefront that has its
// SIMD to itself issues one instruction every four clocks, and the step of mp_bwd.hip is some 230
// instructions (R = 3, dunary alone; 374 issue slots with its waits), of which the next pixel waits for
// perhaps a third.  So the work is divided by what the recurrence needs:
//   * three helper wavefronts, every third pixel each (six and every sixth: launch_vj), load the planes, form the
//     gradient terms that do not depend on the recurrence and the addresses of the scatter, and put them into an LDS slot
//     per pixel; two blocks of pixels later they take dU of the pixel from the slot, finish the planes
//     it goes into, store them, and add to dedge_weights and dcontext,
//   * the main wavefront touches LDS only: gradient of the message, its sum (the normalisation), the
//     scatter to the argmin labels, dU of the next pixel.
// The wavefronts meet once per block of kT pixels: in iteration k the helpers finish block k - 2 and
// prepare block k while the main wavefront runs block k - 1.  The slots of a block are reused two
// iterations on by the helpers that own them, so two sets suffice.
//
// The scatter: with a truncated pairwise term an argmin label lies within a few labels of its own
// label or is the pixel's argmin(a), which all the others share.  The helpers say for every label
// which of its neighbours up to kWin labels away point at it (five bits) and whether it belongs to
// the ones that share a target (one bit); the main wavefront adds up masked neighbours from registers
// and sums the others with the wave reduction that the normalisation needs anyway (two interleaved
// chains of lane shifts).  In launches of few chains (launch_vj) the bits come as masks as well, 1 or 0 in half precision,
// so that a masked add is one instruction (v_fma_mix) in place of three.  Where labels are left that share a second target (either side of a slope
// under a linear table) another wave reduction sums them; a pixel with any further argmin label scatters
// through LDS float adds.  The normalisation (g[norm_index] -= sum g) reaches dU through its argmin label
// only, and is subtracted there.
//
// Measured, TRWP backward on 4 directions, 5 iterations, min(k, 3) table, one wavefront per chain ->
// this: 256x512x192 5.16 -> 2.12 ms (rows of 256 chains: 645 -> 246 ns per pixel and walk; the main
// wavefront issues 112 instructions per pixel, some five clocks each; masks take another 0.2 ms off), with dedge_weights and dcontext
// 7.18 -> 3.8, 500x800x192 8.91 -> 5.87; bent table 240x320x96 with dcontext 5.95 -> 3.18.  Argmin labels
// anywhere, so that every pixel scatters through LDS adds, 459 instead of 243 ns with 192 labels.  Three helpers with
// two pixels each of a block; with one pixel 2.14, with four 2.36; six helpers of one pixel: launch_vj.  Which launches take it: team_chains_per_cu (mp_api.hip).
//
// Errors against 64 bits, one wavefront -> four, geometric means of the relative 2-norm over bands, a bent
// band, linear and random tables, gradients of a cross entropy, normal and positive ones, 65 to 254
// labels, images up to 300x450, chains up to 8000 pixels: TRWP dunary 1.47e-7 -> 1.42e-7, dcontext
// 8.4e-7 -> 6.8e-7, dedge_weights 1.46e-7 both; ISGMR 2.49e-7 -> 2.31e-7, 4.1e-7 -> 3.8e-7, 1.35e-7 ->
// 1.33e-7; by table and kind of gradient 0.71 to 1.04 times the former.
//
// Compiled once per R (labels per lane, 2 to 4) with -DMPL_INST_R=<R>.

#include <type_traits>

#include "mp_common.h"

namespace mpl {
namespace {

constexpr int kT = 6;                    // pixels per block, shared out among three or six helpers (launch_vj)

constexpr int kWin = 2;                  // labels on either side whose gradients move in registers

// dcontext of a helper's pixels, in LDS: a word per bin, but for the bins up to kNearBins one per lane
// (two with four labels per lane).  Most labels of a pixel may lie that near their argmin label; in one
// word a long chain's sum loses digits, and the adds of a pixel wait for each other.
constexpr int kNearBins = 3;
constexpr int near_words(int R) { return R == 4 ? 2 * kWave : kWave; }  // per bin
constexpr int hist_floats(int R, int n_ctx) { return (kNearBins + 1) * near_words(R) + n_ctx; }

// Slot of a pixel, per lane: the gradient of the message without what the recurrence adds and the
// codes of its labels (one 16-byte read for up to three labels), the argmin labels, dU of the pixel
// (main wavefront) and A' (even walk).
constexpr int in_words(int R) { return R == 4 ? 8 : 4; }
constexpr int vec_words(int R) { return R == 3 ? 4 : R; }
template <int R>
struct alignas(16) Slot {
  float in[kWave][in_words(R)];    // base[R], codes
  float sc[kWave][vec_words(R)];
  float ap[kWave][vec_words(R)];
  int fds[kWave];                  // argmin labels, a byte each
};
struct Scalars {
  float tot;   // sum of the message's gradient (main wavefront)
  float w, de;
  int nidx;
};
// code byte of a label l: bits 0 .. 2 kWin say that the label l + b - kWin points at l,
constexpr int kPop = 5;    // l points at the shared target,
constexpr int kIsPop = 6;  // l is the shared target,
constexpr int kIsNrm = 7;  // l is the argmin label of the normalisation label
// in every lane's word, with up to three labels (from bit 24 on), or the word after it:
constexpr int kRest = 24;  // some argmin label of the pixel is neither near nor the shared one,
constexpr int kMore = 31;  // nor the second shared one,
// and, where kMore is not set, of label j of the lane
constexpr int pop2_bit(int R) { return R == 4 ? 0 : 25; }    // (+ j) it points at the second shared target,
constexpr int is_pop2_bit(int R) { return R == 4 ? 4 : 28; }  // (+ j) it is the second shared target

constexpr int kAccFloats = kMaxL + kWave;  // one per label, one spare word per lane

template <int R>
struct PixT {
  float a[R], hd[R], hi[R];
  int fd[R];
  int nidx;
  float w, de;
};

// LDS of a workgroup, but for the masks of a code byte per label that may follow
template <int R>
__host__ __device__ inline size_t team_lds_bytes(int L, bool gr, int helpers) {
  const size_t bytes = 2 * kT * (sizeof(Slot<R>) + sizeof(Scalars)) +
                       sizeof(float) * (kAccFloats + (gr ? L + helpers * hist_floats(R, L) : 0));
  return (bytes + 15) & ~(size_t)15;
}
constexpr size_t mask_lds_bytes(int R) { return 2 * kT * R * kWave * 16; }

// sums of x and y over the 64 lanes, the two chains of lane-shifted adds interleaved (a lane shift
// may read a register two slots after it was written); the same association as wave_sum_fast
__device__ __forceinline__ void wave_sum2(float& x, float& y) {
#define MPL_ADD2(CTRL)                                        \
  "v_add_f32_dpp %0, %0, %0 " CTRL " bank_mask:0xf\n\t"       \
  "v_add_f32_dpp %1, %1, %1 " CTRL " bank_mask:0xf\n\ts_nop 0\n\t"
  asm("s_nop 1\n\t" MPL_ADD2("row_shr:1 row_mask:0xf") MPL_ADD2("row_shr:2 row_mask:0xf")
      MPL_ADD2("row_shr:4 row_mask:0xf") MPL_ADD2("row_shr:8 row_mask:0xf")
      MPL_ADD2("row_bcast:15 row_mask:0xa") MPL_ADD2("row_bcast:31 row_mask:0xc")
      : "+v"(x), "+v"(y));
#undef MPL_ADD2
  x = readlane_f(x, 63);
  y = readlane_f(y, 63);
}

// A code byte as eight numbers, 1 where the bit is set, in one 16-byte read: a multiply-add with such a mask (v_fma_mix)
// takes the place of an extraction, an AND and an add.
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f16x8 masks_of(int byte) {
  i32x4 m;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int two = (byte >> (2 * k)) & 3;
    m[k] = (int)__umul24((unsigned)((two | (two << 15)) & 0x10001), 0x3c00u);  // (1 in half precision, in either half)
  }
  return __builtin_bit_cast(f16x8, m);
}
// the same masks (left to itself the compiler shifts upper halves down ahead of the branch that uses them)
__device__ __forceinline__ f16x8 opaque(f16x8 m) {
  i32x4 x = __builtin_bit_cast(i32x4, m);
  int x0 = x[0], x1 = x[1], x2 = x[2];
  asm("" : "+v"(x0), "+v"(x1), "+v"(x2));
  return __builtin_bit_cast(f16x8, i32x4{x0, x1, x2, x[3]});
}
__device__ __forceinline__ float mask_add(_Float16 mask, float x, float sum) { return fmaf((float)mask, x, sum); }

// x where bit BIT of the code is set, else 0 (the compiler makes a comparison, a wait state and a
// select of an arithmetic form)
template <int BIT>
__device__ __forceinline__ float if_bit(int code, float x) {
  int m;
  asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(m) : "v"(code), "n"(BIT));
  return __builtin_bit_cast(float, __builtin_bit_cast(int, x) & m);
}
// sum of the masked neighbours of one label (this and the next two are one statement each: the
// compiler puts a wait state between two; BIT0: first bit of the label's code byte)
template <int BIT0>
__device__ __forceinline__ float window_sum(int code, float x0, float x1, float x2, float x3, float x4) {
  float r;
  int m0, m1, m2, m3;
  static_assert(kWin == 2, "five neighbours");
  asm("v_bfe_i32 %0, %5, %11, 1\n\t"
      "v_bfe_i32 %1, %5, %12, 1\n\t"
      "v_bfe_i32 %2, %5, %13, 1\n\t"
      "v_bfe_i32 %3, %5, %14, 1\n\t"
      "v_bfe_i32 %4, %5, %15, 1\n\t"
      "v_and_b32 %0, %0, %6\n\t"
      "v_and_b32 %1, %1, %7\n\t"
      "v_and_b32 %2, %2, %8\n\t"
      "v_add_f32 %0, %0, %1\n\t"
      "v_and_b32 %3, %3, %9\n\t"
      "v_add_f32 %0, %0, %2\n\t"
      "v_and_b32 %4, %4, %10\n\t"
      "v_add_f32 %0, %0, %3\n\t"
      "v_add_f32 %0, %0, %4"
      : "=&v"(r), "=&v"(m0), "=&v"(m1), "=&v"(m2), "=&v"(m3)
      : "v"(code), "v"(x0), "v"(x1), "v"(x2), "v"(x3), "v"(x4), "n"(BIT0), "n"(BIT0 + 1), "n"(BIT0 + 2),
        "n"(BIT0 + 3), "n"(BIT0 + 4));
  return r;
}
// near + (pop if the label is the shared target) - (tot if the normalisation reaches it)
// (the two extractions come first: a scalar register that v_readlane has just written may be read by
// the vector unit two issue slots later)
template <int BIT0>
__device__ __forceinline__ float window_finish(int code, float near, float pop, float tot) {
  int m0, m1;
  asm("v_bfe_i32 %1, %3, %6, 1\n\t"
      "v_bfe_i32 %2, %3, %7, 1\n\t"
      "v_and_b32 %1, %4, %1\n\t"
      "v_and_b32 %2, %5, %2\n\t"
      "v_sub_f32 %1, %1, %2\n\t"
      "v_add_f32 %0, %0, %1"
      : "+v"(near), "=&v"(m0), "=&v"(m1)
      : "v"(code), "s"(pop), "s"(tot), "n"(BIT0 + kIsPop), "n"(BIT0 + kIsNrm));
  return near;
}

// pop += g where the label points at the shared target
template <int BIT0>
__device__ __forceinline__ void add_popular(int code, float g, float& pop) {
  int m;
  asm("v_bfe_i32 %1, %2, %4, 1\n\t"
      "v_and_b32 %1, %1, %3\n\t"
      "v_add_f32 %0, %0, %1"
      : "+v"(pop), "=&v"(m)
      : "v"(code), "v"(g), "n"(BIT0 + kPop));
}

// f(0) .. f(N - 1) with constant arguments
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(const F& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>());
    static_for<N, I + 1>(f);
  }
}

// x of the labels lab0 - kWin .. lab0 + R - 1 + kWin, 0 outside the wavefront's labels
template <int R, typename T>
__device__ __forceinline__ void neighbours(const T (&x)[R], T (&nb)[R + 2 * kWin]) {
  auto up = [](T v) { return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true)); };
  auto dn = [](T v) { return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true)); };
#pragma unroll
  for (int j = 0; j < R; ++j) nb[kWin + j] = x[j];
#pragma unroll
  for (int o = 1; o <= kWin; ++o) {
    nb[kWin - o] = up(nb[kWin - o + R]);
    nb[kWin + R - 1 + o] = dn(nb[kWin - 1 + o]);
  }
}

template <int N>
__device__ __forceinline__ void lds_get(const float* src, float (&x)[N]) {
  if constexpr (N == 4) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(src);
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = v[i];
  } else {
    static_assert(N == 2, "words of a slot come in twos and fours");
    const f32x2 v = *reinterpret_cast<const f32x2*>(src);
    x[0] = v[0];
    x[1] = v[1];
  }
}
template <int N>
__device__ __forceinline__ void lds_put(float* dst, const float (&x)[N]) {
  if constexpr (N == 4) {
    *reinterpret_cast<f32x4*>(dst) = f32x4{x[0], x[1], x[2], x[3]};
  } else if constexpr (N == 3) {
    *reinterpret_cast<f32x4*>(dst) = f32x4{x[0], x[1], x[2], 0.f};
  } else {
    static_assert(N == 2, "words of a slot come in twos and fours");
    *reinterpret_cast<f32x2*>(dst) = f32x2{x[0], x[1]};
  }
}
// an R-label vector of a slot (three labels: padded to four words)
template <int R>
__device__ __forceinline__ void lds_get_labels(const float* src, float (&x)[R]) {
  float t[vec_words(R)];
  lds_get(src, t);
#pragma unroll
  for (int j = 0; j < R; ++j) x[j] = t[j];
}
// base[R] and the codes
template <int R>
__device__ __forceinline__ void get_in(const float* src, float (&base)[R], int& code, int& rest) {
  if constexpr (R == 4) {
    float t[2];
    lds_get(src, base);
    lds_get(src + 4, t);
    code = __builtin_bit_cast(int, t[0]);
    rest = __builtin_bit_cast(int, t[1]);
  } else {
    float t[4];
    lds_get(src, t);
#pragma unroll
    for (int j = 0; j < R; ++j) base[j] = t[j];
    code = rest = __builtin_bit_cast(int, t[R]);
  }
}
template <int R>
__device__ __forceinline__ void put_in(float* dst, const float (&base)[R], int code, int rest) {
  const float c = __builtin_bit_cast(float, R == 4 ? code : code | rest);
  if constexpr (R == 4) {
    const float t[2] = {c, __builtin_bit_cast(float, rest)};
    lds_put(dst, base);
    lds_put(dst + 4, t);
  } else {
    float t[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) t[j] = j < R ? base[j < R ? j : 0] : c;
    lds_put(dst, t);
  }
}

// workgroup barrier over LDS contents only: global loads in flight stay in flight
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
__device__ __forceinline__ void lds_order() {  // of this wavefront's own LDS instructions; none emitted
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}

// GR: dedge_weights and / or dcontext are wanted.  MASKS: the helpers put the codes into LDS as masks too (masks_of).
template <int R, bool VEC, bool JACOBI, bool GR, int kHelpers, bool MASKS>
__global__ void __launch_bounds__((kHelpers + 1) * kWave) sweep_bwd_team_kernel(const BackParams p, const int turn_every) {
  constexpr int kPer = kT / kHelpers;  // pixels of a block per helper
  constexpr int kTeam = (kHelpers + 1) * kWave;
  extern __shared__ __align__(16) char smem_raw[];
  Slot<R>* slots = reinterpret_cast<Slot<R>*>(smem_raw);  // two sets of kT
  Scalars* scal = reinterpret_cast<Scalars*>(slots + 2 * kT);
  float* acc = reinterpret_cast<float*>(scal + 2 * kT);
  float* ctx_s = acc + kAccFloats;
  const int L = p.L;
  const int n_ctx = L;  // (1-D tables only)
  float* hist_s = ctx_s + n_ctx;  // dcontext, one histogram per helper
  f16x8* masks = reinterpret_cast<f16x8*>(smem_raw + team_lds_bytes<R>(L, GR, kHelpers));  // [2 kT][R][kWave]
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  // The last wavefront is the main one in every workgroup: the wavefronts of the workgroups that a compute
  // unit gets one after another start one SIMD further each (read from the hardware-id registers for 2, 3
  // and 4 workgroups per unit), so the main wavefronts of up to four of them are on SIMDs of their own.
  // With four labels per lane and turn_every > 0 (launch_vj) it moves on by one every so many workgroups.
  const int turn = R == 4 && turn_every > 0 ? (int)blockIdx.x / turn_every : 0;
  // (of seven wavefronts the main one is the fourth, whose SIMD has only one of them)
  const int wave = uniform_i(tid / kWave);
  const int role = kHelpers == 3 ? (wave + turn) & 3 : wave == 3 ? kHelpers : wave - (wave > 3 ? 1 : 0);  // kHelpers: main
  const int64_t HW = (int64_t)p.H * p.W;
  const int64_t P = (int64_t)p.B * HW;
  const int64_t N = P * L;
  const ChainCtx ch0 = locate_chain<false>(p);
  const int n = ch0.n;
  const int lab0 = R * lane;
  const bool lane_ok = lab0 < L;
  const float rho = p.rho;
  const bool want_dc = GR && p.dctx != nullptr;
  const bool same = p.same_label != 0;

  for (int i = tid; i < kAccFloats; i += kTeam) acc[i] = 0.f;
  const int n_hist = hist_floats(R, n_ctx);
  if (GR) {
    for (int i = tid; i < n_ctx; i += kTeam) ctx_s[i] = p.ctx[i];
    for (int i = tid; i < kHelpers * n_hist; i += kTeam) hist_s[i] = 0.f;
  }
  __syncthreads();

  const int blocks = (n + kT - 1) / kT;
  const int iters = (blocks + 2 + 1) & ~1;  // (the helpers' loop is unrolled by two)

  auto main_walk = [&]() __attribute__((always_inline)) {
    float sc[R];
#pragma unroll
    for (int j = 0; j < R; ++j) sc[j] = 0.f;
    float* const mine = acc + lab0;
    // one pixel: sc is dU of the one before, then of this one
    auto pixel = [&](Slot<R>& s, Scalars& sv, const float (&base)[R], const int code, const int rest, const f16x8 (&m)[R],
                     const auto read_next, const auto masked) __attribute__((always_inline)) {
      constexpr bool M = decltype(masked)::value;
      float g[R], part, pop;
#pragma unroll
      for (int j = 0; j < R; ++j)
        // gradient w.r.t. the normalised message of this pixel, including what the previous
        // step added through the recurrence (dmsg[front] += rho * value, TRWP_backward.cu:108)
        g[j] = fmaf(rho, sc[j], base[j]);
      lds_put(s.sc[lane], sc);
      read_next();
      part = g[0];
      pop = M ? mask_add(m[0][kPop], g[0], 0.f) : if_bit<kPop>(code, g[0]);
      static_for<R - 1>([&](auto jj) __attribute__((always_inline)) {
        constexpr int j = decltype(jj)::value + 1;
        part += g[j];
        if constexpr (M)
          pop = mask_add(m[j][kPop], g[j], pop);
        else
          add_popular<8 * j>(code, g[j], pop);
      });
      wave_sum2(part, pop);
      float near[R];
      auto near_sums = [&]() __attribute__((always_inline)) {
        float nb[R + 2 * kWin];
        neighbours<R>(g, nb);
        if constexpr (M) {
          f16x8 mj[R];
#pragma unroll
          for (int j = 0; j < R; ++j) mj[j] = opaque(m[j]);
          // (the labels' sums side by side: one that follows another of its label waits a slot)
#pragma unroll
          for (int b = 0; b <= 2 * kWin; ++b)
#pragma unroll
            for (int j = 0; j < R; ++j) near[j] = mask_add(mj[j][b], nb[j + b], b == 0 ? 0.f : near[j]);
        } else {
          static_for<R>([&](auto jj) __attribute__((always_inline)) {
            constexpr int j = decltype(jj)::value;
            near[j] = window_sum<8 * j>(code, nb[j], nb[j + 1], nb[j + 2], nb[j + 3], nb[j + 4]);
          });
        }
      };
      const int kind = __builtin_amdgcn_readfirstlane(rest);
      if (__builtin_expect((kind & (1 << kRest)) == 0, 1)) {
        near_sums();
      } else if (kind >= 0) {  // (bit kMore) two shared targets
        near_sums();
        float pop2 = 0.f;
        static_for<R>([&](auto jj) __attribute__((always_inline)) {
          constexpr int j = decltype(jj)::value;
          pop2 += if_bit<pop2_bit(R) + j>(rest, g[j]);
        });
        pop2 = wave_sum_fast(pop2);
        static_for<R>([&](auto jj) __attribute__((always_inline)) {
          constexpr int j = decltype(jj)::value;
          near[j] += if_bit<is_pop2_bit(R) + j>(rest, pop2);
        });
      } else {
        const int fds = s.fds[lane];
#pragma unroll
        for (int j = 0; j < R; ++j) {
          const bool skip = ((code >> (8 * j + kPop)) & 1) != 0 || lab0 + j >= L;
          atomicAdd(&acc[skip ? kMaxL + lane : ((fds >> (8 * j)) & 0xff)], g[j]);
        }
        lds_order();
#pragma unroll
        for (int j = 0; j < R; ++j) near[j] = mine[j];
        lds_order();
#pragma unroll
        for (int j = 0; j < R; ++j) mine[j] = 0.f;
        lds_order();
      }
      if (GR) sv.tot = part;  // (every lane stores the same value to the same address)
      static_for<R>([&](auto jj) __attribute__((always_inline)) {
        constexpr int j = decltype(jj)::value;
        if constexpr (M)
          sc[j] = near[j] + mask_add(-m[j][kIsNrm], part, mask_add(m[j][kIsPop], pop, 0.f));
        else
          sc[j] = window_finish<8 * j>(code, near[j], pop, part);
      });
    };
    for (int k = 0; k < iters; ++k) {
      if (k >= 1 && k <= blocks) {
        Slot<R>* s = slots + ((k - 1) & 1) * kT;
        Scalars* sv = scal + ((k - 1) & 1) * kT;
        const f16x8* const mk = masks + (((k - 1) & 1) * kT * R) * kWave + lane;
        auto block = [&](const auto masked) __attribute__((always_inline)) {
          constexpr bool M = decltype(masked)::value;
          float base[R];
          int code, rest;
          f16x8 m[R] = {};
          get_in<R>(s[0].in[lane], base, code, rest);
          if constexpr (M) {
#pragma unroll
            for (int j = 0; j < R; ++j) m[j] = mk[j * kWave];
          }
#pragma unroll
          for (int i = 0; i < kT; ++i) {
            float nbase[R];
            int ncode = 0, nrest = 0;
            f16x8 nm[R] = {};
            pixel(
                s[i], sv[i], base, code, rest, m,
                [&]() __attribute__((always_inline)) {  // (the next pixel's reads, once this one's dU is on its way)
                  if (i + 1 < kT) {
                    get_in<R>(s[i + 1].in[lane], nbase, ncode, nrest);
                    if constexpr (M) {
#pragma unroll
                      for (int j = 0; j < R; ++j) nm[j] = mk[((i + 1) * R + j) * kWave];
                    }
                  }
                },
                masked);
            if (i + 1 < kT) {
#pragma unroll
              for (int j = 0; j < R; ++j) {
                base[j] = nbase[j];
                m[j] = nm[j];
              }
              code = ncode;
              rest = nrest;
            }
          }
        };
        if constexpr (MASKS) {
          float sc_was[R];
#pragma unroll
          for (int j = 0; j < R; ++j) sc_was[j] = sc[j];
          block(std::true_type());
          // A zero mask does not switch off what is not finite: an infinity or a NaN in a gradient, or in a sum, makes
          // NaN of every label's dU, there and from there on (tested as an integer: the compiler may take NaN for
          // anything).  The pixels of such a block go by the codes, one after another.
          int probe = uniform_i(__builtin_bit_cast(int, sc[0]));
          asm("" : "+s"(probe));
          if (__builtin_expect((probe & 0x7f800000) == 0x7f800000, 0)) {
#pragma unroll
            for (int j = 0; j < R; ++j) sc[j] = sc_was[j];
            const f16x8 none[R] = {};
#pragma clang loop unroll(disable)
            for (int i = 0; i < kT; ++i) {
              float base[R];
              int code, rest;
              get_in<R>(s[i].in[lane], base, code, rest);
              pixel(s[i], sv[i], base, code, rest, none, []() {}, std::false_type());
            }
          }
        } else {
          block(std::false_type());
        }
      }
      lds_barrier();
    }
  };

  // even_walk: a constant; which of the two walks of a pair this is (Gauss-Seidel, mp_bwd.hip)
  auto helper_walk = [&](const ChainCtx& ch, const auto even_walk) __attribute__((always_inline)) {
    constexpr bool EVEN = !JACOBI && decltype(even_walk)::value;
    const int dir = ch.dir;
    const int64_t img_p = (int64_t)ch.bv * HW;
    const int64_t img_e = img_p * L;
    const bool read_h = !p.first_touch;
    const float* bA =
        (JACOBI ? p.gu_in + (int64_t)(p.gu_pair_share ? (dir & ~1) : dir) * p.gu_stride : p.a_in) + img_e;
    float* hbase = JACOBI ? p.du_out : p.h;
    float* bHd = hbase + (int64_t)dir * N + img_e;
    float* bHi = hbase + (int64_t)(dir ^ 1) * N + img_e;
    float* bAo = EVEN ? p.a_out + img_e : bHd;
    const int img_bytes = (int)(unsigned)(HW * L * 4);
    const int img_bytes_p = (int)(HW * 4 > 0x7fffffff ? 0x7fffffff : HW * 4);
    const rsrc_t rA = make_rsrc(bA, img_bytes);
    const rsrc_t rAo = make_rsrc(bAo, img_bytes);
    const rsrc_t rHdIn = make_rsrc(bHd, (!JACOBI && read_h) ? img_bytes : 0);
    const rsrc_t rHiIn = make_rsrc(bHi, EVEN ? img_bytes : 0);
    const rsrc_t rHiOut = make_rsrc(bHi, (EVEN && !p.skip_h_store) ? img_bytes : 0);
    const rsrc_t rImin = make_rsrc(p.idx_min + (int64_t)dir * N + img_e, (int)(HW * L));
    const rsrc_t dInorm = make_rsrc(p.idx_norm + (int64_t)dir * P + img_p, (int)HW);
    const rsrc_t dW = make_rsrc(p.edge + (int64_t)dir * P + img_p, img_bytes_p);
    const bool want_de = GR && p.dedge != nullptr;
    const rsrc_t dDe = make_rsrc(want_de ? p.dedge + (int64_t)dir * P + img_p : nullptr,
                                 want_de ? img_bytes_p : 0);
    const int p_last = ch.pix0 + (n - 1) * ch.pstep;

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
    auto store_plane = [&](rsrc_t r, bool on, unsigned so, const float (&x)[R]) __attribute__((always_inline)) {
      if constexpr (VEC) {
        buf_store<R, true>(r, vec_off(on, so, 0), 0u, x);
      } else {
#pragma unroll
        for (int j = 0; j < R; ++j)
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x[j]), r, vec_off(on, so, j), 0, MPL_ST_AUX);
      }
    };
    // the loads of walk position s (nothing is read past the end of the chain)
    auto load_pix = [&](const int s) __attribute__((always_inline)) {
      PixT<R> r;
      const bool on = s < n;
      const unsigned pp = (unsigned)(p_last - s * ch.pstep);
      const unsigned so = pp * (unsigned)L * 4u;
      load_plane(rA, on, so, r.a);
#pragma unroll
      for (int j = 0; j < R; ++j) r.hd[j] = r.hi[j] = 0.f;
      if (!JACOBI) load_plane(rHdIn, on, so, r.hd);
      if (EVEN) load_plane(rHiIn, on, so, r.hi);
      if constexpr (VEC) {
        buf_load_u8<R, true, load_policy(false)>(rImin, (int)((on && lane_ok) ? pp * (unsigned)L + (unsigned)lab0 : kDeadWide), 0u, r.fd);
      } else {
#pragma unroll
        for (int j = 0; j < R; ++j)
          r.fd[j] = __builtin_amdgcn_raw_buffer_load_b8(
              rImin, (int)((on && lab0 + j < L) ? pp * (unsigned)L + (unsigned)(lab0 + j) : kDeadWide), 0, load_policy(false));
      }
      r.nidx = __builtin_amdgcn_raw_buffer_load_b8(dInorm, on ? (int)pp : kDeadOffset, 0, 0);
      r.w = r.de = 0.f;
      if (GR) {
        r.w = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(dW, on ? (int)(pp * 4u) : kDeadOffset, 0, 0));
        r.de = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(dDe, on ? (int)(pp * 4u) : kDeadOffset, 0, 0));
      }
      return r;
    };

    // what the recurrence needs of a pixel, into its slot
    auto prepare = [&](const PixT<R>& px, Slot<R>& s, Scalars& sv, f16x8* const mk) __attribute__((always_inline)) {
      const int nidx = __builtin_amdgcn_readfirstlane(px.nidx);
      int fn = 0;  // argmin label of the normalisation label
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int v = __builtin_amdgcn_readlane(px.fd[j], (nidx / R) & (kWave - 1));
        fn = (j == nidx % R) ? v : fn;
      }
      // labels that point into the window, as the bit their target has for them; the target most of
      // the others share is taken to be the first one's
      int src[R], pop = -1, fds = 0;
      bool out[R];
#pragma unroll
      for (int j = R - 1; j >= 0; --j) {
        const int d = px.fd[j] - (lab0 + j);
        const bool valid = lab0 + j < L;
        const bool win = (unsigned)(d + kWin) <= 2u * kWin;
        src[j] = (win && valid) ? 1 << ((kWin - d) & 31) : 0;
        out[j] = valid && !win;
        const uint64_t m = ballot(out[j]);
        if (m != 0) pop = __builtin_amdgcn_readlane(px.fd[j], __builtin_ctzll(m));
        fds |= px.fd[j] << (8 * j);
      }
      int nb[R + 2 * kWin];
      neighbours<R>(src, nb);
      int code = 0;
      bool left[R];
      float base[R], ap[R];
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int l = lab0 + j;
        int c = 0;
#pragma unroll
        for (int b = 0; b <= 2 * kWin; ++b) c |= nb[j + b] & (1 << b);
        const bool is_pop = out[j] && px.fd[j] == pop;
        left[j] = out[j] && !is_pop;
        c |= is_pop ? 1 << kPop : 0;
        c |= l == pop ? 1 << kIsPop : 0;
        c |= l == fn ? 1 << kIsNrm : 0;
        code |= c << (8 * j);
        if constexpr (MASKS) mk[j * kWave + lane] = masks_of(c);
        ap[j] = EVEN ? fmaf(rho, px.hi[j], px.a[j]) : px.a[j];
        base[j] = JACOBI ? px.a[j] : ap[j] + (EVEN ? -px.hd[j] - px.hi[j] : px.hd[j]);
        if (l >= L) base[j] = 0.f;
      }
      // of the others, those that point where the last of them does
      bool any_left = left[0];
#pragma unroll
      for (int j = 1; j < R; ++j) any_left |= left[j];
      int rest = 0;
      const uint64_t lm = ballot(any_left);
      if (lm != 0) {
        const int last = 63 - __builtin_clzll(lm);
        int fl = 0;
#pragma unroll
        for (int j = 0; j < R; ++j) fl = left[j] ? px.fd[j] : fl;
        const int pop2 = __builtin_amdgcn_readlane(fl, last);
        bool more = false;
#pragma unroll
        for (int j = 0; j < R; ++j) {
          const bool is_pop2 = left[j] && px.fd[j] == pop2;
          more |= left[j] && !is_pop2;
          rest |= is_pop2 ? 1 << (pop2_bit(R) + j) : 0;
          rest |= lab0 + j == pop2 ? 1 << (is_pop2_bit(R) + j) : 0;
        }
        rest |= 1 << kRest;
        if (ballot(more) != 0) rest |= 1 << kMore;
      }
      put_in<R>(s.in[lane], base, code, rest);
      s.fds[lane] = fds;
      if (EVEN) lds_put(s.ap[lane], ap);
      if (GR) {
        sv.w = px.w;
        sv.de = px.de;
        sv.nidx = nidx;
      }
    };

    // what is left of a pixel once its dU is known (chain position t; nothing outside the chain)
    auto finish = [&](const int t, const Slot<R>& s, const Scalars& sv) __attribute__((always_inline)) {
      const bool on = t >= 0 && t < n;
      const unsigned pp = (unsigned)(ch.pix0 + t * ch.pstep);
      const unsigned so = pp * (unsigned)L * 4u;
      float sc[R];
      lds_get_labels<R>(s.sc[lane], sc);
      if constexpr (!EVEN) {
        store_plane(rAo, on, so, sc);
      } else {
        float ap[R], an[R], hin[R];
        lds_get_labels<R>(s.ap[lane], ap);
#pragma unroll
        for (int j = 0; j < R; ++j) {
          an[j] = fmaf(rho, sc[j], ap[j]);  // g_k += rho*dU for every k, dunary too
          hin[j] = -ap[j] - sc[j];          // g_o was 0 after its own walk (h_o = -A'), then g_o -= dU
        }
        store_plane(rAo, on, so, an);
        store_plane(rHiOut, on, so, hin);
      }
      if constexpr (GR) {
        const bool edge = t >= 1 && t < n;  // the chain start has no incoming edge
        float det = 0.f, de_old = 0.f;
        if (edge) {  // wave-uniform
          const float tot = sv.tot, w = sv.w;
          float base[R];
          int code, rest;
          get_in<R>(s.in[lane], base, code, rest);
          const int fds = s.fds[lane];
          const int nidx = sv.nidx;
          de_old = sv.de;
          float* const hist = hist_s + role * n_hist;
#pragma unroll
          for (int j = 0; j < R; ++j) {
            const int cd = lab0 + j;
            const int fd = (fds >> (8 * j)) & 0xff;
            float g = fmaf(rho, sc[j], base[j]);
            if (cd == nidx) g -= tot;  // MsgNormNaiveBack, commonCUDA.cuh:131-145
            const int ci = fd > cd ? fd - cd : cd - fd;
            if (cd < L) {
              det = fmaf(ctx_s[ci], g, det);
              const int near = ci * near_words(R) + (j * kWave) % near_words(R) + lane;
              const int at = ci <= kNearBins ? near : (kNearBins + 1) * near_words(R) + ci;
              if (want_dc && (same || cd != fd)) atomicAdd(&hist[at], w * g);
            }
          }
          if (want_de) det = wave_sum_fast(det);
        }
        // each pixel receives over exactly one edge per direction: plain read-modify-write
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, de_old + det), dDe,
                                              edge ? (int)(pp * 4u) : kDeadOffset, 0, 0);
      }
    };

    PixT<R> ring0[kPer], ring1[kPer];  // blocks k and k + 1
#pragma unroll
    for (int u = 0; u < kPer; ++u) ring0[u] = load_pix(role + kHelpers * u);
    MPL_ORDER_LOADS();
#pragma unroll
    for (int u = 0; u < kPer; ++u) ring1[u] = load_pix(kT + role + kHelpers * u);
    MPL_ORDER_LOADS();
    auto iteration = [&](const int k, PixT<R> (&ring)[kPer], const int set) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int i = role + kHelpers * u;
        Slot<R>& s = slots[set * kT + i];
        Scalars& sv = scal[set * kT + i];
        finish(n - 1 - ((k - 2) * kT + i), s, sv);
        lds_order();
        prepare(ring[u], s, sv, masks + (set * kT + i) * R * kWave);
        ring[u] = load_pix((k + 2) * kT + i);
      }
      lds_barrier();
    };
#pragma clang loop unroll(disable)
    for (int k = 0; k < iters; k += 2) {
      iteration(k, ring0, 0);
      iteration(k + 1, ring1, 1);
    }
  };

  const bool is_main = role == kHelpers;
  if (is_main) __builtin_amdgcn_s_setprio(3);
  auto walk = [&](const ChainCtx& ch, const auto even_walk) __attribute__((always_inline)) {
    if (is_main)
      main_walk();
    else
      helper_walk(ch, even_walk);
  };
  if constexpr (JACOBI) {
    walk(ch0, std::false_type());
  } else {
    // the second walk of a pair reads what the first one's helpers stored: on the same compute unit,
    // once their stores are complete
    if (is_main) {
      main_walk();
      if ((ch0.dir & 1) && p.fused_pair) {
        __syncthreads();
        main_walk();
      }
    } else {
      if (ch0.dir & 1) helper_walk(ch0, std::false_type());
      if (!(ch0.dir & 1) || p.fused_pair) {
        ChainCtx ch = ch0;
        if (ch0.dir & 1) {
          ch.dir = ch0.dir ^ 1;
          ch.pix0 = ch0.pix0 + (n - 1) * ch0.pstep;
          ch.pstep = -ch0.pstep;
          wait_vmem<0>();
          __syncthreads();
        }
        helper_walk(ch, std::true_type());
      }
    }
  }
  if (!want_dc) return;
  __syncthreads();
  if (!is_main) {  // the words of a near bin into its place in the histogram
    float* const hist = hist_s + role * n_hist;
#pragma unroll
    for (int o = 0; o <= kNearBins; ++o) {
      float v = hist[o * near_words(R) + lane];
      if (R == 4) v += hist[o * near_words(R) + kWave + lane];
      v = wave_sum(v);
      if (lane == 0) hist[(kNearBins + 1) * near_words(R) + o] = v;
    }
  }
  __syncthreads();
  float* const dctx = dctx_table(p);
  for (int i = tid; i < n_ctx; i += kTeam) {
    float v = 0.f;
#pragma unroll
    for (int h = 0; h < kHelpers; ++h) v += hist_s[h * n_hist + (kNearBins + 1) * near_words(R) + i];
    if (has_value(v)) atomicAdd(&dctx[i], v);
  }
}

template <int R, bool VEC, bool JACOBI>
void launch_vj(const BackParams& p, hipStream_t st) {
  const int blocks = p.block_prefix[p.n_dirs];
  const bool gr = p.dedge != nullptr || p.dctx != nullptr;
  const auto launch = [&](auto kernel, int helpers, int turn_every, size_t extra = 0) {
    const size_t lds = team_lds_bytes<R>(p.L, gr, helpers) + extra;
    if (lds > (64 << 10))  // (a refusal shows as the launch's, and is reported with it)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    kernel<<<blocks, (helpers + 1) * kWave, lds, st>>>(p, turn_every);
  };
  // With four labels per lane the LDS holds two workgroups of a unit, and a launch of more runs in rounds.  When
  // both end together the next ones are placed in pairs again and the last round takes as long as the first;
  // with the main wavefronts of a unit's workgroups on one SIMD they do not.  Measured, 760 rows of 300 pixels,
  // 2 iterations, ms on SIMDs of their own / on one: 256 labels, min(k, 4) 1.38 / 1.25, linear 3.07 / 2.50, random 3.38 / 2.75;
  // 500 rows 0.710 / 0.723, 1.55 / 1.60, 1.72 / 1.78.
  const int n_cu = launch_policy().n_simd / 4;
  const int turn_every = R == 4 && blocks > 2 * n_cu ? n_cu : 0;
  // Six helpers where the launch has at most three chains per unit: what they do for a pixel bounds the scan wherever
  // dcontext or dedge_weights are wanted, and three of them on a SIMD of their own each issue less than half of the
  // time.  Over three helpers, dunary alone / with dedge_weights / with both, rows of 129: 192 labels, min(k, 3), 256
  // chains 0.95 / 0.81 / 0.82, 512 chains 0.98 / 0.84 / 0.92, 768 chains 1.00 / 0.92 / 0.98; 96 labels, a random table, 256
  // chains 0.98 / 0.96 / 0.99, 768 chains 0.99 / 0.98 / 0.99; 65 labels 768 chains 0.93 / 0.83 / 0.85; labels one by one,
  // 191 labels 256 chains 0.92 / 0.72 / 0.79; ISGMR 96 labels 96x96 0.99 / 1.00 / 0.99, 192 labels 64x64 0.97 / 0.91 / 0.86;
  // 500x700, 192 labels, 1199 diagonals 1.04 / 0.94 / 1.04.
  if constexpr (R < 4) {
    if (blocks <= 3 * n_cu) {
      // Masks where the LDS holds those of all the launch's chains (160 KB a unit, given out in 1280 bytes): a chain per
      // unit more would wait for another to end.  Over the codes, the layer's whole pass, 4 directions, 5 iterations, dunary
      // alone: 192 labels 256x512 0.946, 130x160 0.92, 96 and 128 labels 240x320 0.91, 191 labels 0.98; with 8 directions, whose
      // diagonals are more chains than that, 200x260 0.93, 375x450 0.99; a learned table 96 labels 240x320 0.975; ISGMR
      // 128 labels 130x160 0.96.
      const size_t with_masks = (team_lds_bytes<R>(p.L, gr, 6) + mask_lds_bytes(R) + 1279) / 1280 * 1280;
      if ((size_t)blocks <= n_cu * ((160 << 10) / with_masks)) {
        launch(gr ? sweep_bwd_team_kernel<R, VEC, JACOBI, true, 6, true> : sweep_bwd_team_kernel<R, VEC, JACOBI, false, 6, true>, 6, 0,
               mask_lds_bytes(R));
        return;
      }
      launch(gr ? sweep_bwd_team_kernel<R, VEC, JACOBI, true, 6, false> : sweep_bwd_team_kernel<R, VEC, JACOBI, false, 6, false>, 6, 0);
      return;
    }
  }
  launch(gr ? sweep_bwd_team_kernel<R, VEC, JACOBI, true, 3, false> : sweep_bwd_team_kernel<R, VEC, JACOBI, false, 3, false>, 3, turn_every);
}

}  // namespace

template <int R>
void launch_team_bwd(const BackParams& p, bool jacobi, hipStream_t st) {
  if (p.block_prefix[p.n_dirs] <= 0) return;
  static_assert(R > 1, "several labels per lane");
  if (p.L % R == 0) {
    if (jacobi)
      launch_vj<R, true, true>(p, st);
    else
      launch_vj<R, true, false>(p, st);
  } else {
    if (jacobi)
      launch_vj<R, false, true>(p, st);
    else
      launch_vj<R, false, false>(p, st);
  }
}

template void launch_team_bwd<MPL_INST_R>(const BackParams&, bool, hipStream_t);

}  // namespace mpl
