// C ABI, host orchestration and the element-wise kernels of the TRWP / ISGMR path (gfx950).
// The scan kernels live in mp_fwd.hip / mp_bwd.hip; shared device helpers in mp_common.h.
//
// Traffic model: instead of re-summing all messages for every sweep (UpdateUnaryKernel of the
// reference, TRWP_forward.cu:60-80), a belief plane S = unary + sum_k m_k is kept, so a sweep of
// direction d reads S, m_d, m_inv and writes m_d (and S for TRWP): 20 B per label.  The backward
// pass keeps the gradient planes as g_k = A + h_k with one shared plane A (which ends up being
// dunary) for the same reason.

#include <limits.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>
#include <vector>

#include "mp_common.h"

using namespace mpl;

namespace {

// 1-D context c[0..L-1]: find the constant tail and recognise a truncated linear table.  One wave,
// every lane looks at the entries lane, lane + 64, ...; the findings are combined with ballots.
__global__ void __launch_bounds__(kWave) analyze_context_kernel(const float* __restrict__ ctx, int L,
                                                                int ctx2d, CtxDesc* __restrict__ d) {
  const int lane = threadIdx.x;
  CtxDesc r;
  r.band_k = 0;
  r.c0_is_min = 0;
  r.cmax = 0.f;
  r.msg_nonzero = 0;
  r.linear = 0;
  r.slope = 0.f;
  if (!ctx2d) {
    const float tail = ctx[L - 1];
    const float c0 = ctx[0];
    const float slope = L >= 2 ? ctx[1] : 0.f;
    int last_ne = -1;  // largest index whose entry differs from the tail
    bool below = true, c0min = true, lin = true;
    for (int i = lane; i < L; i += kWave) {
      const float v = ctx[i];
      if (!(v == tail)) last_ne = i;
      below = below && (v <= tail);
      c0min = c0min && (c0 <= v);
      lin = lin && (v == fminf(slope * (float)i, tail));
    }
    int k = (int)-wave_min(-(float)last_ne) + 1;  // c[k..L-1] == tail  (indices < 2^24: exact)
    // a NaN tail disables both fast paths; tested on the bit pattern because the library is
    // compiled without NaN semantics, where `tail == tail` may be folded to true
    const bool tail_is_nan = (__builtin_bit_cast(unsigned, tail) & 0x7fffffffu) > 0x7f800000u;
    const bool ok = !tail_is_nan && ballot(!below) == 0;
    const bool all_c0min = ballot(!c0min) == 0;
    const bool all_lin = ballot(!lin) == 0;
    if (k < 1) k = 1;  // a constant context: the centre tap alone is the band
    if (ok && k <= kMaxBandK) {
      r.band_k = k;
      r.cmax = tail;
      r.c0_is_min = all_c0min ? 1 : 0;
    }
    // truncated linear, bit for bit: c[k] == min(c[1] * k, c[L-1])
    if (ok && L >= 2 && c0 == 0.f && slope >= 0.f && all_lin) {
      r.linear = 1;
      r.slope = slope;
      r.cmax = tail;
    }
  }
  if (lane == 0) *d = r;
}

// ------------------------------------------------------------------------------------------------
// elementwise kernels.  V floats per lane and access (4 when every plane is 16-byte aligned and the
// plane size is a multiple of 4, else 1); ND: number of directions when it is one of the usual ones
// (loads of all planes are then issued back to back), 0: run-time loop.
// ------------------------------------------------------------------------------------------------
// NT: the non-temporal hint on loads and stores (planes are streamed once; ew_hint).
template <int V>
struct Pack {
  float v[V];
};
template <int V, bool NT>
__device__ __forceinline__ Pack<V> ld_pack(const float* p) {
  Pack<V> r;
  if constexpr (V == 4) {
    const f32x4 t = NT ? __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p))
                              : *reinterpret_cast<const f32x4*>(p);
    r.v[0] = t.x;
    r.v[1] = t.y;
    r.v[2] = t.z;
    r.v[3] = t.w;
  } else {
    r.v[0] = NT ? __builtin_nontemporal_load(p) : *p;
  }
  return r;
}
template <int V, bool NT>
__device__ __forceinline__ void st_pack(float* p, const Pack<V>& r) {
  if constexpr (V == 4) {
    f32x4 t;
    t.x = r.v[0];
    t.y = r.v[1];
    t.z = r.v[2];
    t.w = r.v[3];
    if (NT)
      __builtin_nontemporal_store(t, reinterpret_cast<f32x4*>(p));
    else
      *reinterpret_cast<f32x4*>(p) = t;
  } else {
    if (NT)
      __builtin_nontemporal_store(r.v[0], p);
    else
      *p = r.v[0];
  }
}

// S = unary + sum_k m_k  (k ascending, as UpdateUnaryKernel sums, TRWP_forward.cu:70-73)
template <int V, int ND, bool NT>
__global__ void __launch_bounds__(256) belief_kernel(const float* __restrict__ unary,
                                                     const float* __restrict__ msg, int n_dir_rt,
                                                     int64_t N, float* __restrict__ S,
                                                     int* nonzero_flag, const int* only_if = nullptr) {
  // (only_if: a flag an earlier kernel of the stream has set or left clear; clear: nothing to do)
  if (only_if != nullptr && *only_if == 0) return;
  const int n_dir = ND > 0 ? ND : n_dir_rt;
  bool any = false;  // some message of this thread's elements is not zero
  for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * V; i < N;
       i += (int64_t)gridDim.x * blockDim.x * V) {
    Pack<V> v = ld_pack<V, NT>(unary + i);
    if constexpr (ND > 0) {
      Pack<V> m[ND];
#pragma unroll
      for (int k = 0; k < ND; ++k) m[k] = ld_pack<V, NT>(msg + (int64_t)k * N + i);
#pragma unroll
      for (int k = 0; k < ND; ++k)
#pragma unroll
        for (int j = 0; j < V; ++j) {
          v.v[j] += m[k].v[j];
          any = any || (m[k].v[j] != 0.f);
        }
    } else {
      for (int k = 0; k < n_dir; ++k) {
        const Pack<V> m = ld_pack<V, NT>(msg + (int64_t)k * N + i);
#pragma unroll
        for (int j = 0; j < V; ++j) {
          v.v[j] += m.v[j];
          any = any || (m.v[j] != 0.f);
        }
      }
    }
    st_pack<V, NT>(S + i, v);
  }
  if (nonzero_flag != nullptr && any) *nonzero_flag = 1;  // every writer stores the same value
}

// Sets *flag when some element of the n_dir message planes is not zero (every writer stores the
// same value).  The reference's callers pass cleared message tensors; knowing that on the device
// lets the first sweeps read the unary terms in place of planes that would have to be built first.
template <int V, int ND, bool NT>
__global__ void __launch_bounds__(256) check_nonzero_kernel(const float* __restrict__ msg,
                                                            int n_dir_rt, int64_t N, int* flag) {
  const int n_dir = ND > 0 ? ND : n_dir_rt;
  bool any = false;
  for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * V; i < N;
       i += (int64_t)gridDim.x * blockDim.x * V) {
    if constexpr (ND > 0) {
      Pack<V> m[ND];
#pragma unroll
      for (int k = 0; k < ND; ++k) m[k] = ld_pack<V, NT>(msg + (int64_t)k * N + i);
#pragma unroll
      for (int k = 0; k < ND; ++k)
#pragma unroll
        for (int j = 0; j < V; ++j) any = any || (m[k].v[j] != 0.f);
    } else {
      for (int k = 0; k < n_dir; ++k) {
        const Pack<V> m = ld_pack<V, NT>(msg + (int64_t)k * N + i);
#pragma unroll
        for (int j = 0; j < V; ++j) any = any || (m.v[j] != 0.f);
      }
    }
  }
  if (any) *flag = 1;
}

// ISGMR: every direction of an iteration reads the old messages only through
//   U_d = rho * (unary + sum_k m_k - m_d) - m_{d^1}      (UpdateUnaryKernel, ISGMR_forward.cu:101-121)
// so U_d is stored once per iteration (in place of m_d, or into the other message buffer) before
// the sweeps: a sweep then reads one plane per pixel, not three.
template <int V, int ND, bool NT>
__global__ void __launch_bounds__(256) isgmr_unary_kernel(const float* __restrict__ unary,
                                                          const float* msg, float* out,
                                                          int n_dir_rt, int64_t N, float rho,
                                                          int pair_share, const int* only_if = nullptr) {
  if (only_if != nullptr && *only_if == 0) return;  // (see belief_kernel)
  constexpr int KD = ND > 0 ? ND : kMaxDirs;
  const int n_dir = ND > 0 ? ND : n_dir_rt;
  for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * V; i < N;
       i += (int64_t)gridDim.x * blockDim.x * V) {
    Pack<V> S = ld_pack<V, NT>(unary + i);
    Pack<V> m[KD];
#pragma unroll
    for (int k = 0; k < KD; ++k) {
      if (k < n_dir) {
        m[k] = ld_pack<V, NT>(msg + (int64_t)k * N + i);
      } else {
#pragma unroll
        for (int j = 0; j < V; ++j) m[k].v[j] = 0.f;
      }
    }
#pragma unroll
    for (int k = 0; k < KD; ++k)
      if (k < n_dir) {
#pragma unroll
        for (int j = 0; j < V; ++j) S.v[j] += m[k].v[j];  // k ascending, as the reference sums
      }
#pragma unroll
    for (int k = 0; k < KD; ++k) {
      // pair_share (rho == 1): U_d and U_{d^1} are both S - m_d - m_{d^1}; one plane per pair is
      // stored (they differ by the order of the two subtractions, at most 2 ulp of S)
      if (k < n_dir && !(pair_share && (k & 1))) {
        Pack<V> u;
#pragma unroll
        for (int j = 0; j < V; ++j) u.v[j] = fmaf(S.v[j] - m[k].v[j], rho, -m[k ^ 1].v[j]);
        st_pack<V, NT>(out + (int64_t)k * N + i, u);  // out == msg: in place
      }
    }
  }
}

// cost = factor*unary + sum_k m_k  (or + min_k m_k): CostAggregateKernel, TRWP_forward.cu:31-58,
// ISGMR_forward.cu:69-99.
template <int V, int ND, bool NT>
__global__ void __launch_bounds__(256) aggregate_kernel(const float* __restrict__ unary,
                                                        const float* __restrict__ msg, int n_dir_rt,
                                                        int64_t N, float factor, int min_a_dir,
                                                        float* __restrict__ cost) {
  const int n_dir = ND > 0 ? ND : n_dir_rt;
  for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * V; i < N;
       i += (int64_t)gridDim.x * blockDim.x * V) {
    Pack<V> v = ld_pack<V, NT>(unary + i);
#pragma unroll
    for (int j = 0; j < V; ++j) v.v[j] *= factor;
    Pack<V> mn;  // min_a_dir only
    auto fold = [&](int k, const Pack<V>& m) {
#pragma unroll
      for (int j = 0; j < V; ++j) {
        if (!min_a_dir)
          v.v[j] += m.v[j];  // ((unary + m_0) + m_1) + ... as the reference adds
        else if (k == 0)
          mn.v[j] = m.v[j];
        else
          mn.v[j] = (m.v[j] < mn.v[j]) ? m.v[j] : mn.v[j];
      }
    };
    if constexpr (ND > 0) {
      Pack<V> m[ND];
#pragma unroll
      for (int k = 0; k < ND; ++k) m[k] = ld_pack<V, NT>(msg + (int64_t)k * N + i);
#pragma unroll
      for (int k = 0; k < ND; ++k) fold(k, m[k]);
    } else {
      for (int k = 0; k < n_dir; ++k) fold(k, ld_pack<V, NT>(msg + (int64_t)k * N + i));
    }
    if (min_a_dir) {
#pragma unroll
      for (int j = 0; j < V; ++j) v.v[j] += mn.v[j];
    }
    st_pack<V, NT>(cost + i, v);
  }
}

// The same with the labels first in the result (MPL_F_COST_LABELS_FIRST): a workgroup sums `tile` consecutive pixels of
// an image, one run of memory in every plane whatever the label count, and turns them over through LDS (an odd row
// stride), so the sums are not stored and read once more to change their layout.  Bound by HBM.  Tiles beside each other
// share lines of the result where a row of it is no whole number of them: groups of tiles go to one die, as the
// transposes' do (mp_layout.hip), and only whole lines carry the hint (NT_ST).  Measured, us, sum and transpose -> this:
// 128 labels 375x1242, 8 directions 414 + 131 -> 416; 96 labels 384x1248, 4 directions 180 + 90 -> 186; 21 labels
// 12x65x65, 8 directions 8.4 + 11 -> 8.4 (32 with tiles of 128 pixels, too few of them), 4x129x129, 4 directions 7 + 14 -> 6.
template <int V, int ND, bool NT, bool NT_ST>
__global__ void __launch_bounds__(256) aggregate_first_kernel(const float* __restrict__ unary,
                                                              const float* __restrict__ msg, int n_dir_rt,
                                                              int64_t N, int HW, int L, int tile_log, float factor,
                                                              int min_a_dir, float* __restrict__ cost) {
  extern __shared__ float turn[];  // [pixel][L | 1]
  const int n_dir = ND > 0 ? ND : n_dir_rt;
  const int tile = 1 << tile_log, stride = L | 1;
  const int p0 = xcd_block((int)blockIdx.x, (int)gridDim.x, 8) << tile_log;
  const int pixels = HW - p0 < tile ? HW - p0 : tile;
  for (int64_t b = blockIdx.y; b * HW * L < N; b += gridDim.y) {
    const int64_t first = (b * HW + p0) * L;
    const int lead = V == 4 ? (int)first & 3 : 0;  // (fours of the planes, not of the tile)
    const bool whole = V == 1 || (lead == 0 && ((pixels * L) & 3) == 0);
    for (int e = (int)threadIdx.x * V - lead; e < pixels * L; e += 256 * V) {
      const int64_t i = first + e;
      Pack<V> v = ld_pack<V, NT>(unary + i);
#pragma unroll
      for (int j = 0; j < V; ++j) v.v[j] *= factor;
      Pack<V> mn;  // min_a_dir only
      auto fold = [&](int k, const Pack<V>& m) {
#pragma unroll
        for (int j = 0; j < V; ++j) {
          if (!min_a_dir)
            v.v[j] += m.v[j];  // ((unary + m_0) + m_1) + ... as the reference adds
          else if (k == 0)
            mn.v[j] = m.v[j];
          else
            mn.v[j] = (m.v[j] < mn.v[j]) ? m.v[j] : mn.v[j];
        }
      };
      if constexpr (ND > 0) {
        Pack<V> m[ND];
#pragma unroll
        for (int k = 0; k < ND; ++k) m[k] = ld_pack<V, NT>(msg + (int64_t)k * N + i);
#pragma unroll
        for (int k = 0; k < ND; ++k) fold(k, m[k]);
      } else {
        int k = 0;
        if constexpr (V == 1) {  // (four planes' loads at a time: 97 labels 241x321, 12 directions 164 -> 85 us, 6 directions 90 -> 64)
          for (; k + 4 <= n_dir; k += 4) {
            Pack<V> m[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) m[q] = ld_pack<V, NT>(msg + (int64_t)(k + q) * N + i);
#pragma unroll
            for (int q = 0; q < 4; ++q) fold(k + q, m[q]);
          }
        }
        for (; k < n_dir; ++k) fold(k, ld_pack<V, NT>(msg + (int64_t)k * N + i));
      }
      if (min_a_dir) {
#pragma unroll
        for (int j = 0; j < V; ++j) v.v[j] += mn.v[j];
      }
      int p = e / L, l = e - p * L;
      const auto put = [&](const auto checked) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < V; ++j) {
          if (!decltype(checked)::value || (unsigned)(e + j) < (unsigned)(pixels * L)) turn[p * stride + l] = v.v[j];
          if (++l == L) {
            l = 0;
            ++p;
          }
        }
      };
      if (whole)
        put(std::false_type());
      else
        put(std::true_type());
    }
    __syncthreads();
    float* const out = cost + b * HW * L + p0;
    for (int x = threadIdx.x; x < L << tile_log; x += 256) {
      const int l = x >> tile_log, p = x & (tile - 1);
      if (p >= pixels) continue;
      if (NT_ST)
        __builtin_nontemporal_store(turn[p * stride + l], out + (int64_t)l * HW + p);
      else
        out[(int64_t)l * HW + p] = turn[p * stride + l];
    }
    __syncthreads();
  }
}

// label = argmin_l cost(l), smallest label on ties: CalLabelKernel, TRWP_forward.cu:8-29, with the
// cost of CostAggregateKernel recomputed on the fly.  One wave per pixel.
__global__ void __launch_bounds__(256) label_kernel(const float* __restrict__ unary,
                                                    const float* __restrict__ msg, int n_dir,
                                                    int64_t P, int L, float factor, int min_a_dir,
                                                    uint8_t* __restrict__ label) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t N = P * L;
  const int64_t wave0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int64_t n_waves = ((int64_t)gridDim.x * blockDim.x) / kWave;
  for (int64_t pix = wave0; pix < P; pix += n_waves) {
    float best = INFINITY;
    int arg = 0x7fffffff;
    for (int l = lane; l < L; l += kWave) {
      int64_t i = pix * L + l;
      float v = unary[i] * factor;
      if (min_a_dir) {
        float mn = msg[i];
        for (int k = 1; k < n_dir; ++k) {
          float m = msg[(int64_t)k * N + i];
          if (m < mn) mn = m;
        }
        v += mn;
      } else {
        for (int k = 0; k < n_dir; ++k) v += msg[(int64_t)k * N + i];
      }
      if (v < best) {
        best = v;
        arg = l;
      }
    }
    float gmin = wave_min(best);
    // smallest label among the lanes that hold the minimum; a lane's own arg is its smallest
    float cand = (best == gmin) ? (float)arg : INFINITY;
    float amin = wave_min(cand);
    if (lane == 0) label[pix] = (uint8_t)((amin < (float)L) ? (int)amin : 0);
  }
}

// The same for label counts that are a multiple of 4: a group of `group` lanes (a power of two
// >= L/4) per pixel, 16 bytes per lane and plane, 64/group pixels per wavefront; the argmin is a
// butterfly over the group on (value, label) pairs.
// The pass reads what three others read (every message plane and the unary terms), and memory bounds
// them all, so where one of them is due next its result is stored from here and it is not run:
//   kLabelSum: the sum itself (cost_final after the last iteration, TRWP's re-summed belief plane),
//   kLabelU:   ISGMR's U planes of the next iteration over the messages (isgmr_unary_kernel).
// The sums are formed in the order of those kernels: the same bits.  50 iterations on 375x450x60 with all
// labels, passes apart -> together: TRWP, 8 directions 33.2 -> 32.4 ms, 4 directions 15.8 -> 15.4; ISGMR,
// 8 directions 19.6 -> 16.8 ms (16 labels 7.03 -> 6.39), 4 directions 11.1 -> 10.9 (its scans form U).
// The loads of all planes going out back to back are not what gives it: 10 iterations, TRWP 6.20 -> 5.99 ms
// and ISGMR 3.75 -> 3.19, but 6.18 -> 6.14 and 3.76 -> 3.72 with min_a_dir, where nothing is merged.
constexpr int kLabelOnly = 0, kLabelSum = 1, kLabelU = 2;
template <int ND, int OUT, bool NT>
__global__ void __launch_bounds__(256) label_quad_kernel(const float* __restrict__ unary,
                                                         const float* msg, int n_dir_rt, int64_t P,
                                                         int L, int group, float factor,
                                                         int min_a_dir, uint8_t* __restrict__ label,
                                                         float* out, float rho, int pair_share) {
  static_assert(ND > 0 || OUT != kLabelU, "the U planes need all messages in registers");
  const int n_dir = ND > 0 ? ND : n_dir_rt;
  const int64_t N = P * L;
  const int sub = threadIdx.x & (group - 1);
  const int64_t pix = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / group;
  float best = INFINITY;
  int arg = 0x7fffffff;
  if (pix < P && sub * 4 < L) {
    const int64_t i = pix * L + sub * 4;
    Pack<4> v = ld_pack<4, NT>(unary + i);
    Pack<4> m[ND > 0 ? ND : 1];
    if constexpr (ND > 0) {
#pragma unroll
      for (int k = 0; k < ND; ++k) m[k] = ld_pack<4, NT>(msg + (int64_t)k * N + i);
    }
    auto message = [&](int k) { return ND > 0 ? m[ND > 0 ? k : 0] : ld_pack<4, NT>(msg + (int64_t)k * N + i); };
#pragma unroll
    for (int j = 0; j < 4; ++j) v.v[j] *= factor;
    if (OUT == kLabelOnly && min_a_dir) {
      Pack<4> mn = message(0);
#pragma unroll
      for (int k = 1; k < n_dir; ++k) {
        const Pack<4> mk = message(k);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (mk.v[j] < mn.v[j]) mn.v[j] = mk.v[j];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) v.v[j] += mn.v[j];
    } else {
#pragma unroll
      for (int k = 0; k < n_dir; ++k) {
        const Pack<4> mk = message(k);
#pragma unroll
        for (int j = 0; j < 4; ++j) v.v[j] += mk.v[j];
      }
    }
    if constexpr (OUT == kLabelSum) st_pack<4, NT>(out + i, v);
    if constexpr (OUT == kLabelU) {
#pragma unroll
      for (int k = 0; k < ND; ++k)
        if (!(pair_share && (k & 1))) {
          Pack<4> u;
#pragma unroll
          for (int j = 0; j < 4; ++j) u.v[j] = fmaf(v.v[j] - m[k].v[j], rho, -m[k ^ 1].v[j]);
          st_pack<4, NT>(out + (int64_t)k * N + i, u);  // out == msg: in place
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (v.v[j] < best) {
        best = v.v[j];
        arg = sub * 4 + j;
      }
  }
  for (int o = 1; o < group; o <<= 1) {
    float ob = __shfl_xor(best, o);
    int oa = __shfl_xor(arg, o);
    if (ob < best || (ob == best && oa < arg)) {
      best = ob;
      arg = oa;
    }
  }
  if (pix < P && sub == 0) label[pix] = (uint8_t)((arg < L) ? arg : 0);
}

// Returns whether `out` has been written (want: what to store there besides the labels).
static bool launch_labels(const float* unary, const float* msg, int n_dir, int64_t P, int L,
                          float factor, int min_a_dir, uint8_t* label, hipStream_t st,
                          bool nt, int want = kLabelOnly, float* out = nullptr, float rho = 1.f,
                          int pair_share = 0) {
  const bool aligned = (((uintptr_t)unary | (uintptr_t)msg) & 15) == 0;
  if ((L & 3) != 0 || !aligned) {
    const int64_t waves = (P < 256 * 64) ? P : 256 * 64;
    label_kernel<<<(int)((waves + 3) / 4), 256, 0, st>>>(unary, msg, n_dir, P, L, factor, min_a_dir,
                                                         label);
    return false;
  }
  int group = 1;
  while (group * 4 < L) group <<= 1;
  const unsigned blocks = (unsigned)((P * group + 255) / 256);
  const bool known = n_dir == 4 || n_dir == 8 || n_dir == 16;
  // SGM's factor (the number of directions) is left to the pass of its own: it belongs to a single
  // iteration, and where it is no power of two its product rounds, or not, as either kernel fuses it into
  // the first sum
  if (min_a_dir || factor != 1.f || out == nullptr || ((uintptr_t)out & 15) != 0 ||
      (want == kLabelU && !known))
    want = kLabelOnly;
#define MPL_LABELS(ND, OUT)                                                                          \
  (nt ? label_quad_kernel<ND, OUT, true> : label_quad_kernel<ND, OUT, false>)<<<blocks, 256, 0, st>>>( \
      unary, msg, n_dir, P, L, group, factor, min_a_dir, label, out, rho, pair_share)
#define MPL_LABELS_ND(ND)                             \
  do {                                                \
    if (want == kLabelU)                              \
      MPL_LABELS(ND, kLabelU);                        \
    else if (want == kLabelSum)                       \
      MPL_LABELS(ND, kLabelSum);                      \
    else                                              \
      MPL_LABELS(ND, kLabelOnly);                     \
  } while (0)
  switch (n_dir) {
    case 4: MPL_LABELS_ND(4); break;
    case 8: MPL_LABELS_ND(8); break;
    case 16: MPL_LABELS_ND(16); break;
    default:
      if (want == kLabelSum)
        MPL_LABELS(0, kLabelSum);
      else
        MPL_LABELS(0, kLabelOnly);
  }
#undef MPL_LABELS_ND
#undef MPL_LABELS
  return want != kLabelOnly;
}

// ISGMR: after all directions of an iteration have been scanned back (X_k = dU_k):
//   dunary += rho * sum_k X_k ;  gu_k = rho * (sum - X_k) - X_{k^1}   (written to G)
// (UpdateUnaryKernelBack summed over directions + SumMsgKernel, ISGMR_backward.cu:39-60, 482-483)
template <int V, int ND, bool NT>
__global__ void __launch_bounds__(256) isgmr_combine_kernel(const float* X, float* G, int n_dir_rt,
                                                            int64_t N, float rho,
                                                            const float* __restrict__ dcost,
                                                            float factor, int init_dunary,
                                                            int write_gu, int pair_share,
                                                            float* __restrict__ dunary) {
  constexpr int KD = ND > 0 ? ND : kMaxDirs;
  const int n_dir = ND > 0 ? ND : n_dir_rt;
  for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * V; i < N;
       i += (int64_t)gridDim.x * blockDim.x * V) {
    Pack<V> x[KD];
#pragma unroll
    for (int k = 0; k < KD; ++k) {
      if (k < n_dir) {
        x[k] = ld_pack<V, NT>(X + (int64_t)k * N + i);
      } else {
#pragma unroll
        for (int j = 0; j < V; ++j) x[k].v[j] = 0.f;
      }
    }
    Pack<V> du = init_dunary ? ld_pack<V, NT>(dcost + i) : ld_pack<V, NT>(dunary + i);
    Pack<V> sum;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      sum.v[j] = 0.f;
#pragma unroll
      for (int k = KD - 1; k >= 0; --k)
        if (k < n_dir) sum.v[j] += x[k].v[j];
      if (init_dunary) du.v[j] *= factor;
      du.v[j] = fmaf(rho, sum.v[j], du.v[j]);
    }
    st_pack<V, NT>(dunary + i, du);
    if (write_gu) {
#pragma unroll
      for (int k = 0; k < KD; ++k) {
        // pair_share (rho == 1): gu_k and gu_{k^1} are both sum - X_k - X_{k^1}; one plane per
        // pair is stored (G == X: in place, every plane)
        if (k < n_dir && !(pair_share && (k & 1))) {
          Pack<V> g;
#pragma unroll
          for (int j = 0; j < V; ++j) g.v[j] = fmaf(rho, sum.v[j] - x[k].v[j], -x[k ^ 1].v[j]);
          st_pack<V, NT>(G + (int64_t)k * N + i, g);
        }
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------------------
// Tables the reverse scans take turns on for dcontext, and the chains of a call, over all its iterations, from
// which they pay for the pass that sums them (mpl_dcontext_copies).  Measured, backward with all gradients, us per
// call without and with 8 tables (16, 32 and 64 are the same): 21 labels, a 2-D table, TRWP 2 directions 205x129
// (4100 chains) 491 -> 465, 4x129x129 680 -> 611, ISGMR 2x65x65 164 -> 136, 12x65x65 560 -> 436, 12x129x129 1525 ->
// 1251; 1-D tables, 64 labels TRWP 103x103 1484 -> 1475, 96 labels ISGMR 240x320 1812 -> 1630, TRWP 1477 both.
constexpr int kDctxCopies = 8;
constexpr int64_t kDctxMinChains = 4096;

thread_local char g_err[512] = "";

// Optional per-kernel timing with HIP events on the launch stream (off unless mpl_profile_begin
// was called): lets a benchmark read each kernel's average duration without an external profiler.
struct ProfRec {
  int kind;
  int sweeps;  // direction sweeps the launch stands for (2 for a fused pair)
  hipEvent_t start, stop;
};
struct Profiler {
  std::atomic<bool> on{false};
  std::vector<ProfRec> recs;
  std::vector<hipEvent_t> pool;
  hipEvent_t get_event() {
    if (!pool.empty()) {
      hipEvent_t e = pool.back();
      pool.pop_back();
      return e;
    }
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
  }
};
Profiler g_prof;
std::mutex g_prof_mu;

struct Timed {
  hipStream_t st;
  hipEvent_t stop = nullptr;
  Timed(int kind, hipStream_t s, int sweeps = 1) : st(s) {
    if (!g_prof.on.load(std::memory_order_acquire)) return;
    std::lock_guard<std::mutex> lk(g_prof_mu);
    ProfRec r;
    r.kind = kind;
    r.sweeps = sweeps;
    r.start = g_prof.get_event();
    r.stop = g_prof.get_event();
    if (r.start == nullptr || r.stop == nullptr) return;
    (void)hipEventRecord(r.start, st);
    stop = r.stop;
    g_prof.recs.push_back(r);
  }
  ~Timed() {
    if (stop != nullptr) (void)hipEventRecord(stop, st);
  }
};

int check_shape(const mpl_shape* s, int n_iter) {
  if (s == nullptr) return fail(MPL_EINVAL, "shape is null");
  if (s->n_dir < 2 || s->n_dir > kMaxDirs || (s->n_dir & 1))
    return fail(MPL_EINVAL, "n_dir must be even and in [2, %d], got %d", kMaxDirs, s->n_dir);
  if (s->batch < 1 || s->height < 1 || s->width < 1)
    return fail(MPL_EINVAL, "batch/height/width must be positive, got %d/%d/%d", s->batch,
                s->height, s->width);
  if (s->n_disp < 1 || s->n_disp > kMaxL)
    return fail(MPL_EINVAL, "n_disp must be in [1, %d] (uint8 argmin indices), got %d", kMaxL,
                s->n_disp);
  if (s->ctx2d && s->n_disp > kMaxCtx2dL)
    return fail(MPL_EINVAL, "a 2-D context table needs n_disp <= %d, got %d", kMaxCtx2dL,
                s->n_disp);
  if (n_iter < 1) return fail(MPL_EINVAL, "n_iter must be positive, got %d", n_iter);
  int64_t P = (int64_t)s->batch * s->height * s->width;
  if (P > 0x7fffffff) return fail(MPL_EINVAL, "more than 2^31 pixels");
  // pixels are addressed with 32-bit byte offsets from the first pixel of their batch item
  if ((int64_t)s->height * s->width * s->n_disp * 4 > kMaxImageBytes)
    return fail(MPL_EINVAL, "one batch item (height*width*n_disp floats) must stay below 4 GiB");
  int64_t max_blocks = 0;
  for (int d = 0; d < s->n_dir; ++d)
    max_blocks += (int64_t)s->batch * make_dir(d, s->height, s->width).n_chains;
  if (max_blocks > 0x7fffffff) return fail(MPL_EINVAL, "more than 2^31 chains");
  return MPL_OK;
}

int launch_ok(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MPL_ELAUNCH, "%s: %s", what, hipGetErrorString(e));
  return MPL_OK;
}

// Workgroups of an element-wise kernel over n accesses (of 4 floats or of 1): one access per thread.
// One pass over the data with as many workgroups as it takes measured 3-8 % faster than a
// grid-stride loop of 32 workgroups per CU on the 2.3 GB planes, and 2 / 4 / 8 accesses per thread
// measured 2 / 5 / 9 % slower than one (workgroups of 64, 128 and 512 threads: 4 to 5 % slower than
// 256); the cap only bounds the grid.
#ifndef MPL_EW_BLOCKS_PER_CU
#define MPL_EW_BLOCKS_PER_CU 4096
#endif
int elementwise_blocks(int64_t n) {
  int64_t b = (n + 256 - 1) / 256;
  if (b < 1) b = 1;
  if (b > 256 * MPL_EW_BLOCKS_PER_CU) b = 256 * MPL_EW_BLOCKS_PER_CU;
  return (int)b;
}

// Whether the element-wise passes over the planes carry the non-temporal hint: not where the messages fit the
// last-level cache (256 MB) and the label vectors share lines, whose scans read and write without it (load_policy).
// Measured, ISGMR with 8 directions, without over with, forward / keeping argmin labels / backward: 21 labels
// 12x65x65 (34 MB of messages) 0.98 / 0.98 / 0.98, 12x129x129 (134 MB) 0.92 / 0.99 / 1.01; 60 labels 100x150 0.93 / 0.97 /
// 0.99, 200x250 0.91 / 0.97 / 1.00, 300x400 (220 MiB) 1.09 / 1.09 / 1.05; 150 labels 180x250 (206 MiB) 0.94 / 0.93 / 0.99,
// 300x400 1.03 / 1.01 / 1.04; 100 labels 200x300 0.93 / 0.94 / 0.98.  Whole lines: 64 labels 100x150 1.04, 300x400 1.03;
// 96 labels 384x1248 1.04.
constexpr int64_t kCachedMessages = (int64_t)208 << 20;
int64_t message_bytes(const mpl_shape* s) { return (int64_t)s->n_dir * s->batch * s->height * s->width * s->n_disp * 4; }
bool ew_hint(const mpl_shape* s) {
  return (s->n_disp * 4) % kLineBytes == 0 || message_bytes(s) > kCachedMessages;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Picks the instantiation of an element-wise kernel: 4 floats per access when the planes allow it,
// the direction count as a compile-time constant when it is 4, 8 or 16.
#define MPL_EW_LAUNCH(KERNEL, VEC4, NT, NDIR, N, ST, ...)                                         \
  do {                                                                                           \
    if (NT)                                                                                      \
      MPL_EW_LAUNCH_NT(KERNEL, VEC4, true, NDIR, N, ST, __VA_ARGS__);                            \
    else                                                                                         \
      MPL_EW_LAUNCH_NT(KERNEL, VEC4, false, NDIR, N, ST, __VA_ARGS__);                           \
  } while (0)
#define MPL_EW_LAUNCH_NT(KERNEL, VEC4, NT, NDIR, N, ST, ...)                                      \
  do {                                                                                           \
    const int blocks_ = elementwise_blocks((VEC4) ? (N) / 4 : (N));                              \
    if (VEC4) {                                                                                  \
      switch (NDIR) {                                                                            \
        case 4: KERNEL<4, 4, NT><<<blocks_, 256, 0, ST>>>(__VA_ARGS__); break;                   \
        case 8: KERNEL<4, 8, NT><<<blocks_, 256, 0, ST>>>(__VA_ARGS__); break;                   \
        case 16: KERNEL<4, 16, NT><<<blocks_, 256, 0, ST>>>(__VA_ARGS__); break;                 \
        default: KERNEL<4, 0, NT><<<blocks_, 256, 0, ST>>>(__VA_ARGS__); break;                  \
      }                                                                                          \
    } else {                                                                                     \
      KERNEL<1, 0, NT><<<blocks_, 256, 0, ST>>>(__VA_ARGS__);                                    \
    }                                                                                            \
  } while (0)

void fill_dirs(const mpl_shape* s, int first, int count, int* dirs, int* prefix, int* n_dirs) {
  *n_dirs = count;
  prefix[0] = 0;
  for (int i = 0; i < count; ++i) {
    dirs[i] = first + i;
    prefix[i + 1] = prefix[i] + s->batch * make_dir(first + i, s->height, s->width).n_chains;
  }
}

int labels_per_lane(int L) { return (L + kWave - 1) / kWave; }

// process defaults of the per-call choices (mpl_set_option); a call reads them once
std::atomic<int> g_packed_scans{1};  // MPL_OPT_PACKED_SCANS: 0 off, 1 by chain count, 2 always
std::atomic<int> g_fused_u{1};       // MPL_OPT_FUSED_U
std::atomic<int> g_belief_rebuild{MPL_BELIEF_REBUILD_DEFAULT};  // MPL_OPT_BELIEF_REBUILD
std::atomic<int> g_team_scans{1};    // MPL_OPT_TEAM_SCANS: 0 never, 1 launches with few chains, 2 whatever their number
std::atomic<int> g_split_waves{0};   // MPL_OPT_DENSE_SPLIT_WAVES: 0 = by the model of choose_split

// what one call does, from its flags and the process defaults
struct CallOpts {
  int packed;   // 0 off, 1 by chain count, 2 always
  bool fused_u;
  bool fused_pairs;
  bool dense_table;
  int split_waves;  // MPL_OPT_DENSE_SPLIT_WAVES
  int team;         // MPL_OPT_TEAM_SCANS
};

int read_flags(unsigned flags, const char* what, CallOpts* o) {
  if (flags & ~MPL_F_ALL) return fail(MPL_EINVAL, "%s: unknown flag bits 0x%x", what, flags & ~MPL_F_ALL);
  if ((flags & MPL_F_PACKED_OFF) && (flags & MPL_F_PACKED_ALWAYS))
    return fail(MPL_EINVAL, "%s: MPL_F_PACKED_OFF and MPL_F_PACKED_ALWAYS exclude each other", what);
  o->packed = (flags & MPL_F_PACKED_OFF) ? 0
              : (flags & MPL_F_PACKED_ALWAYS) ? 2 : g_packed_scans.load(std::memory_order_relaxed);
  o->fused_u = (flags & MPL_F_FUSED_U_OFF) ? false : g_fused_u.load(std::memory_order_relaxed) != 0;
  o->fused_pairs = (flags & MPL_F_FUSED_PAIRS_OFF) == 0;
  o->dense_table = (flags & MPL_F_DENSE_TABLE) != 0;
  o->split_waves = g_split_waves.load(std::memory_order_relaxed);
  o->team = g_team_scans.load(std::memory_order_relaxed);
  return MPL_OK;
}

// Chains per wavefront of the launch described by p (its directions filled in): the one place where
// a launch is given to the packed scans (>= 2) or to the one-chain-per-wavefront kernels (0).
// Everything that depends on that choice (the launcher, the number of wavefronts, whether the
// Jacobi scans form U themselves) reads p.pack.
template <typename Params>
int decide_pack(const mpl_shape* s, const Params& p, const CallOpts& o) {
  if (!o.packed) return 0;
  const int G = packed_chains_per_wave(s->batch, s->height, s->width, s->n_disp, s->ctx2d != 0,
                                       p.block_prefix[p.n_dirs], o.packed == 2);
  return G >= 2 ? G : 0;
}

// Chains that run at once in a launch of one direction: its pixels over its longest chain.  The chains of rows
// and columns are of one length, and this is their number; those of a diagonal start long before the
// longest ends, and what bounds the launch is its longest chain and the pixels the chip has to walk, not how
// many workgroups there are.  With it in place of the number of chains, TRWP with 8 directions, 3 iterations,
// ms per call: forward, 60 labels 375x450 (824 diagonals) 1.28 -> 1.08; training 96 labels 350x500 3.08 / 3.31 ->
// 2.18 / 2.07, 192 labels 500x700 (1199 diagonals) 6.66 / 6.39 -> 6.03 / 4.87; energy minimisation 375x450x60
// 23.2 -> 20.4.
int chains_at_once(int dir, int B, int H, int W) {
  int hs, ws;
  dir_step(dir, &hs, &ws);
  hs = hs < 0 ? -hs : hs;
  ws = ws < 0 ? -ws : ws;
  int longest = INT_MAX;
  if (hs) longest = std::min(longest, (H + hs - 1) / hs);
  if (ws) longest = std::min(longest, (W + ws - 1) / ws);
  return (int)(((int64_t)B * H * W + longest - 1) / longest);
}
template <typename Params>
int chains_at_once(const Params& p) {
  return chains_at_once(p.dirs[0], p.B, p.H, p.W);
}

// Four wavefronts per chain in the reverse scans (mp_bwd_team.hip): chains per compute unit up to which
// a launch takes them, 0 for never.  The time of such a launch steps up with every further chain per
// compute unit, so the lines lie between those steps, where no kind of call measured slower than with
// one wavefront per chain by more than two runs of it differ.  The table and which gradients are wanted
// change the ratio but may not change the route: the table is not known here, and dunary is promised to be
// the same bits whichever gradients are wanted.  Measured, backward of 2 iterations on square images with
// 4, 8 and 16 directions (TRWP: chains of one direction per launch, ISGMR: of all), time with one over
// time with four wavefronts: the least of dunary alone and of all gradients on a band of four labels, a
// bent band, a linear and a random table / the greatest.  (Taken while the main wavefronts of a unit's chains
// shared a SIMD, which cost this side where there are two or three: 150 labels 300x500 2.68 -> 2.20 ms since.)
//   * up to 64 labels: TRWP 256 chains 0.78 / 1.65, 768 chains with 33 labels 0.75 / 1.2, ISGMR 0.69 / 1.5.
//     With one label per lane the step of mp_bwd.hip is short, and labels that point anywhere cost this
//     kernel more (64 labels, dunary alone: 199 ns per pixel and walk there, 245 here).  Never taken.
//   * TRWP, 768 chains: 65 labels 1.12 / 2.2, 128 labels 1.23 / 2.0, 192 labels 1.17 / 1.84, 224 labels
//     1.21 / 1.63, 256 labels 1.04 / 1.38; 800 chains: 65 labels 0.95 / 1.8, 256 labels 0.88 / 1.25; 832
//     chains: 192 labels 0.95 / 1.34.
//   * Labels loaded and stored one by one (their number no multiple of the labels per lane), which gains
//     less where several chains share a compute unit.  TRWP: 127 labels 768 chains 1.21 / 1.9; 152 / 158 / 190
//     labels 768 chains 1.04 / 1.64, 0.99 / 1.59, 0.83 / 1.44, 190 labels 512 chains 1.35 / 2.1; 193 labels
//     512 / 528 chains 1.14 / 2.0 and 0.89 / 1.31, 215 labels 1.02 / 1.81 and 0.79 / 1.32; 255 labels 256 /
//     384 / 512 chains 1.59 / 2.3, 0.97 / 1.71 and 0.78 / 1.45.  ISGMR: 191 labels 764 chains 1.05 / 1.37; 193
//     labels 512 chains 1.18 / 1.71; 255 labels 256 / 512 chains 1.48 / 2.0 and 0.95 / 1.54.
//   * ISGMR, 688 to 768 chains: 65 labels 0.98 / 1.9, 96 labels 1.06 / 1.6, 128 labels 0.99 / 1.46, 160 labels
//     1.07 / 1.46, 192 labels 0.98 / 1.32; 988 chains 0.91 / 2.1.  256 labels 512 chains 1.03 / 1.48, 640 chains
//     0.81 / 1.4; 200 labels 500 chains 1.24 / 1.64.
int team_chains_per_cu(int L, bool jacobi) {
  const int R = labels_per_lane(L);
  if (R == 1) return 0;  // (not compiled)
  if (L % R != 0) {      // labels one by one
    if (R == 4) return L <= 216 ? 2 : 1;
    if (R == 3 && !jacobi && L > 152) return 2;
  }
  return R == 4 && jacobi ? 2 : 3;
}

// 21 labels with a 2-D table (mp_team21.hip), one over four wavefronts on images of 129x129, batch 1 / 4 / 8 /
// 12 (129 / 516 / 1032 / 1548 chains).  Forward, argmin labels kept: 2.05 / 1.95 / 1.51 / 1.48; rows without
// them 1.51 with 256, 1.46 with 1024, 1.53 with 2048 chains.  Backward, dunary alone: 1.35 / 1.21 / 0.99 /
// 0.82, with both other gradients 1.85 / 1.47 / 1.08 / 1.21; 65x65, batch 12 (780 chains) 0.85 and 1.11.
// Soft-weighted, five iterations forward and backward, ms with the reverse scan on one -> on four wavefronts, the
// forward scan on one: 135 chains 1.85 -> 1.53, 258 chains 3.85 -> 3.10, 516 chains 4.97 -> 4.02, 516 / 660
// chains 5.74 -> 4.70.
// (More than 2048 chains: the packed scans.)
constexpr int kTeam21FwdChainsPerCu = 8;
constexpr int kTeam21BwdChainsPerCu = 3;
// Its forward scan, two iterations on images of 129x129, one over four wavefronts, duals kept / not: 129 chains 1.65
// / 1.32, 516 chains 1.57 / 1.35, 774 chains 1.16 / 1.22, 1032 chains 1.07 / 1.00, 2064 chains 1.07 / 0.89.
constexpr int kTeam21SoftFwdChainsPerCu = 4;

int decide_team(const BackParams& p, const CallOpts& o, bool jacobi) {
  if (p.pack >= 2 || o.team == 0) return 0;
  if (p.ctx2d && p.L == 21 && !jacobi)
    return o.team == 2 || chains_at_once(p) <= kTeam21BwdChainsPerCu * (launch_policy().n_simd / 4) ? 1 : 0;
  if (p.ctx2d || p.L <= kWave) return 0;
  if (o.team == 2) return 1;
  const int cus = launch_policy().n_simd / 4;
  // (A Jacobi launch holds every direction; its lines were measured in chains of all of them.  With four labels
  // per lane the LDS holds two workgroups of a unit and every chain counts, however early it ends: 200 labels
  // 32x34, batch 12, 8 directions, min(k, 14)^2, 780 diagonals, all directions 0.69 ms so, 0.74 by chains_at_once.)
  const int chains = jacobi || labels_per_lane(p.L) == 4 ? p.block_prefix[p.n_dirs] : chains_at_once(p);
  return chains <= team_chains_per_cu(p.L, jacobi) * cus ? 1 : 0;
}

// The same for the forward scans of TRWP (mp_fwd_team.hip; the same bits either way).  Measured on rows of
// 300 pixels with 192 to 1024 chains, Potts, truncated linear and quadratic, random tables, ns per pixel
// with one over ns with four wavefronts, the least over the tables / the greatest.  With argmin labels kept,
// which the helpers find:
//   * up to 64 labels: 256 chains 1.26 / 1.70, 768 chains 1.16 / 1.35, 1024 chains 0.98 / 1.30;
//   * up to 128: 256 chains 1.41 / 3.72, 768 chains 1.22 / 2.37, 1024 chains 0.96 / 1.88;
//   * up to 192: 256 chains 1.36 / 1.94, 768 chains 1.11 / 1.75, 1024 chains 0.66 / 1.05;
//   * up to 256: 256 chains 2.07 / 2.60, 512 chains 1.38 / 1.81, 768 chains 0.92 / 1.05.
// Without them:
//   * up to 64 labels: 768 chains 1.02 / 1.62, 1024 chains 0.89 / 1.37;
//   * up to 128: 512 chains 1.05 / 1.36, 768 chains 0.86 / 1.12;
//   * up to 192: 768 chains 1.03 / 1.24;  up to 256: 768 chains 1.05 / 1.08.
// Labels loaded and stored one by one (their number no multiple of the labels per lane), kept / not: up to 128
// 768 chains 1.11, 1024 chains 0.88 / 256 chains 1.28, 384 chains 1.02, 512 chains 0.98; up to 192 512
// chains 1.32, 768 chains 0.92 / 256 chains 1.27, 384 chains 0.76; up to 256 256 chains 1.37, 384 chains
// 0.89 / 192 chains 0.84.
int team_fwd_chains_per_cu(int L, bool train) {
  const int R = labels_per_lane(L);
  if (L % R == 0) return (R == 4 && train) || (R == 2 && !train) ? 2 : 3;
  if (train) return 5 - R;
  return R < 4 ? 1 : 0;
}

int decide_team_fwd(const SweepParams& p, const CallOpts& o, bool train) {
  if (p.pack >= 2 || p.split >= 2 || o.team == 0) return 0;
  if (o.team == 2) return 1;
  const int per_cu = p.ctx2d && p.L == 21 ? kTeam21FwdChainsPerCu : team_fwd_chains_per_cu(p.L, train);
  return chains_at_once(p) <= per_cu * (launch_policy().n_simd / 4) ? 1 : 0;
}

bool decide_team21_soft_fwd(const SweepParams& p, const CallOpts& o) {
  if (o.team == 0) return false;
  return o.team == 2 || chains_at_once(p) <= kTeam21SoftFwdChainsPerCu * (launch_policy().n_simd / 4);
}

// Wavefronts per chain for the forward scan of a launch whose caller declared a dense 1-D table
// (MPL_F_DENSE_TABLE) with several labels per lane: four (one on every SIMD of a compute unit, each
// scanning a quarter of the front labels of a pixel), two, or one.  A lone wavefront on a SIMD
// reaches some 70 % of what the SIMD issues with three of them, and the wavefronts of a chain meet
// at a barrier every pixel and repeat what is not the scan (loads, the update of the unary term,
// normalisation; the first one also finds the argmin labels), so the split pays as long as it fills
// idle SIMDs and stops paying once one wavefront per chain loads every SIMD.  Measured on 192
// labels, forward scan, ms per launch with 1 / 2 / 4 / 8 wavefronts per chain; keeping argmin
// labels: 384 chains 5.6 / 4.4 / 3.3 / 6.4, 768 chains 5.4 / 4.5 / 3.8 / 9.4, 1248 chains
// 22.7 / 18.5 / 21.3 / 50.8, 1536 chains 7.3 / 5.9 / 7.4 / 18.9, 1920 chains 8.6 / 9.6 / 10.0 / 25.1,
// 2496 chains 32.3 / 30.9 / 40.1 / 102, 3072 chains 10.2 / 12.4 / 14.3 / 37.8; without them: 384
// chains 4.5 / 2.9 / 1.9 / 3.2, 768 chains 4.1 / 2.9 / 3.2 / 4.8, 1248 chains 18.4 / 15.9 / 15.7 / 26.0,
// 1536 chains 5.9 / 6.0 / 5.6 / 9.6, 1920 chains 5.8 / 6.1 / 7.3 / 12.8, 2496 chains
// 29.9 / 27.5 / 29.2 / 51.8, 3072 chains 8.9 / 9.2 / 10.7 / 19.2.  In chains per SIMD: four
// wavefronts up to 1 (0.5 without argmin labels), two up to 1.5, one beyond.
template <typename Params>
int choose_split(const mpl_shape* s, const Params& p, const CallOpts& o, bool train) {
  if (!o.dense_table || s->ctx2d || s->n_disp <= kWave || p.pack >= 2) return 0;
  const int L = s->n_disp, R = labels_per_lane(L);
  int w;
  if (o.split_waves > 0) {
    w = o.split_waves;
  } else {
    const int64_t chains4 = 4 * (int64_t)p.block_prefix[p.n_dirs];  // in quarters of a chain
    const int64_t n_simd = launch_policy().n_simd;
    if (chains4 <= (train ? 4 : 2) * n_simd)
      w = 4;
    else if (chains4 <= 6 * n_simd)
      w = 2;
    else
      return 0;
  }
  // every wavefront needs a share of the front labels
  while (w > 1 && (w - 1) * split_share(L, R, w) >= L) --w;
  return w >= 2 ? w : 0;
}

// Four wavefronts per chain for a table declared dense, TRWP forward (mp_fwd_dense.hip), in place of those of
// choose_split and of mp_fwd_team.hip.  Measured on rows of 300 pixels with a random table, ns per pixel with one
// wavefront / as choose_split has it / mp_fwd_team.hip / this.  Argmin labels kept, 256 chains: 16 labels 613 / -
// / 357 / 367, 32 labels 824 / - / 536 / 371, 64 labels 1175 / - / 880 / 414, 96 labels 2324 / 1400 / 1540 / 674,
// 192 labels 4172 / 2242 / 3079 / 1223; 1248 chains: 16 labels 681 / - / 480 / 563, 32 labels 922 / - / 718 /
// 563, 96 labels 2858 / 2115 / 2635 / 1555, 192 labels 5568 / 4356 / 6342 / 3742.  Without them, 256 chains: 32
// labels 551 / - / 498 / 313, 96 labels 1602 / 770 / 1459 / 587, 192 labels 3078 / 1167 / 2962 / 915; 1248
// chains: 96 labels 2083 / 1486 / 1902 / 1300, 192 labels 4159 / 3701 / 4141 / 2813.  (The last column before it had
// servers; with them, kept / not, 256 chains: 17 and 32 labels 287 / 285, 64 labels 327 / 322, 96 labels 458 / 447, 192
// labels 838 / 789; 1248 chains: 96 labels 1454 / 1411, 192 labels, which have none there, 3705 / 2856.)
constexpr int kDenseTeamMinL = 17;
constexpr int kDenseTeamChainsPerCu = 5;
int decide_dense_team(const SweepParams& p, const CallOpts& o, bool train) {
  if (!o.dense_table || p.ctx2d || p.L < kDenseTeamMinL || p.L > kDenseTeamMaxL || p.pack >= 2 || o.team == 0 || o.split_waves > 0) return 0;
  if (o.team == 2) return 1;
  // (up to 64 labels the launch that takes any other kind of table is one of mp_fwd_team.hip)
  const int per_cu = p.L <= kWave ? team_fwd_chains_per_cu(p.L, train) : kDenseTeamChainsPerCu;
  return chains_at_once(p) <= per_cu * (launch_policy().n_simd / 4) ? 1 : 0;
}

// wavefronts of a one-direction launch: one per chain, or one per group of p.pack chains
template <typename Params>
int launch_waves(const Params& p) {
  const int chains = p.block_prefix[p.n_dirs];
  return p.pack >= 2 ? (chains + p.pack - 1) / p.pack : chains;
}

void launch_fwd(const SweepParams& p, bool train, bool jacobi, hipStream_t st) {
  Timed timed(jacobi ? MPL_KERNEL_FWD_SWEEP_ALL : MPL_KERNEL_FWD_SWEEP, st, p.fused_pair ? 2 : 1);
  if (p.pack >= 2) {
    launch_packed_fwd(p, train, jacobi, p.pack, st);  // (u_fused is never set together with pack)
    return;
  }
  if (p.dense_team) {
    switch (labels_per_lane(p.L)) {
      case 1: launch_dense_fwd<1>(p, train, st); break;
      case 2: launch_dense_fwd<2>(p, train, st); break;
      default: launch_dense_fwd<3>(p, train, st); break;
    }
    if (!p.skip_dense) return;
  }
  if (p.team && p.ctx2d && p.L == 21) {
    launch_team21_fwd(p, train, st);
    return;
  }
  if (p.team) {
    switch (labels_per_lane(p.L)) {
      case 1: launch_team_fwd<1>(p, train, st); break;
      case 2: launch_team_fwd<2>(p, train, st); break;
      case 3: launch_team_fwd<3>(p, train, st); break;
      default: launch_team_fwd<4>(p, train, st); break;
    }
    return;
  }
  switch (labels_per_lane(p.L)) {
    case 1: launch_sweep_fwd<1>(p, train, jacobi, st); break;
    case 2: launch_sweep_fwd<2>(p, train, jacobi, st); break;
    case 3: launch_sweep_fwd<3>(p, train, jacobi, st); break;
    default: launch_sweep_fwd<4>(p, train, jacobi, st); break;
  }
}

void launch_bwd(const BackParams& p, bool jacobi, hipStream_t st) {
  Timed timed(jacobi ? MPL_KERNEL_BWD_SWEEP_ALL : MPL_KERNEL_BWD_SWEEP, st, p.fused_pair ? 2 : 1);
  if (p.pack >= 2) {
    launch_packed_bwd(p, jacobi, p.pack, st);
    return;
  }
  if (p.team && p.ctx2d) {
    launch_team21_bwd(p, st);
    return;
  }
  if (p.team) {
    switch (labels_per_lane(p.L)) {
      case 2: launch_team_bwd<2>(p, jacobi, st); break;
      case 3: launch_team_bwd<3>(p, jacobi, st); break;
      default: launch_team_bwd<4>(p, jacobi, st); break;
    }
    return;
  }
  switch (labels_per_lane(p.L)) {
    case 1: launch_sweep_bwd<1>(p, jacobi, st); break;
    case 2: launch_sweep_bwd<2>(p, jacobi, st); break;
    case 3: launch_sweep_bwd<3>(p, jacobi, st); break;
    default: launch_sweep_bwd<4>(p, jacobi, st); break;
  }
}

SweepParams base_fwd_params(const mpl_shape* s, float rho, const float* edge, const float* ctx,
                            const CtxDesc* desc) {
  SweepParams p;
  memset(&p, 0, sizeof(p));
  p.xcd_group = xcd_group_size(s->n_disp);
  p.B = s->batch;
  p.H = s->height;
  p.W = s->width;
  p.L = s->n_disp;
  p.ctx2d = s->ctx2d ? 1 : 0;
  p.rho = rho;
  p.edge = edge;
  p.ctx = ctx;
  p.desc = desc;
  p.u_stride = (int64_t)s->batch * s->height * s->width * s->n_disp;
  return p;
}

// plain zero fill (a kernel, so that a caller may capture the call in a graph); V floats per store
template <int V>
__global__ void __launch_bounds__(256) zero_fill_kernel(float* __restrict__ dst, int64_t n) {
  Pack<V> z;
#pragma unroll
  for (int j = 0; j < V; ++j) z.v[j] = 0.f;
  for (int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * V; i < n;
       i += (int64_t)gridDim.x * blockDim.x * V)
    st_pack<V, true>(dst + i, z);
}

void zero_fill(float* dst, int64_t n, hipStream_t st) {
  if ((n & 3) == 0 && aligned16(dst))
    zero_fill_kernel<4><<<elementwise_blocks(n / 4), 256, 0, st>>>(dst, n);
  else
    zero_fill_kernel<1><<<elementwise_blocks(n), 256, 0, st>>>(dst, n);
}

// Zeros in the blocks of duals and the normalisation indices of chain-start pixels (MPL_F_CHAIN_STARTS), of all
// iterations and directions: grid.x the chains of p's directions, grid.y the iterations.  The rest of both tensors
// is the scans' to write, so nothing else needs clearing: 2x129x129, 21 labels, 4 directions, 5 iterations 156 us
// (a fill of 1.17 GB) -> 5 us.
__global__ void __launch_bounds__(256) chain_starts_kernel(const SweepParams p, int n_iter, float* __restrict__ duals,
                                                           uint8_t* __restrict__ norm) {
  const ChainCtx ch = locate_chain<false>(p);
  const int64_t P = (int64_t)p.B * p.H * p.W;
  const int block = p.L * p.L;
  for (int64_t it = blockIdx.y; it < n_iter; it += gridDim.y) {
    const int64_t pix = (it * p.n_dirs + ch.dir) * P + (int64_t)ch.bv * p.H * p.W + ch.pix0;
    for (int i = threadIdx.x; i < block; i += 256) duals[pix * block + i] = 0.f;
    if (threadIdx.x == 0) norm[pix] = 0;
  }
}

// The sweeps keep the belief plane up to date by differences, S <- (S - m_old) + m_new, where the
// reference re-sums unary + sum_k m_k before every sweep (UpdateUnaryKernel, TRWP_forward.cu:60-80):
// the rounding of each update stays in the plane.  Between two iterations the plane holds S itself,
// so it can be re-summed there exactly as the reference sums it, which bounds the drift of long
// runs (the 50 iterations of energy minimisation) at what a few iterations accumulate.
// Iterations between two re-summations for a call (0: none).  Left to the library (-1), calls of at
// most kShortCallSweeps direction sweeps are not re-summed (what they accumulate is below the
// rounding of the reference's own fp32 sums), longer ones whenever kSweepsPerRebuild sweeps have
// passed.
constexpr int kShortCallSweeps = 64;
constexpr int kSweepsPerRebuild = 32;
int belief_rebuild_interval(int n_dir, int n_iter) {
  const int opt = g_belief_rebuild.load(std::memory_order_relaxed);
  if (opt >= 0) return opt;
  if ((int64_t)n_dir * n_iter <= kShortCallSweeps) return 0;
  return kSweepsPerRebuild / n_dir > 1 ? kSweepsPerRebuild / n_dir : 1;
}

void rebuild_belief(const mpl_shape* s, const float* unary, const float* msg, float* S,
                    hipStream_t st) {
  Timed timed(MPL_KERNEL_BELIEF, st);
  const int64_t N = (int64_t)s->batch * s->height * s->width * s->n_disp;
  const bool v4 = (N % 4 == 0) && aligned16(unary) && aligned16(msg) && aligned16(S);
  MPL_EW_LAUNCH(belief_kernel, v4, ew_hint(s), s->n_dir, N, st, unary, msg, s->n_dir, N, S, (int*)nullptr);
}

// dcontext = the sum of the tables the reverse scans added to (MPL_F_DCONTEXT_COPIES), always in the same order
__global__ void __launch_bounds__(kWave) dcontext_fold_kernel(const float* __restrict__ tables, int entries,
                                                              float* __restrict__ dcontext) {
  const int i = (int)blockIdx.x * kWave + (int)threadIdx.x;
  if (i >= entries) return;
  float x[kDctxCopies];
#pragma unroll
  for (int k = 0; k < kDctxCopies; ++k) x[k] = tables[k * entries + i];
#pragma unroll
  for (int w = kDctxCopies / 2; w > 0; w /= 2)
#pragma unroll
    for (int k = 0; k < w; ++k) x[k] += x[k + w];
  dcontext[i] = x[0];
}

// Where the reverse scans of a backward call add their parts of dcontext: the caller's tensor, or tables in its
// scratch tensor that fold_dcontext sums at the end of the call.  False: no scratch to take.
bool place_dcontext(const mpl_shape* s, unsigned flags, int n_iter, float* dcontext, float* scratch, BackParams* p) {
  p->dctx = dcontext;
  p->dctx_mask = 0;
  if ((flags & MPL_F_DCONTEXT_COPIES) == 0 || dcontext == nullptr || mpl_dcontext_copies(s, n_iter) == 0) return true;
  if (scratch == nullptr) return false;
  p->dctx = scratch;
  p->dctx_mask = kDctxCopies - 1;
  return true;
}
void fold_dcontext(const BackParams& p, float* dcontext, hipStream_t st) {
  if (p.dctx_mask == 0) return;
  Timed timed(MPL_KERNEL_OTHER, st);
  const int entries = p.ctx2d ? p.L * p.L : p.L;
  dcontext_fold_kernel<<<(entries + kWave - 1) / kWave, kWave, 0, st>>>(p.dctx, entries, dcontext);
}

// 16 directions, labels first: the loads of all planes go out together, but of four floats each only up to this much of
// messages.  Measured, us, one plane after another / together: 96 labels 150x200 30.8 / 30.5, 240x320 92 / 77, 300x400
// 123 / 122, 64 labels 480x640 (1.2 GiB) 241 / 237, 96 labels 384x800 (1.8 GiB) 348 / 385, 384x1248 516 / 596, 190 labels
// 375x450 (1.9 GiB) 420 / 432.  Single floats: 21 labels 65x65 14.9 / 4.0, 97 labels 241x321 213 / 99, 383x1247
// 1167 / 752.
constexpr int64_t kFirst16Bytes = (int64_t)5 << 28;

// cost_final from the unary terms and the messages, in either layout.
void aggregate(const mpl_shape* s, unsigned flags, const float* unary, const float* msg, float factor, int min_a_dir,
               float* cost_final, hipStream_t st) {
  Timed timed(MPL_KERNEL_AGGREGATE, st);
  const int L = s->n_disp, n_dir = s->n_dir;
  const int64_t HW = (int64_t)s->height * s->width, N = s->batch * HW * L;
  const bool nt = ew_hint(s);
  if ((flags & MPL_F_COST_LABELS_FIRST) == 0) {
    const bool v4 = (N % 4 == 0) && aligned16(unary) && aligned16(msg) && aligned16(cost_final);
    MPL_EW_LAUNCH(aggregate_kernel, v4, nt, n_dir, N, st, unary, msg, n_dir, N, factor, min_a_dir, cost_final);
    return;
  }
  // Some 32 KB of LDS at most, a run of a few KB per plane; one line of the result, where that is not enough to go
  // round, and less of it for the few tiles of a small image with many labels, whose workgroups pass over theirs again
  // and again.  Tiles of 32 pixels -> this, us: 255 labels 23x29, 8 directions 26 -> 10, batch 4 16 -> 10; 191 labels 4x46x65,
  // 12 directions 51 -> 30; 256 labels 60x80, 4 directions 14 -> 10; 97 labels 4x63x77, 6 directions 22 -> 16; 192 labels
  // 100x150 15.9 -> 16.2.
  const auto tiles = [&](int log) { return (((HW - 1) >> log) + 1) * s->batch; };
  const int n_simd = launch_policy().n_simd;
  int tile_log = L <= 32 ? 7 : L <= 128 ? 6 : 5;
  while (tile_log > 5 && tiles(tile_log) < 2 * n_simd) --tile_log;
  while (L > 32 && tile_log > 3 && tiles(tile_log) < n_simd) --tile_log;
  // (fours that lie across two tiles are loaded for both: 191 labels 4x46x65, 12 directions 60 -> 51 us, 21 labels
  // 4x129x129 9.5 -> 8.8)
  const bool v4 = N % 4 == 0 && aligned16(unary) && aligned16(msg);
  const bool lines = (HW * (int64_t)sizeof(float)) % kLineBytes == 0 && ((uintptr_t)cost_final & (kLineBytes - 1)) == 0;
  const dim3 grid((unsigned)(((HW - 1) >> tile_log) + 1), (unsigned)std::min(s->batch, 65535));
  const size_t lds = sizeof(float) * ((size_t)(L | 1) << tile_log);
  const auto launch = [&](auto kernel) {
    kernel<<<grid, 256, lds, st>>>(unary, msg, n_dir, N, (int)HW, L, tile_log, factor, min_a_dir, cost_final);
  };
#define MPL_FIRST(V, ND)                                                                                             \
  launch(nt ? (lines ? aggregate_first_kernel<V, ND, true, true> : aggregate_first_kernel<V, ND, true, false>)       \
            : (lines ? aggregate_first_kernel<V, ND, false, true> : aggregate_first_kernel<V, ND, false, false>))
  if (v4 && n_dir == 4)
    MPL_FIRST(4, 4);
  else if (v4 && n_dir == 8)
    MPL_FIRST(4, 8);
  else if (v4 && n_dir == 16 && message_bytes(s) <= kFirst16Bytes)
    MPL_FIRST(4, 16);
  else if (v4)
    MPL_FIRST(4, 0);
  else if (n_dir == 4)
    MPL_FIRST(1, 4);
  else if (n_dir == 8)
    MPL_FIRST(1, 8);
  else if (n_dir == 16)
    MPL_FIRST(1, 16);
  else
    MPL_FIRST(1, 0);
#undef MPL_FIRST
}

// cost_final is not written before the final aggregation, so its first bytes carry the context
// descriptor during the sweeps (no allocation, no state shared between streams).
const CtxDesc* make_desc(const mpl_shape* s, const float* ctx, float* cost_final, hipStream_t st) {
  int64_t N = (int64_t)s->batch * s->height * s->width * s->n_disp;
  if (N * (int64_t)sizeof(float) < (int64_t)sizeof(CtxDesc)) return nullptr;  // dense path
  CtxDesc* d = reinterpret_cast<CtxDesc*>(cost_final);
  Timed timed(MPL_KERNEL_OTHER, st);
  analyze_context_kernel<<<1, kWave, 0, st>>>(ctx, s->n_disp, s->ctx2d ? 1 : 0, d);
  return d;
}

}  // namespace

namespace mpl {
// SIMDs of the current device: four per compute unit.  Without a device (argument validation on a
// host that has none) the MI355X's 256 compute units are assumed.
const LaunchPolicy& launch_policy() {
  constexpr int kMaxDevices = 64;
  static LaunchPolicy table[kMaxDevices];
  static std::atomic<int> ready[kMaxDevices];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) dev = 0;
  if (ready[dev].load(std::memory_order_acquire) == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) {
      (void)hipGetLastError();
      cus = 256;
    }
    LaunchPolicy pol;
    pol.n_simd = 4 * cus;
    pol.fused_pair_max_waves = pol.n_simd;
    pol.packed_min_chains = pol.n_simd + 1;
    pol.packed_min_chains21 = 2 * pol.n_simd + 1;
    pol.packed_min_chains_1d8 = 6 * pol.n_simd + 1;
    pol.packed_min_chains_1d16 = 9 * pol.n_simd + 1;
    pol.direct_max_chains = 2 * pol.n_simd;
    static std::mutex mu;
    std::lock_guard<std::mutex> lk(mu);
    if (ready[dev].load(std::memory_order_relaxed) == 0) {
      table[dev] = pol;
      ready[dev].store(1, std::memory_order_release);
    }
  }
  return table[dev];
}

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}
}  // namespace mpl

// ------------------------------------------------------------------------------------------------
// C ABI
// ------------------------------------------------------------------------------------------------
extern "C" {

const char* mpl_last_error(void) { return g_err; }

int mpl_version(void) { return 210; }  // (2.10: the probes left the library; MPL_OPT_BELIEF_REBUILD; CPU forward)

int mpl_set_option(int option, int value) {
  if (option == MPL_OPT_PACKED_SCANS) {
    if (value < 0 || value > 2) return fail(MPL_EINVAL, "set_option: packed scans take 0, 1 or 2");
    g_packed_scans.store(value, std::memory_order_relaxed);
    return MPL_OK;
  }
  if (option == MPL_OPT_FUSED_U) {
    if (value < 0 || value > 1) return fail(MPL_EINVAL, "set_option: fused U takes 0 or 1");
    g_fused_u.store(value, std::memory_order_relaxed);
    return MPL_OK;
  }
  if (option == MPL_OPT_BELIEF_REBUILD) {
    if (value < -1) return fail(MPL_EINVAL, "set_option: the belief rebuild interval is >= -1");
    g_belief_rebuild.store(value, std::memory_order_relaxed);
    return MPL_OK;
  }
  if (option == MPL_OPT_CPU_THREADS) return set_cpu_threads(value);
  if (option == MPL_OPT_DENSE_SPLIT_WAVES) {
    if (value < 0 || value > 8) return fail(MPL_EINVAL, "set_option: 0 to 8 wavefronts per chain");
    g_split_waves.store(value, std::memory_order_relaxed);
    return MPL_OK;
  }
  if (option == MPL_OPT_TEAM_SCANS) {
    if (value < 0 || value > 2) return fail(MPL_EINVAL, "set_option: team scans take 0, 1 or 2");
    g_team_scans.store(value, std::memory_order_relaxed);
    return MPL_OK;
  }
  return fail(MPL_EINVAL, "set_option: unknown option %d", option);
}

int mpl_profile_begin(void) {
  std::lock_guard<std::mutex> lk(g_prof_mu);
  for (auto& r : g_prof.recs) {
    g_prof.pool.push_back(r.start);
    g_prof.pool.push_back(r.stop);
  }
  g_prof.recs.clear();
  g_prof.on.store(true, std::memory_order_release);
  return MPL_OK;
}

int mpl_profile_end(mpl_kernel_stat* stats, int n_stats) {
  std::lock_guard<std::mutex> lk(g_prof_mu);
  g_prof.on.store(false, std::memory_order_release);
  for (int i = 0; i < n_stats; ++i) {
    stats[i].launches = 0;
    stats[i].total_ms = 0.0;
  }
  int rc = MPL_OK;
  for (auto& r : g_prof.recs) {
    float ms = 0.f;
    hipError_t e = hipEventSynchronize(r.stop);
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, r.start, r.stop);
    if (e != hipSuccess) {
      rc = fail(MPL_ELAUNCH, "profile_end: %s", hipGetErrorString(e));
    } else if (r.kind >= 0 && r.kind < n_stats) {
      stats[r.kind].launches += r.sweeps;
      stats[r.kind].total_ms += ms;
    }
    g_prof.pool.push_back(r.start);
    g_prof.pool.push_back(r.stop);
  }
  g_prof.recs.clear();
  return rc;
}

// The rule of analyze_context_kernel on a table in host memory: neither a band nor truncated linear.
int mpl_table_is_dense(const float* context, int n_disp) {
  if (!context || n_disp < 1) return -1;
  const int L = n_disp;
  const float tail = context[L - 1], c0 = context[0], slope = L >= 2 ? context[1] : 0.f;
  unsigned tail_bits;
  memcpy(&tail_bits, &tail, sizeof tail_bits);
  if ((tail_bits & 0x7fffffffu) > 0x7f800000u) return 1;  // a NaN tail: no fast path
  int last_ne = -1;
  bool below = true, lin = true;
  for (int i = 0; i < L; ++i) {
    const float v = context[i];
    if (!(v == tail)) last_ne = i;
    below = below && (v <= tail);
    lin = lin && (v == fminf(slope * (float)i, tail));
  }
  if (!below) return 1;
  const bool band = last_ne + 1 <= kMaxBandK;
  const bool linear = L >= 2 && c0 == 0.f && slope >= 0.f && lin;
  return (band || linear) ? 0 : 1;
}

int mpl_dcontext_copies(const mpl_shape* s, int n_iter) {
  if (check_shape(s, n_iter) != MPL_OK) return -1;
  int64_t chains = 0;
  for (int d = 0; d < s->n_dir; ++d) chains += (int64_t)s->batch * make_dir(d, s->height, s->width).n_chains;
  return chains * n_iter >= kDctxMinChains ? kDctxCopies : 0;
}

int mpl_n_chains(int dir, int height, int width) {
  if (dir < 0 || dir >= kMaxDirs || height < 1 || width < 1) return -1;
  return make_dir(dir, height, width).n_chains;
}

int mpl_trwp_forward(const mpl_shape* s, unsigned flags, float rho, int n_iter,
                     int enable_min_a_dir, const float* unary, const float* context,
                     const float* edge_weights, float* msg, float* cost_final,
                     uint8_t* msg_min_index, uint8_t* msg_norm_index, float* unary_update,
                     uint8_t* label_all, void* stream) {
  int rc = check_shape(s, n_iter);
  if (rc) return rc;
  CallOpts opts;
  if ((rc = read_flags(flags, "trwp_forward", &opts)) != MPL_OK) return rc;
  const bool msg_uninit = (flags & MPL_F_MSG_UNINIT) != 0;
  if (!unary || !context || !edge_weights || !msg || !cost_final || !unary_update)
    return fail(MPL_EINVAL, "trwp_forward: null tensor pointer");
  if ((msg_min_index == nullptr) != (msg_norm_index == nullptr))
    return fail(MPL_EINVAL, "trwp_forward: msg_min_index and msg_norm_index go together");
  hipStream_t st = (hipStream_t)stream;
  const int64_t P = (int64_t)s->batch * s->height * s->width;
  const int64_t N = P * s->n_disp;
  const bool train = msg_min_index != nullptr;

  const CtxDesc* desc = make_desc(s, context, cost_final, st);
  // Messages that start at zero by declaration: S = unary, so the belief plane need not be built
  // (the first pair of sweeps reads `unary` in its place: Q = S - m_0 - m_1 = unary, too, and the
  // even sweep has nothing to store), no plane of initial messages is read (the descriptor's
  // flag stays 0), and the first sweep of every direction writes the zero of its chain starts.
  const bool uninit = msg_uninit && desc != nullptr;
  if (msg_uninit && !uninit) zero_fill(msg, (int64_t)s->n_dir * N, st);
  // The reference's contract: `msg` holds the initial messages, which its callers always clear.
  // With more labels than the packed scans take, the messages are first only looked at (n_dir
  // planes in, nothing out): when they are all zero the belief plane is not built (the kernel
  // that builds it finds the flag clear and ends) and the first pair of sweeps does what it does
  // for messages declared zero, choosing on the device (SweepParams::zero_first).
  const bool probe_zero = !uninit && desc != nullptr && s->n_disp > kPackedMaxL;
  if (!uninit) {
    Timed timed(MPL_KERNEL_BELIEF, st);
    const bool v4 = (N % 4 == 0) && aligned16(unary) && aligned16(msg) && aligned16(unary_update);
    int* flag = desc != nullptr ? &const_cast<CtxDesc*>(desc)->msg_nonzero : nullptr;
    if (probe_zero) {
      MPL_EW_LAUNCH(check_nonzero_kernel, v4, ew_hint(s), s->n_dir, N, st, msg, s->n_dir, N, flag);
      MPL_EW_LAUNCH(belief_kernel, v4, ew_hint(s), s->n_dir, N, st, unary, msg, s->n_dir, N, unary_update,
                    (int*)nullptr, (const int*)flag);
    } else {
      MPL_EW_LAUNCH(belief_kernel, v4, ew_hint(s), s->n_dir, N, st, unary, msg, s->n_dir, N, unary_update, flag);
    }
  }

  SweepParams p = base_fwd_params(s, rho, edge_weights, context, desc);
  p.belief_zero = unary;
  p.belief_out = unary_update;
  p.msg_in = msg;
  p.msg_out = msg;
  const int rebuild = belief_rebuild_interval(s->n_dir, n_iter);
  bool have_belief = false, have_cost = false;  // the pass that writes the labels has stored it
  float* const cost_plane = (flags & MPL_F_COST_LABELS_FIRST) ? nullptr : cost_final;  // (where it can)
  for (int it = 0; it < n_iter; ++it) {
    if (rebuild > 0 && it > 0 && it % rebuild == 0 && !have_belief)
      rebuild_belief(s, unary, msg, unary_update, st);
    have_belief = false;
    for (int d = 0; d < s->n_dir; ++d) {  // Gauss-Seidel over directions: TRWP_forward.cu:440-518
      fill_dirs(s, d, 1, p.dirs, p.block_prefix, &p.n_dirs);
      p.pack = decide_pack(s, p, opts);
      p.split = choose_split(s, p, opts, train);
      p.dense_team = decide_dense_team(p, opts, train);
      p.team = decide_team_fwd(p, opts, train);
      p.skip_dense = (p.dense_team && s->n_disp <= kWave) ? 1 : 0;
      p.through = message_bytes(s) <= kCachedMessages ? 1 : 0;
      p.first_iter = (it == 0);
      p.pair_q = 1;
      p.belief = (uninit && it == 0 && d <= 1) ? unary : unary_update;
      p.zero_start = (uninit && it == 0) ? 1 : 0;
      p.zero_first = (probe_zero && it == 0 && d <= 1) ? 1 : 0;
      auto skip_s = [&](int dd) {
        return (((it == n_iter - 1) && (dd == s->n_dir - 1)) ||  // cost_final is re-summed
                (uninit && it == 0 && dd == 0)) ? 1 : 0;
      };
      p.skip_s_store = skip_s(d);
      // few chains: the wavefront of a chain sweeps d and then d + 1 (the same pixels in reverse)
      p.fused_pair = (opts.fused_pairs && !(d & 1) &&
                      launch_waves(p) <= launch_policy().fused_pair_max_waves) ? 1 : 0;
      p.skip_s_store2 = skip_s(d + 1);
      if (train) {
        p.idx_min = msg_min_index + (int64_t)it * s->n_dir * N;
        p.idx_norm = msg_norm_index + (int64_t)it * s->n_dir * P;
      }
      launch_fwd(p, train, false, st);
      if (p.fused_pair) ++d;
    }
    if (label_all) {
      Timed timed(MPL_KERNEL_LABEL, st);
      // the next pass over the same planes, if one is due: cost_final, the re-summed belief plane
      const bool last = it + 1 == n_iter;
      float* out = last ? cost_plane : (rebuild > 0 && (it + 1) % rebuild == 0) ? unary_update : nullptr;
      const bool stored = launch_labels(unary, msg, s->n_dir, P, s->n_disp, 1.f, enable_min_a_dir,
                                        label_all + it * P, st, ew_hint(s), kLabelSum, out);
      (last ? have_cost : have_belief) = stored;
    }
  }
  if (!have_cost) aggregate(s, flags, unary, msg, 1.f, enable_min_a_dir, cost_final, st);
  return launch_ok("trwp_forward");
}

int mpl_isgmr_forward(const mpl_shape* s, unsigned flags, int enable_sgm, float rho, int n_iter,
                      int enable_min_a_dir, const float* unary, const float* context,
                      const float* edge_weights, float* msg, float* cost_final,
                      uint8_t* msg_min_index, uint8_t* msg_norm_index, float* unary_update,
                      float* msg_update, uint8_t* label_all, void* stream) {
  int rc = check_shape(s, n_iter);
  if (rc) return rc;
  CallOpts opts;
  if ((rc = read_flags(flags, "isgmr_forward", &opts)) != MPL_OK) return rc;
  const bool msg_uninit = (flags & MPL_F_MSG_UNINIT) != 0;
  if (!unary || !context || !edge_weights || !msg || !cost_final || !unary_update || !msg_update)
    return fail(MPL_EINVAL, "isgmr_forward: null tensor pointer");
  if ((msg_min_index == nullptr) != (msg_norm_index == nullptr))
    return fail(MPL_EINVAL, "isgmr_forward: msg_min_index and msg_norm_index go together");
  hipStream_t st = (hipStream_t)stream;
  const int64_t P = (int64_t)s->batch * s->height * s->width;
  const int64_t N = P * s->n_disp;
  const bool train = msg_min_index != nullptr;
  const float factor = enable_sgm ? (float)s->n_dir : 1.f;

  const CtxDesc* desc = make_desc(s, context, cost_final, st);
  SweepParams p = base_fwd_params(s, rho, edge_weights, context, desc);
  p.belief = unary_update;
  p.belief_out = nullptr;
  fill_dirs(s, 0, s->n_dir, p.dirs, p.block_prefix, &p.n_dirs);
  p.u_pair_share = (rho == 1.f) ? 1 : 0;
  // Messages that start at zero by declaration: U_d = rho * unary in the first iteration, so at
  // rho = 1 its sweeps read `unary` itself and the pass that would store U is skipped (the
  // sweeps write every element of their output buffer, chain starts included).
  const bool unary_as_u = msg_uninit && rho == 1.f;
  // Four directions at rho = 1: U of a pair of opposite directions is the unary plus the two
  // messages of the other pair, so the scans can form it on the fly (3 planes read per direction
  // instead of 1) and the pass that stores U (5 planes in, 2 out per iteration) is dropped; with
  // more directions the scans would read more than that pass moves.  (Not where the packed scans
  // of small label counts run: they are bound by the instructions of a step, and two more loads
  // per step cost them more than the pass.)
  p.pack = decide_pack(s, p, opts);
  p.split = choose_split(s, p, opts, train);
  const bool fuse_u = opts.fused_u && s->n_dir == 4 && rho == 1.f && p.pack == 0;
  if (msg_uninit && !unary_as_u) zero_fill(msg, (int64_t)s->n_dir * N, st);
  // The reference's contract at rho = 1, one chain per wavefront: the initial messages are looked
  // at first (n_dir planes in, nothing out); when they are all zero, as the reference's callers
  // pass them, the first iteration's U pass finds the flag clear and ends, and its scans read the
  // unary terms, chosen on the device (SweepParams::zero_first).
  const bool probe_zero = !msg_uninit && rho == 1.f && desc != nullptr && s->n_disp > kPackedMaxL &&
                          p.pack == 0;
  p.belief_zero = unary;
  float* have = msg;  // the buffer that holds the current messages
  bool have_u = false, have_cost = false;  // the pass that writes the labels has stored it
  float* const cost_plane = (flags & MPL_F_COST_LABELS_FIRST) ? nullptr : cost_final;  // (where it can)
  for (int it = 0; it < n_iter; ++it) {
    // Jacobi over directions (ISGMR_forward.cu:506-622): every direction reads the old messages,
    // through U; the two buffers alternate instead of being copied.  U normally overwrites the
    // old messages and the new ones go to the other buffer; with an odd number of iterations the
    // first one stores U in the other buffer and the new messages in `msg`, so that the final
    // messages always end up in `msg` as in the reference.
    float* other = (have == msg) ? msg_update : msg;
    const bool out_of_place = (it == 0) && (n_iter & 1);
    float* ubuf = out_of_place ? other : have;
    float* nxt = out_of_place ? have : other;
    p.u_fused = 0;
    if (it == 0 && unary_as_u) {
      p.msg_in = unary;
      p.u_stride = 0;
    } else if (fuse_u && !out_of_place) {
      // the scans read the unary and the old messages of the other pair of directions themselves
      p.belief = unary;
      p.msg_in = have;
      p.u_stride = N;
      p.u_fused = 1;
    } else if (have_u) {  // over the old messages, as the pass below leaves them
      p.msg_in = ubuf;
      p.u_stride = N;
    } else {
      Timed timed(MPL_KERNEL_UNARY_ALL, st);
      const bool v4 = (N % 4 == 0) && aligned16(unary) && aligned16(msg) && aligned16(msg_update);
      const int* only_if = nullptr;
      if (probe_zero && it == 0) {
        int* flag = &const_cast<CtxDesc*>(desc)->msg_nonzero;
        MPL_EW_LAUNCH(check_nonzero_kernel, v4, ew_hint(s), s->n_dir, N, st, have, s->n_dir, N, flag);
        only_if = flag;
        p.zero_first = 1;
      }
      MPL_EW_LAUNCH(isgmr_unary_kernel, v4, ew_hint(s), s->n_dir, N, st, unary, have, ubuf, s->n_dir, N, rho,
                    p.u_pair_share, only_if);
      p.msg_in = ubuf;
      p.u_stride = N;
    }
    p.msg_out = nxt;
    if (train) {
      p.idx_min = msg_min_index + (int64_t)it * s->n_dir * N;
      p.idx_norm = msg_norm_index + (int64_t)it * s->n_dir * P;
    }
    launch_fwd(p, train, true, st);
    p.zero_first = 0;
    if (label_all) {
      Timed timed(MPL_KERNEL_LABEL, st);
      // the next pass over the same planes: cost_final, or the U planes of the next iteration in
      // place of these messages, unless its scans form U themselves
      const bool last = it + 1 == n_iter;
      const bool stored = launch_labels(unary, nxt, s->n_dir, P, s->n_disp, factor, enable_min_a_dir,
                                        label_all + it * P, st, ew_hint(s), last ? kLabelSum : kLabelU,
                                        last ? cost_plane : fuse_u ? nullptr : nxt, rho, p.u_pair_share);
      (last ? have_cost : have_u) = stored;
    }
    have = nxt;
  }
  if (!have_cost) aggregate(s, flags, unary, msg, factor, enable_min_a_dir, cost_final, st);
  return launch_ok("isgmr_forward");
}

int mpl_trwp_backward(const mpl_shape* s, unsigned flags, float rho, int n_iter,
                      const float* context, const float* edge_weights, const float* dcost_final,
                      const uint8_t* msg_min_index, const uint8_t* msg_norm_index, float* dunary,
                      float* dcontext, float* dedge_weights, float* dmsg, float* dunary_update,
                      void* stream) {
  int rc = check_shape(s, n_iter);
  if (rc) return rc;
  CallOpts opts;
  if ((rc = read_flags(flags, "trwp_backward", &opts)) != MPL_OK) return rc;
  // dcontext / dedge_weights may be null: gradients the caller has no use for
  if (!context || !edge_weights || !dcost_final || !msg_min_index || !msg_norm_index || !dunary ||
      !dmsg)
    return fail(MPL_EINVAL, "trwp_backward: null tensor pointer");
  hipStream_t st = (hipStream_t)stream;
  const int64_t P = (int64_t)s->batch * s->height * s->width;
  const int64_t N = P * s->n_disp;

  BackParams p;
  memset(&p, 0, sizeof(p));
  p.B = s->batch;
  p.H = s->height;
  p.W = s->width;
  p.L = s->n_disp;
  p.ctx2d = s->ctx2d ? 1 : 0;
  p.rho = rho;
  p.h = dmsg;
  p.edge = edge_weights;
  p.ctx = context;
  p.dedge = dedge_weights;
  if (!place_dcontext(s, flags, n_iter, dcontext, dunary_update, &p))
    return fail(MPL_EINVAL, "MPL_F_DCONTEXT_COPIES needs the tables in dunary_update");
  p.same_label = (flags & MPL_F_DCONTEXT_SAME_LABEL) ? 1 : 0;
  const float* a_cur = dcost_final;  // CostAggregateKernelBack: every g_k starts as dcost
  for (int it = n_iter - 1; it >= 0; --it) {
    for (int d = s->n_dir - 1; d >= 0; --d) {  // TRWP_backward.cu:337-424
      fill_dirs(s, d, 1, p.dirs, p.block_prefix, &p.n_dirs);
      p.pack = decide_pack(s, p, opts);
      p.team = decide_team(p, opts, false);
      p.a_in = a_cur;
      float* const plane_e = dmsg + (int64_t)(d & ~1) * N;
      p.a_out = (it == 0 && d <= 1) ? dunary : plane_e;
      p.first_touch = (it == n_iter - 1) ? 1 : 0;
      // in the last iteration walked the even sweeps leave h planes nobody reads again
      p.skip_h_store = (it == 0) ? 1 : 0;
      p.idx_min = msg_min_index + (int64_t)it * s->n_dir * N;
      p.idx_norm = msg_norm_index + (int64_t)it * s->n_dir * P;
      // few chains: the wavefront of a chain walks d (odd) and then d - 1 (same pixels, reversed)
      p.fused_pair = (opts.fused_pairs && (d & 1) &&
                      launch_waves(p) <= launch_policy().fused_pair_max_waves) ? 1 : 0;
      launch_bwd(p, false, st);
      if (p.fused_pair) --d;
      if (!(d & 1)) a_cur = p.a_out;
    }
  }
  fold_dcontext(p, dcontext, st);
  return launch_ok("trwp_backward");
}

int mpl_isgmr_backward(const mpl_shape* s, unsigned flags, int enable_sgm, float rho, int n_iter,
                       const float* context, const float* edge_weights, const float* dcost_final,
                       const uint8_t* msg_min_index, const uint8_t* msg_norm_index, float* dunary,
                       float* dcontext, float* dedge_weights, float* dmsg, float* dunary_update,
                       float* dmsg_update, void* stream) {
  int rc = check_shape(s, n_iter);
  if (rc) return rc;
  CallOpts opts;
  if ((rc = read_flags(flags, "isgmr_backward", &opts)) != MPL_OK) return rc;
  // dcontext / dedge_weights may be null: gradients the caller has no use for
  if (!context || !edge_weights || !dcost_final || !msg_min_index || !msg_norm_index || !dunary ||
      !dmsg_update)
    return fail(MPL_EINVAL, "isgmr_backward: null tensor pointer");
  // The reverse scans write X_k = dU_k into dmsg_update; the recombined gradients gu_k of the next
  // (earlier) iteration go to dmsg when the caller passes it, so that at rho == 1 one plane per
  // pair of opposite directions suffices; without dmsg they overwrite X_k in place.
  {
    const int64_t planes = (int64_t)s->n_dir * s->batch * s->height * s->width * s->n_disp;
    if (dmsg != nullptr && dmsg < dmsg_update + planes && dmsg_update < dmsg + planes)
      dmsg = nullptr;  // overlaps dmsg_update: not usable as a second buffer
  }
  float* gu_buf = dmsg != nullptr ? dmsg : dmsg_update;
  const int pair_share = (dmsg != nullptr && rho == 1.f) ? 1 : 0;
  hipStream_t st = (hipStream_t)stream;
  const int64_t P = (int64_t)s->batch * s->height * s->width;
  const int64_t N = P * s->n_disp;
  const float factor = enable_sgm ? (float)s->n_dir : 1.f;

  BackParams p;
  memset(&p, 0, sizeof(p));
  p.B = s->batch;
  p.H = s->height;
  p.W = s->width;
  p.L = s->n_disp;
  p.ctx2d = s->ctx2d ? 1 : 0;
  p.rho = rho;
  p.du_out = dmsg_update;
  p.edge = edge_weights;
  p.ctx = context;
  p.dedge = dedge_weights;
  if (!place_dcontext(s, flags, n_iter, dcontext, dunary_update, &p))
    return fail(MPL_EINVAL, "MPL_F_DCONTEXT_COPIES needs the tables in dunary_update");
  p.same_label = (flags & MPL_F_DCONTEXT_SAME_LABEL) ? 1 : 0;
  fill_dirs(s, 0, s->n_dir, p.dirs, p.block_prefix, &p.n_dirs);
  p.pack = decide_pack(s, p, opts);
  p.team = decide_team(p, opts, true);
  for (int it = n_iter - 1; it >= 0; --it) {
    const bool first = (it == n_iter - 1);
    p.gu_in = first ? dcost_final : gu_buf;  // gu_k = dcost_final for every k at the start
    p.gu_stride = first ? 0 : N;
    p.gu_pair_share = first ? 0 : pair_share;
    p.idx_min = msg_min_index + (int64_t)it * s->n_dir * N;
    p.idx_norm = msg_norm_index + (int64_t)it * s->n_dir * P;
    launch_bwd(p, true, st);
    Timed timed(MPL_KERNEL_COMBINE, st);
    const bool v4 = (N % 4 == 0) && aligned16(dmsg_update) && aligned16(gu_buf) &&
                    aligned16(dcost_final) && aligned16(dunary);
    MPL_EW_LAUNCH(isgmr_combine_kernel, v4, ew_hint(s), s->n_dir, N, st, dmsg_update, gu_buf, s->n_dir, N, rho,
                  dcost_final, factor, first ? 1 : 0, it > 0 ? 1 : 0, pair_share, dunary);
  }
  fold_dcontext(p, dcontext, st);
  return launch_ok("isgmr_backward");
}

// ---- soft-weighted TRWP ------------------------------------------------------------------------
int mpl_trwp_soft_forward(const mpl_shape* s, unsigned flags, float rho, int n_iter,
                          const float* unary, const float* context, const float* edge_weights,
                          float* msg, float* msg_edge_label, uint8_t* msg_norm_index,
                          float* cost_final, float* unary_update, uint8_t* label_all,
                          void* stream) {
  int rc = check_shape(s, n_iter);
  if (rc) return rc;
  CallOpts opts;
  if ((rc = read_flags(flags, "trwp_soft_forward", &opts)) != MPL_OK) return rc;
  if (!unary || !context || !edge_weights || !msg || !cost_final || !unary_update)
    return fail(MPL_EINVAL, "trwp_soft_forward: null tensor pointer");
  if ((msg_edge_label == nullptr) != (msg_norm_index == nullptr))
    return fail(MPL_EINVAL, "trwp_soft_forward: msg_edge_label and msg_norm_index go together");
  hipStream_t st = (hipStream_t)stream;
  const int64_t P = (int64_t)s->batch * s->height * s->width;
  const int64_t N = P * s->n_disp;
  const bool train = msg_edge_label != nullptr;
  if (train && (flags & MPL_F_CHAIN_STARTS)) {
    Timed timed(MPL_KERNEL_OTHER, st);
    SweepParams p = base_fwd_params(s, rho, edge_weights, context, nullptr);
    fill_dirs(s, 0, s->n_dir, p.dirs, p.block_prefix, &p.n_dirs);
    const dim3 grid((unsigned)p.block_prefix[p.n_dirs], (unsigned)std::min(n_iter, 65535));
    chain_starts_kernel<<<grid, 256, 0, st>>>(p, n_iter, msg_edge_label, msg_norm_index);
  }
  if (flags & MPL_F_MSG_UNINIT) zero_fill(msg, (int64_t)s->n_dir * N, st);
  {
    Timed timed(MPL_KERNEL_BELIEF, st);
    const bool v4 = (N % 4 == 0) && aligned16(unary) && aligned16(msg) && aligned16(unary_update);
    MPL_EW_LAUNCH(belief_kernel, v4, ew_hint(s), s->n_dir, N, st, unary, msg, s->n_dir, N, unary_update,
                  (int*)nullptr);
  }
  SweepParams p = base_fwd_params(s, rho, edge_weights, context, nullptr);
  p.belief = unary_update;
  p.belief_out = unary_update;
  p.msg_in = msg;
  p.msg_out = msg;
  const int rebuild = belief_rebuild_interval(s->n_dir, n_iter);
  bool have_belief = false, have_cost = false;  // the pass that writes the labels has stored it
  float* const cost_plane = (flags & MPL_F_COST_LABELS_FIRST) ? nullptr : cost_final;  // (where it can)
  for (int it = 0; it < n_iter; ++it) {
    if (rebuild > 0 && it > 0 && it % rebuild == 0 && !have_belief)
      rebuild_belief(s, unary, msg, unary_update, st);
    have_belief = false;
    for (int d = 0; d < s->n_dir; ++d) {  // TRWP_forward_soft.cu:441-520
      fill_dirs(s, d, 1, p.dirs, p.block_prefix, &p.n_dirs);
      if (train) {
        p.edge_label = msg_edge_label + (int64_t)it * s->n_dir * N * s->n_disp;
        p.idx_norm = msg_norm_index + (int64_t)it * s->n_dir * P;
      }
      // few chains of at most 32 labels: the wavefront of a chain sweeps d and then d + 1
      p.fused_pair = (opts.fused_pairs && s->n_disp <= 32 &&
                      p.block_prefix[p.n_dirs] <= launch_policy().fused_pair_max_waves) ? 1 : 0;
      Timed timed(MPL_KERNEL_FWD_SWEEP, st, p.fused_pair ? 2 : 1);
      if (p.ctx2d && p.L == 21 && decide_team21_soft_fwd(p, opts))
        launch_team21_soft_fwd(p, st);
      else
        launch_soft_fwd(p, train, st);
      if (p.fused_pair) ++d;
    }
    if (label_all) {
      Timed timed(MPL_KERNEL_LABEL, st);
      // the next pass over the same planes, if one is due: cost_final, the re-summed belief plane
      const bool last = it + 1 == n_iter;
      float* out = last ? cost_plane : (rebuild > 0 && (it + 1) % rebuild == 0) ? unary_update : nullptr;
      const bool stored = launch_labels(unary, msg, s->n_dir, P, s->n_disp, 1.f, 0,
                                        label_all + it * P, st, ew_hint(s), kLabelSum, out);
      (last ? have_cost : have_belief) = stored;
    }
  }
  if (!have_cost) aggregate(s, flags, unary, msg, 1.f, 0, cost_final, st);
  return launch_ok("trwp_soft_forward");
}

int mpl_trwp_soft_backward(const mpl_shape* s, unsigned flags, float rho, int n_iter,
                           const float* dcost_final, const float* context,
                           const float* edge_weights, const float* msg_edge_label,
                           const uint8_t* msg_norm_index, float* dunary, float* dcontext,
                           float* dedge_weights, float* dmsg, float* dunary_update, void* stream) {
  int rc = check_shape(s, n_iter);
  if (rc) return rc;
  CallOpts opts;
  if ((rc = read_flags(flags, "trwp_soft_backward", &opts)) != MPL_OK) return rc;
  if (!context || !edge_weights || !dcost_final || !msg_edge_label || !msg_norm_index || !dunary ||
      !dmsg)
    return fail(MPL_EINVAL, "trwp_soft_backward: null tensor pointer");
  hipStream_t st = (hipStream_t)stream;
  const int64_t P = (int64_t)s->batch * s->height * s->width;
  const int64_t N = P * s->n_disp;
  BackParams p;
  memset(&p, 0, sizeof(p));
  p.B = s->batch;
  p.H = s->height;
  p.W = s->width;
  p.L = s->n_disp;
  p.ctx2d = s->ctx2d ? 1 : 0;
  p.rho = rho;
  p.a_out = dunary;
  p.h = dmsg;
  p.edge = edge_weights;
  p.ctx = context;
  p.dedge = dedge_weights;
  if (!place_dcontext(s, flags, n_iter, dcontext, dunary_update, &p))
    return fail(MPL_EINVAL, "MPL_F_DCONTEXT_COPIES needs the tables in dunary_update");
  bool first = true;
  for (int it = n_iter - 1; it >= 0; --it) {
    for (int d = s->n_dir - 1; d >= 0; --d) {  // TRWP_backward_soft.cu:454-538
      fill_dirs(s, d, 1, p.dirs, p.block_prefix, &p.n_dirs);
      p.a_in = first ? dcost_final : dunary;
      p.first_touch = (it == n_iter - 1) && (d & 1);
      p.edge_label = msg_edge_label + (int64_t)it * s->n_dir * N * s->n_disp;
      p.idx_norm = msg_norm_index + (int64_t)it * s->n_dir * P;
      // few chains of at most 32 labels: the wavefront of a chain walks d (odd) and then d - 1
      p.fused_pair = (opts.fused_pairs && s->n_disp <= 32 &&
                      p.block_prefix[p.n_dirs] <= launch_policy().fused_pair_max_waves) ? 1 : 0;
      Timed timed(MPL_KERNEL_BWD_SWEEP, st, p.fused_pair ? 2 : 1);
      if (p.ctx2d && p.L == 21 && decide_team(p, opts, false))
        launch_team21_bwd(p, st);
      else
        launch_soft_bwd(p, st);
      first = false;
      if (p.fused_pair) --d;
    }
  }
  fold_dcontext(p, dcontext, st);
  return launch_ok("trwp_soft_backward");
}

int mpl_soft_weighted_message(int n_trees, int n_disp, const float* message,
                              float* message_soft_sum_norm, uint8_t* message_soft_sum_min_ind,
                              void* stream) {
  if (n_trees < 0 || n_disp < 1 || n_disp > kMaxL)
    return fail(MPL_EINVAL, "soft_weighted_message: n_trees >= 0 and 1 <= n_disp <= %d needed", kMaxL);
  if (!message || !message_soft_sum_norm || !message_soft_sum_min_ind)
    return fail(MPL_EINVAL, "soft_weighted_message: null tensor pointer");
  launch_swm_fwd(message, n_trees, n_disp, message_soft_sum_norm, message_soft_sum_min_ind,
                 (hipStream_t)stream);
  return launch_ok("soft_weighted_message");
}

int mpl_soft_weighted_message_back(int n_trees, int n_disp, const float* dmessage_soft_sum_norm,
                                   const float* message, const uint8_t* message_soft_sum_min_ind,
                                   float* dmessage, void* stream) {
  if (n_trees < 0 || n_disp < 1 || n_disp > kMaxL)
    return fail(MPL_EINVAL, "soft_weighted_message_back: n_trees >= 0 and 1 <= n_disp <= %d needed",
                kMaxL);
  if (!dmessage_soft_sum_norm || !message || !message_soft_sum_min_ind || !dmessage)
    return fail(MPL_EINVAL, "soft_weighted_message_back: null tensor pointer");
  launch_swm_bwd(dmessage_soft_sum_norm, message, message_soft_sum_min_ind, n_trees, n_disp,
                 dmessage, (hipStream_t)stream);
  return launch_ok("soft_weighted_message_back");
}

}  // extern "C"
