// Layout change between the network's (batch, labels, H, W) tensors and the label-innermost
// (batch, H, W, labels) layout of the message-passing kernels: a batched 2-D transpose.
//
// The reference's module does this with permute().contiguous() on the way in and out
// (pytorch/MP_module.py:199, 203, 233); the generic strided copy behind that moves 0.4-1.9 TB/s at
// 1500 x 2000 x 192, the tiled transpose below is bound by HBM like any other streaming kernel.

#include "mp_common.h"

using namespace mpl;

namespace {

constexpr int kTile = 64;

// src (batch, rows, cols) -> dst (batch, cols, rows).  One 64 x 64 tile per workgroup of 64 x 4 threads:
// rows of 256 contiguous bytes in, through LDS (padded against bank conflicts), rows of 256 contiguous
// bytes out.  Bound by HBM.  Where rows are not whole cache lines the tiles beside each other share lines:
// groups of kGroup tiles along the long side go to one die of the chip (locate_chain), and what is shared
// carries no non-temporal hint -- all loads, and the stores unless NT (whole lines).  Measured, us into the
// label-innermost layout / out of it, every access with the hint and tiles dealt out one by one -> this:
// 128 labels 375x1242 143 / 188 -> 86 / 130; 96 labels 384x1248 99 / 114 -> 71 / 75; 192 labels 256x512 60 / 64 ->
// 46 / 46, 1500x2000 1000 / 999 -> 1005 / 961; 150 labels 301x405 68 / 71 -> 42 / 45; 60 labels 375x450 37 / 44 ->
// 29 / 30.  (Tiles of 64 x 128: 118 / 148 on the first.)
constexpr int kGroup = 8;
template <bool LONG_ROWS, bool NT>
__global__ void __launch_bounds__(256) transpose_kernel(const float* __restrict__ src,
                                                        float* __restrict__ dst, int64_t rows,
                                                        int64_t cols) {
  __shared__ float tile[kTile][kTile + 1];
  const int tx = threadIdx.x, ty = threadIdx.y;
  // the long side of the matrix runs along the grid's x axis
  const int bx = xcd_block((int)blockIdx.x, (int)gridDim.x, kGroup);
  const int64_t r0 = (int64_t)(LONG_ROWS ? bx : (int)blockIdx.y) * kTile;
  const int64_t c0 = (int64_t)(LONG_ROWS ? (int)blockIdx.y : bx) * kTile;
  const int64_t plane = rows * cols;
  const float* s = src + (int64_t)blockIdx.z * plane;
  float* d = dst + (int64_t)blockIdx.z * plane;
#pragma unroll
  for (int k = 0; k < kTile; k += 4) {
    const int64_t r = r0 + ty + k, c = c0 + tx;
    if (r < rows && c < cols) tile[ty + k][tx] = s[r * cols + c];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kTile; k += 4) {
    const int64_t c = c0 + ty + k, r = r0 + tx;
    if (r < rows && c < cols) {
      if (NT)
        __builtin_nontemporal_store(tile[tx][ty + k], d + c * rows + r);
      else
        d[c * rows + r] = tile[tx][ty + k];
    }
  }
}

}  // namespace

extern "C" {

int mpl_transpose(const float* src, float* dst, int batch, int64_t rows, int64_t cols,
                  void* stream) {
  if (src == nullptr || dst == nullptr) return fail(MPL_EINVAL, "transpose: null pointer");
  if (batch < 0 || rows < 0 || cols < 0) return fail(MPL_EINVAL, "transpose: negative size");
  if (batch == 0 || rows == 0 || cols == 0) return MPL_OK;
  // the shorter side goes on the grid's y axis (65535 tiles at most)
  const int long_rows = rows > cols ? 1 : 0;
  const int64_t ny = ((long_rows ? cols : rows) + kTile - 1) / kTile;
  const int64_t nx = ((long_rows ? rows : cols) + kTile - 1) / kTile;
  if (ny > 65535 || nx > 0x7fffffff || batch > 65535)
    return fail(MPL_EINVAL, "transpose: too large (the shorter side must stay below 4 M elements)");
  const dim3 grid((unsigned)nx, (unsigned)ny, (unsigned)batch), block(kTile, 4);
  const bool whole_lines = (rows * (int64_t)sizeof(float)) % kLineBytes == 0;
  auto kernel = long_rows ? (whole_lines ? transpose_kernel<true, true> : transpose_kernel<true, false>)
                          : (whole_lines ? transpose_kernel<false, true> : transpose_kernel<false, false>);
  kernel<<<grid, block, 0, (hipStream_t)stream>>>(src, dst, rows, cols);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MPL_ELAUNCH, "transpose: %s", hipGetErrorString(e));
  return MPL_OK;
}

}  // extern "C"
