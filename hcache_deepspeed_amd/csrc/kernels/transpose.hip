// 2-D bf16 transpose dst[c][r] = src[r][c] (src row stride lds elements, dst contiguous [cols, rows]).
// Used to put weight-gradient GEMMs dW = dY^T X into hipBLASLt's fast NT layout (ops/gemm.py wgrad): the transposed
// copies are written once at HBM rate instead of the TN GEMM running ~25 % below the NT one at the bench shapes.
// Tile 64 x 64 through LDS: 16-B global loads along src rows, 16-B global stores along dst rows; the LDS tile is
// padded to 66 elements per row so the column reads of the store phase spread over the banks.
#include "transpose_tile.h"

namespace {
using namespace hds;

constexpr int TT = 64, PAD = 66;

__global__ __launch_bounds__(256) void transpose_bf16_kernel(const bf16* __restrict__ src, bf16* __restrict__ dst,
                                                             int rows, int cols, int64_t lds) {
  __shared__ bf16 tile[TT * PAD];
  const int r0 = blockIdx.y * TT, c0 = blockIdx.x * TT;
  const int tid = threadIdx.x;
  // load: 64 rows x 8 vectors of 8 -> 512 vectors, 2 per thread
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int v = tid + 256 * i, rr = v >> 3, cc = (v & 7) * 8;
    const int r = r0 + rr, c = c0 + cc;
    bf16x8 x;
    if (r < rows && c + 7 < cols) {
      x = *reinterpret_cast<const bf16x8*>(src + (int64_t)r * lds + c);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = (r < rows && c + j < cols) ? src[(int64_t)r * lds + c + j] : (bf16)0.f;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) tile[rr * PAD + cc + j] = x[j];
  }
  __syncthreads();
  // store: dst row = source column c0 + cr, 8 consecutive source rows per vector
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int v = tid + 256 * i, cr = v >> 3, rc = (v & 7) * 8;
    const int c = c0 + cr, r = r0 + rc;
    if (c >= cols) continue;
    bf16x8 y;
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = tile[(rc + j) * PAD + cr];
    if (r + 7 < rows) {
      *reinterpret_cast<bf16x8*>(dst + (int64_t)c * rows + r) = y;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (r + j < rows) dst[(int64_t)c * rows + r + j] = y[j];
    }
  }
}

// v2: 64 x 128 tiles, every LDS access 8 or 16 B wide (transpose_tile.h). v1's LDS traffic is one 2-B write and one 2-B read
// per element (32 LDS instructions per thread per 16 B moved). v1 / v2: [8192, 28672] 216 / 176 us, [8192, 4096] 32 / 22, [1024,
// 5632] 6.9 / 4.9, [1016, 11264] 13.1 / 12.3, [72, 4096] 2.8 / 3.2. v2 makes the padded transposes and runs where variant 2 is
// asked for, v1 is ops/gemm.py's default. dst rows may be longer than src has rows: zeros.
template <bool LINES>
__global__ __launch_bounds__(256) void transpose_bf16_v2_kernel(const bf16* __restrict__ src, bf16* __restrict__ dst,
                                                                int rows, int cols, int64_t lds, int ldd) {
  __shared__ __attribute__((aligned(16))) bf16 tile[kTrRows * kTrCols];
  const TileAt at = tile_at<LINES>(ldd, cols);
  const int tid = threadIdx.x;
  const bool full = (at.r0 + kTrRows <= rows) && (at.c0 + kTrCols <= cols);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int v = tid + 256 * i, rr = v >> 4, ch = v & 15;
    const int r = at.r0 + rr, c = at.c0 + 8 * ch;
    bf16x8 x;
    if (full || (r < rows && c + 7 < cols)) {
      x = *reinterpret_cast<const bf16x8*>(src + (int64_t)r * lds + c);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = (r < rows && c + j < cols) ? src[(int64_t)r * lds + c + j] : (bf16)0.f;
    }
    *reinterpret_cast<bf16x8*>(&tile[tile_chunk(rr, ch)]) = x;
  }
  __syncthreads();
  store_transposed<LINES>(tile, dst, at, ldd, cols);
}

}  // namespace

// rows % 8 == 0 and lds % 8 == 0 keep the vector accesses aligned (checked by the caller)
// variant 1: 64 x 64 tile, 2-B LDS accesses; 2: 64 x 128 tile, 16-B writes / 8-B reads + v_perm
HDS_EXPORT int hds_transpose_bf16_var(const void* src, void* dst, int rows, int cols, long lds, int variant,
                                      hipStream_t st) {
  if (rows <= 0 || cols <= 0) return hipSuccess;
  if (rows % 8 || lds % 8 || ((uintptr_t)src & 15) || ((uintptr_t)dst & 15)) return hipErrorInvalidValue;
  if (variant == 1) {
    dim3 grid((cols + TT - 1) / TT, (rows + TT - 1) / TT);
    hipLaunchKernelGGL(transpose_bf16_kernel, grid, dim3(256), 0, st, (const bf16*)src, (bf16*)dst, rows, cols,
                       (int64_t)lds);
  } else {
    const dim3 grid(tile_count(rows, cols));
    if (tile_lines(rows, dst))
      hipLaunchKernelGGL(transpose_bf16_v2_kernel<true>, grid, dim3(256), 0, st, (const bf16*)src, (bf16*)dst, rows,
                         cols, (int64_t)lds, rows);
    else
      hipLaunchKernelGGL(transpose_bf16_v2_kernel<false>, grid, dim3(256), 0, st, (const bf16*)src, (bf16*)dst, rows,
                         cols, (int64_t)lds, rows);
  }
  return hipGetLastError();
}

// The same for any number of rows, to rows of ldd (a multiple of 64, at least `rows`) whose ends are zeros: as operands of a
// product over the rows they are aligned and add nothing. dst 128-byte aligned. [1018, 11264] 9 us; by strided copies 28 us
// for half as many columns.
HDS_EXPORT int hds_transpose_bf16_pad(const void* src, void* dst, int rows, int cols, long lds, int ldd, hipStream_t st) {
  if (rows <= 0 || cols <= 0) return hipSuccess;
  if (lds % 8 || ldd % 64 || ldd < rows || ((uintptr_t)src & 15) || ((uintptr_t)dst & 127)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(transpose_bf16_v2_kernel<true>, dim3(tile_count(ldd, cols)), dim3(256), 0, st, (const bf16*)src,
                     (bf16*)dst, rows, cols, (int64_t)lds, ldd);
  return hipGetLastError();
}
