// A tile of 64 rows x 128 columns of 16-bit elements that goes through LDS to its transposed place.
//
// What bounds such a kernel is how its lines meet memory: the tile's rows are 256 bytes apiece on one side, its columns 128
// bytes on the other. Workgroups in a row take tiles below each other, so that the 128-byte pieces of a transposed row are
// written side by side; eight lanes write a piece whole, and it passes the caches by. Reading LDS costs no bank conflict:
// chunk c (16 bytes) of row r lies at c ^ 2 (r / 8). [8192, 28672]: tiles beside each other 232 us, below each other 187,
// pieces by eight lanes 185 and non-temporal 174 (5.4 TB/s); tiles of 128 rows 184 and 175.
// Where the pieces are no whole lines (LINES: false), neighbours below each other would share lines between XCDs: tiles beside
// each other there, and through the caches ([1016, 11264]: 14.5 us, 15.9 below each other).
#pragma once
#include "hds_common.h"

namespace hds {

constexpr int kTrRows = 64, kTrCols = 128;

struct TileAt {
  int r0, c0;
};
template <bool LINES>
__device__ __forceinline__ TileAt tile_at(int rows, int cols) {
  if constexpr (LINES) {
    const int nr = rows / kTrRows;
    return {(int)(blockIdx.x % nr) * kTrRows, (int)(blockIdx.x / nr) * kTrCols};
  } else {
    const int nc = (cols + kTrCols - 1) / kTrCols;
    return {(int)(blockIdx.x / nc) * kTrRows, (int)(blockIdx.x % nc) * kTrCols};
  }
}
__host__ inline int64_t tile_count(int rows, int cols) {
  return (int64_t)((rows + kTrRows - 1) / kTrRows) * ((cols + kTrCols - 1) / kTrCols);
}
// whole lines: every transposed row begins on one
__host__ inline bool tile_lines(int rows, const void* dst) { return rows % 64 == 0 && (uintptr_t)dst % 128 == 0; }

// chunk ch (8 elements) of row r
__device__ __forceinline__ int tile_chunk(int r, int ch) { return r * kTrCols + 8 * (ch ^ (2 * (r >> 3))); }

// the tile's columns c0 .. to the rows of dst [cols, rows] (rows % 8 == 0); 256 threads
template <bool LINES>
__device__ __forceinline__ void store_transposed(const bf16* tile, bf16* __restrict__ dst, TileAt at, int rows, int cols) {
  const int lr = threadIdx.x & 7, lc = threadIdx.x >> 3, r = at.r0 + 8 * lr;
  u32x2 v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    v[j] = *reinterpret_cast<const u32x2*>(&tile[tile_chunk(8 * lr + j, lc >> 1) + 4 * (lc & 1)]);
  if (r >= rows) return;  // a block of eight rows is all in or all out
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = at.c0 + 4 * lc + i;
    if (c >= cols) break;
    // element i of row j sits in dword i / 2 of v[j], low half for even i; pack rows (2k, 2k+1) into word k
    const uint32_t sel = (i & 1) ? 0x07060302u : 0x05040100u;
    u32x4 y;
#pragma unroll
    for (int k = 0; k < 4; ++k) y[k] = __builtin_amdgcn_perm(v[2 * k + 1][i >> 1], v[2 * k][i >> 1], sel);
    u32x4* to = reinterpret_cast<u32x4*>(dst + (int64_t)c * rows + r);
    if constexpr (LINES) store_nt(to, y);
    else *to = y;
  }
}

}  // namespace hds
