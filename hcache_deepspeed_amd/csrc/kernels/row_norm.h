// RMS norms of a few rows (up to 16) without a launch of their own, for the products of decode steps (gemv.hip, linear.hip).
//
// norm(y + res) = r rstd gamma with r = y + res, and rstd is one number of a row. The product that makes y adds the residual,
// stores r and bf16(r gamma), and leaves each workgroup's sums of r^2; the product behind it reads bf16(r gamma) as its rows and
// multiplies its finished 32-bit sums by rstd. The rows are rounded once, as bf16(r rstd gamma) is. A norm's launch in a chain
// of products takes 4 to 5 us, which are its two round trips; the sums are read beside the first weights.
#pragma once
#include "hds_common.h"

namespace hds {

// Rows are to be scaled by rsqrt(sum of ssq[i][row] over the parts / (16 parts) + eps); ssq null: not
struct RowScale {
  const float* ssq;  // [parts][16]
  int parts;
  float eps;
};

// What becomes of a product's rows y: r = bf16(y + res) and, in place of y, bf16(r gamma); ssq [tile of 16 columns][16 rows]
struct RowNorm {
  const bf16* res;  // [M, N], null: nothing
  const bf16* gamma;  // [N]
  bf16* r;  // [M, N]
  float* ssq;
};

// The sums of a workgroup of T threads: loaded at its beginning, added at its end. 4 parts a thread are on their way at once
template <int T>
struct RowSums {
  f32x4 v[4];
  __device__ __forceinline__ void load(const RowScale& s) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = (int)threadIdx.x + T * i;
      v[i] = at < 4 * s.parts ? reinterpret_cast<const f32x4*>(s.ssq)[at] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  // red: [T / 64][16] floats; a barrier has to follow
  __device__ __forceinline__ void add(const RowScale& s, float* red) {
    f32x4 sum = (v[0] + v[1]) + (v[2] + v[3]);
    for (int at = (int)threadIdx.x + T * 4; at < 4 * s.parts; at += T) sum += reinterpret_cast<const f32x4*>(s.ssq)[at];
    const int lane = threadIdx.x & 63;  // of rows 4 (lane & 3) .. + 3
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma unroll
      for (int o = 4; o < 64; o *= 2) sum[e] += __shfl_xor(sum[e], o, 64);
    }
    if (lane < 4) *reinterpret_cast<f32x4*>(red + (threadIdx.x >> 6) * 16 + 4 * lane) = sum;
  }
  static __device__ __forceinline__ float rstd(const RowScale& s, const float* red, int row) {
    float sum = red[row];
#pragma unroll
    for (int w = 1; w < T / 64; ++w) sum += red[w * 16 + row];
    return rsqrtf(sum / (16.f * (float)s.parts) + s.eps);
  }
};

// A tile's finished sums: lane = row lane & 15, columns n .. n + 3 of the 16 of `tile`. res and gamma: loaded before.
__device__ __forceinline__ void store_normed(const RowNorm& o, bf16* y, int64_t at, const f32x4& acc, const bf16x4& res,
                                             const bf16x4& gamma, int tile, int lane, bool live) {
  bf16x4 r, g;
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    r[e] = (bf16)((float)(bf16)acc[e] + (float)res[e]);  // (rounded twice, as the product and the sum by themselves are)
    const float v = (float)r[e];
    g[e] = (bf16)(v * (float)gamma[e]);
    ss += v * v;
  }
  if (live) {
    *reinterpret_cast<bf16x4*>(o.r + at) = r;
    *reinterpret_cast<bf16x4*>(y + at) = g;
  }
  ss += __shfl_xor(ss, 16, 64);
  ss += __shfl_xor(ss, 32, 64);
  if (lane < 16) o.ssq[tile * 16 + lane] = ss;
}

}  // namespace hds
