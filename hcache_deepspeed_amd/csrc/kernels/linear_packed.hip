// y[M, N] = x[M, K] . dequant(w)[N, K]^T (+ bias) for weight-only quantized w (int8, int4, FP6 e3m2 / e2m3, fp32 scales of
// groups along k), x and y bf16, with the gated unit of w = [gate; up] in the epilogue: more rows than the streams of
// wmix_gemm.hip take.
//
// What bounds these shapes is the weight stream, as in linear.hip, whose ring of LDS-DMA stages, tiles, slices of K and walks
// it shares; a stage is 128 k here, for one scale a weight row. Weights stay packed until a wave has its 32 rows' k in
// registers: codes become bf16, which holds them exactly (packed_codes.h), and a group's 32-bit sum is scaled, so no weight
// is rounded. The tile kernel of wmix_gemm.hip loads 32 bytes a lane from rows that lie apart and scales before it rounds.
//
// Loads from the ring have to be of native vector types: where they were of uint2 and uint4 the compiler, which then sees
// that they may alias the LDS-DMA, waited for every stage on its way (int8 [28672, 4096] gated, 24 rows 41.3 instead of 28.9
// us).
//
// Weights not in the caches, us, tile kernel (to 64 rows) or dequantized for the library -> here, [28672, 4096] gated 24 / 64
// / 128 / 256 rows: int8 50 / 59 / 119 / 142 -> 29 / 37 / 60 / 116, fp6 76 / 89 / 128 / 153 -> 29 / 38 / 60 / 116 (int8 at 16
// rows reads 117 MB in 26 us); [4096, 14336]: int8 29 / 33 / 91 / 92 -> 21 / 26 / 38 / 66, fp6 36 / 53 / 105 / 105 -> 20 / 26
// / 40 / 66. Rows of 96 bytes a stage hold fp6 at 3.8 TB/s.
#include <algorithm>
#include <cmath>

#include "linear_common.h"
#include "packed_codes.h"

namespace {

constexpr int BK = 128;     // reduction depth of a stage: one scale a weight row
constexpr int kGroups = 32;  // scales of a weight row that a workgroup keeps

struct PackedArgs {
  const bf16* x;  // [M, K]
  const uint8_t* w;
  const float* scales;  // [N, K / G]
  const bf16* bias;  // [N] or null
  bf16* y;  // [M, N]
  float* part;  // [S, M, N] where S > 1 (gated: [S, M, 2N])
  int M, N, K, G, S, tm, tn, act, nt;
};

// RB, CB: 16-row blocks of x and of w a wave; NW waves side by side along w, OCC workgroups a CU. GLU: 16 weight rows are 8 of
// gate and the same 8 of up.
template <int FMT, int E, int RB, int CB, int NW, int OCC, bool GLU>
__global__ __launch_bounds__(64 * NW, NW * OCC / 4) void linear_packed_kernel(PackedArgs p) {
  constexpr int R = 16 * RB, W = 16 * CB * NW;
  constexpr int PW = FMT == kInt8 ? 8 : FMT == kInt4 ? 4 : 6;  // 16-byte pieces of a weight row a stage
  constexpr int XU = R / 4, WU = W * PW / 64, PER = (XU + WU + NW - 1) / NW;  // loads of a wave's 64 pieces
  constexpr int kStage = R * 256 + W * PW * 16, kScales = kGroups * W * 4;
  constexpr int D = std::min(8, (160 * 1024 / OCC - kScales) / kStage);
  static_assert(D >= 3 && W * PW % 64 == 0, "tile");
  __shared__ __attribute__((aligned(1024))) char smem[D * kStage + kScales];
  const float* sc = reinterpret_cast<const float*>(smem + D * kStage);
  const int lane = threadIdx.x & 63, g = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // an XCD takes neighbouring tiles, those of the same weight rows first: they meet in its L2
  const int nwg = gridDim.x, orig = blockIdx.x;
  const int q = nwg / 8, r = nwg % 8, xcd = orig % 8;
  int id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + orig / 8;
  const int s = id / (p.tm * p.tn);
  id -= s * p.tm * p.tn;
  const int m0 = id % p.tm * R, tile = id / p.tm;
  const int KT = p.K / BK, k0 = (int)((int64_t)KT * s / p.S), n = (int)((int64_t)KT * (s + 1) / p.S) - k0;
  // weight row of a tile's row; the last one again behind the matrix
  auto row_of = [&](int row) {
    if constexpr (GLU) {
      const int c = std::min(tile * (W / 2) + (row >> 4) * 8 + (row & 7), p.N - 1);
      return row & 8 ? p.N + c : c;
    }
    return std::min(tile * W + row, p.N - 1);
  };

  // scales [row][group]: two rows a load
  const int per_row = p.K / p.G, g0 = k0 * BK / p.G, ng = ((k0 + n) * BK - 1) / p.G - g0 + 1;
  const uint32_t ss = (GLU ? 2u : 1u) * (uint32_t)p.N * (uint32_t)per_row * 4;
#pragma unroll
  for (int i = 0; i < W / 2 / NW; ++i) {
    const int two = i * NW + wv;
    load_lds_4(p.scales, ss, smem + D * kStage + two * 256,
                       ((uint32_t)row_of(2 * two + (lane >> 5)) * (uint32_t)per_row + g0 + std::min(lane & 31, ng - 1)) * 4);
  }

  const bf16* xb = p.x + (int64_t)m0 * p.K;
  const uint32_t xs = (uint32_t)std::min(p.M - m0, R) * (uint32_t)p.K * 2;
  const uint32_t row_bytes = (uint32_t)(p.K / 64) * (PW * 8), ws = (GLU ? 2u : 1u) * (uint32_t)p.N * row_bytes;
  uint32_t src[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int u = std::min(NW * i + wv, XU + WU - 1);  // (loads that are left over repeat the last one)
    if (u < XU) {
      const int row = 4 * u + g;
      src[i] = (uint32_t)row * (uint32_t)p.K * 2 + 16 * ((lane & 15) ^ (row & 15));
    } else {
      const int e = 64 * (u - XU) + lane, row = e / PW, at = e % PW;
      const int c = FMT == kInt8 ? at ^ ((row >> 1) & 7) : FMT == kInt4 ? at ^ ((row >> 2) & 3) : (at + PW - ((row >> 3) & 1)) % PW;
      src[i] = (uint32_t)row_of(row) * row_bytes + 16 * c;
    }
  }
  const int turn = (int)__umulhi((unsigned)tile * 2654435769u, (unsigned)n);
  auto issue = [&](int t, int slot) {
    const int k = k0 + (t + turn < n ? t + turn : t + turn - n);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int u = std::min(NW * i + wv, XU + WU - 1);
      char* d = smem + slot * kStage + u * 1024;
      if (u < XU) load_lds<false>(xb, xs, d, src[i], k * (BK * 2));
      else if (p.nt) load_lds<true>(p.w, ws, d, src[i], k * (PW * 16));
      else load_lds<false>(p.w, ws, d, src[i], k * (PW * 16));
    }
  };
#pragma unroll
  for (int t = 0; t < D - 1; ++t)
    if (t < n) issue(t, t);
  // the lane's 32 k of a weight row: k = 32 g .. 32 g + 31 of the stage
  const int lr = lane & 15, wo = XU * 1024 + (wv * 16 * CB + lr) * PW * 16;
  int woff[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if constexpr (FMT == kInt8) woff[i] = 16 * ((2 * g + (i & 1)) ^ ((lr >> 1) & 7));
    else if constexpr (FMT == kInt4) woff[i] = 16 * (g ^ ((lr >> 2) & 3));
    else woff[i] = 16 * (((3 * g + i) / 2 + (lr >> 3)) % PW) + 8 * ((3 * g + i) & 1);
  }
  f32x4 acc[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  int slot = 0, next = D - 1;
  for (int t = 0; t < n; ++t) {
    if (t + D - 1 <= n) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((D - 2) * PER) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (t + D - 1 < n) issue(t + D - 1, next);
    const char* st = smem + slot * kStage;
    const int grp = (k0 + (t + turn < n ? t + turn : t + turn - n)) * BK / p.G - g0;
    bf16x8 f[CB][4];
    f32x4 by[CB];
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      const char* wr = st + wo + j * 16 * PW * 16;
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      WRaw<FMT> raw;
      if constexpr (FMT == kFp6) {
        u32x2 v[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) v[i] = *reinterpret_cast<const u32x2*>(wr + woff[i]);
        raw = {{v[0].x, v[0].y}, {v[1].x, v[1].y}, {v[2].x, v[2].y}};
      } else {
        u32x4 v = *reinterpret_cast<const u32x4*>(wr + woff[0]);
        raw.a = {v.x, v.y, v.z, v.w};
        if constexpr (FMT == kInt8) {
          v = *reinterpret_cast<const u32x4*>(wr + woff[1]);
          raw.b = {v.x, v.y, v.z, v.w};
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) by[j][e] = sc[(wv * 16 * CB + 16 * j + 4 * g + e) * kGroups + grp];
      codes<FMT, E>(raw, f[j]);
    }
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      f32x4 sum[CB];
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const bf16x8 x = *reinterpret_cast<const bf16x8*>(st + (16 * i + lr) * 256 + 16 * ((4 * g + h) ^ lr));
#pragma unroll
        for (int j = 0; j < CB; ++j) sum[j] = mfma16(f[j][h], x, h == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : sum[j]);
      }
#pragma unroll
      for (int j = 0; j < CB; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][j][e] += sum[j][e] * by[j][e];
    }
    slot = slot + 1 == D ? 0 : slot + 1;
    next = next + 1 == D ? 0 : next + 1;
  }

  // lane: row lane % 16 of x, 4 neighbouring weight rows; gated: lanes from 32 on hold the up rows of those 32 below
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int m = m0 + 16 * i + lr;
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      const int block = wv * CB + j;
      const int c = GLU ? tile * (W / 2) + 8 * block + 4 * (g & 1) : tile * W + 16 * block + 4 * g;
      f32x4 v = acc[i][j];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= kUnit<FMT>;
      if (p.S > 1) {
        const int width = GLU ? 2 * p.N : p.N;
        if (m < p.M && c < p.N)
          *reinterpret_cast<f32x4*>(p.part + ((int64_t)s * p.M + m) * width + c + (GLU && g > 1 ? p.N : 0)) = v;
        continue;
      }
      bf16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (GLU) o[e] = gated(v[e], __shfl_down(v[e], 32, 64), p.act);
        else o[e] = (bf16)(v[e] + (p.bias != nullptr && c < p.N ? (float)p.bias[c + e] : 0.f));
      }
      if (m < p.M && c < p.N && (!GLU || g < 2)) *reinterpret_cast<bf16x4*>(p.y + (int64_t)m * p.N + c) = o;
    }
  }
}

// tiles: workgroups a CU, time of a workgroup in us: once + a stage
struct Tile {
  int rows, cols, each;
  float once, stage;
};
constexpr Tile kTiles[] = {{16, 64, 2, 8.f, 0.25f}, {32, 64, 2, 8.1f, 0.28f}, {64, 64, 2, 8.7f, 0.39f}, {128, 128, 1, 10.3f, 1.29f}};
constexpr int kMaxSlices = 14;

// The tile and the slices of K that take least by this estimate: the stages of the fullest CU, the weights at 8.8 TB/s and
// all stages at 16.5 TB/s from L2, cubes added, since they overlap in part; a further round costs 2.9 us and a sum of slices
// 0.2 + 1.1 a million floats. Fitted to 7,700 times of 17 shapes, 4 to 512 rows (7 % rms); the choice is 3 % slower than the
// best one measured.
static int packed_choice(int M, int N, int K, int G, int fmt) {
  const float bytes = fmt == kInt8 ? 1.f : fmt == kInt4 ? 0.5f : 0.75f;
  float least = 0.f;
  int best = 0;
  for (int t = 0; t < (int)(sizeof(kTiles) / sizeof(Tile)); ++t)
    for (int S = 1; S <= kMaxSlices && (S == 1 || K / BK / S >= 2); ++S) {
      const Tile& c = kTiles[t];
      const int stages = (K / BK + S - 1) / S;
      if (std::min(stages, stages * BK / G + 2) > kGroups) continue;
      const float groups = (float)((M + c.rows - 1) / c.rows) * ((N + c.cols - 1) / c.cols) * S;
      const float fullest = std::ceil(groups / 256.f);
      const float a = fullest * c.stage * stages, b = 1e-6f / 8.8f * N * K * bytes * fullest * 256.f / std::max(128.f, groups);
      const float d = groups * (c.rows * 256 + c.cols * 128 * bytes) * stages / 16.5e6f;
      float us = c.once + std::cbrt(a * a * a + b * b * b + d * d * d) + 2.9f * (std::ceil(groups / (256.f * c.each)) - 1);
      if (S > 1) us += 0.2f + 1.1e-6f * S * M * N;
      if (best == 0 || us < least) {
        least = us;
        best = t + 16 * S;
      }
    }
  return best;
}

}  // namespace

// How hds_packed_rows takes these rows, as tile + 16 x slices of K, or 0 where other kernels are faster or it does not apply.
// N: columns of y; glu: of 2N rows of w; fmt: 0 int8, 1 int4, 2 fp6. For callers to keep by size, as hds_linear_plan.
HDS_EXPORT int hds_packed_plan(int M, int N, int K, int G, int fmt, int glu) {
  if (M < 4 || M > 512 || N < 4 || N % 4 || K < 2 * BK || K % BK || G < BK || G % BK || K % G || fmt < 0 || fmt > 2 ||
      N > 1 << 22 || K > 1 << 20)
    return 0;
  const int rows = glu ? 2 * N : N;
  const int64_t size = (int64_t)rows * K;
  if (size >= (int64_t)1 << 31) return 0;
  // Weights not in the caches, times as fast as what runs otherwise:
  // - up to 16 rows the streams of wmix_gemm.hip. Large int8 matrices 4 / 8 rows [10240, 8192] 1.22 / 1.34, [22016, 6144]
  //   gated 1.08 / 1.16, [28672, 4096] gated 8 rows 1.11; 9 / 16 rows [4096, 14336] 1.09 / 1.23, [20480, 5120] 1.22 / 1.28,
  //   [6144, 4096] 0.96 / 1.13, [2048, 2048] 0.67 / 0.75. int4 and fp6 where the streams keep no rows resident: fp6 9 / 16
  //   rows [15360, 5120] 1.28 / 1.37, [8192, 8192] 1.02 / 1.13, [28672, 4096] gated 0.71 / 0.80; int4 12 rows [10240, 8192]
  //   1.42, [22016, 6144] gated 0.96.
  if (M <= 16 && size < (int64_t)1 << (fmt == kInt8 && M > 8 ? 25 : 26)) return 0;
  if (M <= 16 && fmt != kInt8 && (K <= 4096 || M < (fmt == kInt4 ? 12 : 9))) return 0;
  // - to 64 rows the tiles of wmix_gemm.hip (and the fp6 stream of up to 32), to 256 the weights dequantized for a library
  //   product: 17 to 64 rows int8 1.16 - 1.77, int4 1.22 - 1.76, fp6 1.3 - 3.1 (small matrices to 32 rows 0.95 - 1.0); 96 and
  //   128 rows 1.45 - 2.6; 192 and 256 rows 1.01 - 2.2.
  if (M <= 32 && fmt == kFp6 && size < 1 << 23) return 0;
  // - beyond, the weights are decoded for more rows than it saves passes: [28672, 4096] 384 / 512 rows 0.91 / 0.76; small
  //   matrices gain by their launches ([2048, 2048] 1.1 / 1.2 - 1.4, [4096, 4096] 1.05 - 1.1 / 1.05 - 1.14, [6144, 4096]
  //   0.9).
  if (M > 256 && (size > 1 << 24 || K > 4096)) return 0;
  return packed_choice(M, rows, K, G, fmt);
}

// x [M, K], w packed, scales [N, K / G], bias [N] or null, y [M, N], plan: hds_packed_plan's, part: S x M x N floats where
// its slices S are more than one. ebits: fp6 3 (e3m2) or 2 (e2m3). glu: 0, or 1 + activation code (0 silu, 1 gelu_tanh, 2
// relu): w is 2N rows, gate, then up, without a bias, and part of 2N columns. x and w begin at 16 bytes, y at 8.
HDS_EXPORT int hds_packed_rows(const void* x, const void* w, const float* scales, const void* bias, void* y, float* part, int M,
                               int N, int K, int G, int fmt, int ebits, int glu, int plan, hipStream_t st) {
  const int S = plan / 16, tile = plan % 16, stages = S < 1 ? 0 : (K / BK + S - 1) / S;
  if (M < 1 || M > 512 || N < 4 || N % 4 || K < BK || K % BK || G < BK || G % BK || K % G || glu < 0 || glu > 3 || (glu && bias) ||
      N > 1 << 22 || K > 1 << 20 || (int64_t)(glu ? 2 * N : N) * K >= (int64_t)1 << 31 || S < 1 || S > kMaxSlices || S > K / BK ||
      std::min(stages, stages * BK / G + 2) > kGroups || tile < 0 || tile >= (int)(sizeof(kTiles) / sizeof(Tile)) ||
      (S > 1 && part == nullptr) || ((uintptr_t)x | (uintptr_t)w) & 15 || (uintptr_t)y & 7)
    return hipErrorInvalidValue;
  const int rows = glu ? 2 * N : N, R = kTiles[tile].rows, W = kTiles[tile].cols;
  // Weights that one row of tiles reads go past the caches where a stage's share of a row is a whole line: int8 [28672, 4096]
  // 16 / 64 rows 27.8 / 37.2 -> 25.8 / 36.8 us; fp6's three quarters of one 28.3 -> 33 us at 24 rows.
  PackedArgs p{(const bf16*)x, (const uint8_t*)w, scales, (const bf16*)bias, (bf16*)y, part, M, N, K, G, S, (M + R - 1) / R,
               glu ? (N + W / 2 - 1) / (W / 2) : (N + W - 1) / W, glu - 1, M <= R && fmt == kInt8};
  auto run = [&](auto kernel, int waves) {
    hipLaunchKernelGGL(kernel, dim3(p.tm * p.tn * S), dim3(64 * waves), 0, st, p);
  };
#define HDS_PACKED_TILE(id, F, E, RB, CB, NW, OCC)                                \
  case id:                                                                        \
    if (glu) run(linear_packed_kernel<F, E, RB, CB, NW, OCC, true>, NW);          \
    else run(linear_packed_kernel<F, E, RB, CB, NW, OCC, false>, NW);             \
    break
#define HDS_PACKED(F, E)                     \
  switch (tile) {                            \
    HDS_PACKED_TILE(0, F, E, 1, 1, 4, 2);    \
    HDS_PACKED_TILE(1, F, E, 2, 1, 4, 2);    \
    HDS_PACKED_TILE(2, F, E, 4, 1, 4, 2);    \
    HDS_PACKED_TILE(3, F, E, 8, 2, 4, 1);    \
  }
  if (fmt == kInt8) {
    HDS_PACKED(kInt8, 0)
  } else if (fmt == kInt4) {
    HDS_PACKED(kInt4, 0)
  } else if (ebits == 3) {
    HDS_PACKED(kFp6, 3)
  } else if (ebits == 2) {
    HDS_PACKED(kFp6, 2)
  } else {
    return hipErrorInvalidValue;
  }
#undef HDS_PACKED
#undef HDS_PACKED_TILE
  if (S > 1) {
    const dim3 grid((M * (N / 4) + 255) / 256);
    const SumArgs sum{part, p.bias, p.y, N, M, N, S, p.act};
    if (glu) hipLaunchKernelGGL(linear_sum_kernel<true>, grid, dim3(256), 0, st, sum);
    else hipLaunchKernelGGL(linear_sum_kernel<false>, grid, dim3(256), 0, st, sum);
  }
  return hipGetLastError();
}
