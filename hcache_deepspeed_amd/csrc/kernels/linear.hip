// y[M, N] = x[M, K] . w[N, K]^T (+ bias) in bf16, sums in 32 bits: projections of more rows than the decode kernels take
// (gemv.hip) and fewer than a library product fills the chip with, with the gated unit of w = [gate; up] in the epilogue.
//
// What bounds these shapes is idle CUs, or a weight stream that library tiles do not keep up: [4096, 14336] at 521 rows has
// 48 tiles of 192 x 256, and the library's smaller ones leave L2 as the limit (111 us, 0.56 PFLOP/s). So the reduction is
// split where that pays: every (tile, slice of K) is a workgroup, partial sums go to memory in 32 bits and a second kernel
// adds them in their order, so that results repeat bit for bit.
//
// A workgroup keeps a ring of D stages of 64 k in LDS, filled by LDS-DMA through a buffer descriptor (what lies behind the
// matrices is read as zeros, and unlike global_load_lds it leaves the compiler its counted LDS waits). Rows of 128 bytes keep
// their 16-byte pieces at c ^ ((row >> 1) & 7), which spreads a fragment read over all banks. Half a stage (32 k) is read
// into registers while the half before it is multiplied, with one barrier a stage; waiting for all reads of a stage first, as
// two groups of waves in turn, took 0.62 instead of 0.50 us a stage at 128 x 128.
//
// Time a stage with a full chip, us (PFLOP/s): 64 x 128 0.32 (0.85), 128 x 128 0.43 - 0.50 (1.1), 192 x 128 0.76 (1.1), 256 x
// 128 0.73 - 0.90 (1.2), 256 x 256 1.36 - 1.59 (1.35). The small ones are bound by the lines that a CU has on the way (64
// bytes a ns), the large ones by LDS reads beside the products. Tiles of 32 rows share a CU, so that one's prologue and
// epilogue lie beside another's stream. Weight rows a multiple of 4 KB apart lie alike in the memory's channels: there each
// column of tiles begins its walk along K somewhere else ([28672, 4096], 24 rows 42.5 -> 38.2 us).
//
// Weights not in the caches, us, library -> here: [4096, 14336] 64 / 128 / 192 / 286 / 521 / 1,018 rows 40 / 75 / 103 / 77 /
// 111 / 129 -> 30 / 35 / 40 / 55 / 83 / 105; [4096, 4096] 96 / 128 / 192 / 256 22 / 24 / 33 / 23 -> 15 / 16 / 19 / 20;
// [28672, 4096] gated 24 / 64 / 128 53 / 54 / 58 -> 38 / 40 / 49; [11264, 2048] gated 24 / 128 / 256 20 / 22 / 31 -> 14 / 20
// / 25.
#include <algorithm>
#include <cmath>

#include "linear_common.h"
#include "row_norm.h"

namespace {

constexpr int BK = 64;  // reduction depth of a stage: rows of 128 bytes

struct LinearArgs {
  const bf16* x;  // [M, ldx]
  const bf16* w;  // [N, K]
  const bf16* bias;  // [N] or null
  bf16* y;  // [M, ldy]
  float* part;  // [S, M, N] where S > 1 (gated: [S, M, 2N])
  int64_t ldx, ldy;
  int M, N, K, S, tm, tn, act, nt, apart;
  RowScale scale;  // SCALE
};

// SCALE: up to 16 rows of a residual stream that is still to be scaled (row_norm.h). RB, CB: 16-row blocks of x and of w a wave; WM x WN waves, OCC workgroups a CU. GLU: w is [gate; up] of N rows each; half
// of a tile's and of a wave's columns are gates, the others the same features of up.
template <int RB, int CB, int WM, int WN, int OCC, bool GLU, bool SCALE = false>
__global__ __launch_bounds__(64 * WM * WN, WM * WN * OCC / 4) void linear_kernel(LinearArgs p) {
  constexpr int R = 16 * RB * WM, W = 16 * CB * WN, NW = WM * WN, PER = (R + W) / (8 * NW);
  constexpr int kStage = (R + W) * 128, D = std::min(12, 160 * 1024 / OCC / kStage);
  static_assert((R + W) % (8 * NW) == 0 && R % 8 == 0 && D >= 2, "tile");
  __shared__ __attribute__((aligned(1024))) char smem[D * kStage];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wv / WN, wc = wv % WN;

  // an XCD takes neighbouring tiles, those of the same weight rows first: they meet in its L2
  const int nwg = gridDim.x, orig = blockIdx.x;
  const int q = nwg / 8, r = nwg % 8, xcd = orig % 8;
  int id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + orig / 8;
  const int s = id / (p.tm * p.tn);
  id -= s * p.tm * p.tn;
  const int m0 = id % p.tm * R, n0 = id / p.tm * (GLU ? W / 2 : W);
  const int KT = p.K / BK, k0 = (int)((int64_t)KT * s / p.S), n = (int)((int64_t)KT * (s + 1) / p.S) - k0;

  // a wave fills 8 rows of a stage with a load: x rows, then w rows. What lies behind the matrices is read as zeros.
  auto rest = [&](int64_t rows, int64_t ld) { return (uint32_t)std::min<int64_t>(((rows - 1) * ld + p.K) * 2, 0xfffffff0); };
  const bf16 *xb = p.x + m0 * p.ldx, *wb = p.w + (int64_t)n0 * p.K;
  const uint32_t xs = rest(p.M - m0, p.ldx), ws = rest((GLU ? 2 : 1) * p.N - n0, p.K);
  uint32_t src[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int row = 8 * (NW * i + wv) + (lane >> 3);
    const int ch = (lane & 7) ^ ((row >> 1) & 7);
    const int of_w = row - R + (GLU && row - R >= W / 2 ? p.N - W / 2 : 0);
    src[i] = 16 * ch + 2 * (row < R ? (uint32_t)row * (uint32_t)p.ldx : (uint32_t)of_w * (uint32_t)p.K);
  }
  const int turn = p.apart ? (int)__umulhi((unsigned)(id / p.tm) * 2654435769u, (unsigned)n) : 0;
  auto issue = [&](int t) {
    char* d = smem + (t % D) * kStage + wv * 1024;
    const int k = (k0 + (t + turn < n ? t + turn : t + turn - n)) * 128;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const bool of_x = 8 * (NW * i + wv) < R;  // wave-uniform
      if (p.nt && !of_x) load_lds<true>(wb, ws, d + i * NW * 1024, src[i], k);
      else load_lds<false>(of_x ? xb : wb, of_x ? xs : ws, d + i * NW * 1024, src[i], k);
    }
  };

  // a fragment: row lane % 16, 16-byte piece 4 ks + lane / 16
  const int sw = (lane >> 1) & 7;
  int foff[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) foff[ks] = (lane & 15) * 128 + 16 * ((4 * ks + (lane >> 4)) ^ sw);
  const int xo = wr * 16 * RB * 128, wo = (R + wc * (GLU ? 8 : 16) * CB) * 128;

  f32x4 acc[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 a[2][RB], b[2][CB];
  auto read = [&](int t, int ks) {
    const char* st = smem + (t % D) * kStage + foff[ks];
#pragma unroll
    for (int i = 0; i < RB; ++i) a[ks][i] = *reinterpret_cast<const bf16x8*>(st + xo + i * 2048);
#pragma unroll
    for (int j = 0; j < CB; ++j) b[ks][j] = *reinterpret_cast<const bf16x8*>(st + wo + j * 2048 + (GLU && j >= CB / 2 ? (W / 2 - 8 * CB) * 128 : 0));
  };
  auto multiply = [&](int ks) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j) acc[i][j] = mfma16(b[ks][j], a[ks][i], acc[i][j]);
  };

  RowSums<64 * NW> sums;  // (ahead of the stages: a wait for them is none for those)
  if constexpr (SCALE) sums.load(p.scale);
#pragma unroll
  for (int t = 0; t < D; ++t)
    if (t < n) issue(t);
  if (D <= n) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((D - 1) * PER) : "memory");
  else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  read(0, 0);
  // this stage's second half is on its way while the first is multiplied, and the next stage's first while the second is
  int t = 0;
  for (; t + D < n; ++t) {
    read(t, 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(0);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((D - 2) * PER) : "memory");
    read(t + 1, 0);
    issue(t + D);
    __builtin_amdgcn_sched_barrier(0);
    multiply(1);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (; t < n; ++t) {
    read(t, 1);
    multiply(0);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (t + 1 < n) read(t + 1, 0);
    multiply(1);
  }

  if constexpr (SCALE) {
    float* red = reinterpret_cast<float*>(smem);
    __syncthreads();  // (the last stage has been read)
    sums.add(p.scale, red);
    __syncthreads();
    const float rstd = RowSums<64 * NW>::rstd(p.scale, red, lane & 15);
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j) acc[i][j] *= rstd;
  }
  // lane: row lane % 16 of x, 4 neighbouring columns
  constexpr int CJ = GLU ? CB / 2 : CB;
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int m = m0 + (wr * RB + i) * 16 + (lane & 15);
    if (m >= p.M) continue;
#pragma unroll
    for (int j = 0; j < CJ; ++j) {
      const int c = n0 + (wc * CJ + j) * 16 + 4 * (lane >> 4);
      if (c >= p.N) continue;
      if (p.S > 1) {
        float* d = p.part + ((int64_t)s * p.M + m) * (GLU ? 2 * p.N : p.N) + c;
        *reinterpret_cast<f32x4*>(d) = acc[i][j];
        if constexpr (GLU) *reinterpret_cast<f32x4*>(d + p.N) = acc[i][j + CJ];
        continue;
      }
      bf16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = acc[i][j][e] + (p.bias != nullptr ? (float)p.bias[c + e] : 0.f);
        if constexpr (GLU) o[e] = gated(v, acc[i][j + CJ][e] + (p.bias != nullptr ? (float)p.bias[p.N + c + e] : 0.f), p.act);
        else o[e] = (bf16)v;
      }
      *reinterpret_cast<bf16x4*>(p.y + m * p.ldy + c) = o;
    }
  }
}

// tiles: workgroups a CU, time of a workgroup in us: once + a stage
struct Tile {
  int rows, cols, each;
  float once, stage;
};
constexpr Tile kTiles[] = {{32, 64, 2, 5.5f, 0.13f},   {32, 128, 2, 5.8f, 0.23f},  {64, 64, 1, 5.8f, 0.26f},   {64, 128, 1, 6.4f, 0.33f},
                           {128, 128, 1, 8.3f, 0.43f}, {192, 128, 1, 9.2f, 0.78f}, {256, 128, 1, 10.f, 0.72f}, {256, 256, 1, 10.7f, 1.41f}};
constexpr int kMaxSlices = 12;

// The tile and the slices of K that take least by this estimate: the stages of the fullest CU, the weights at 8.4 TB/s (fewer
// bytes a second where CUs have fewer workgroups than the fullest) and all stages at 19 TB/s from L2, cubes added, since they
// overlap in part; a further round costs 2.6 us and a sum of slices 1.8 + 1.1 a million floats, and 2 of the host's. Fitted
// to 11,000 times of 20 shapes, 5 to 1,018 rows (8 % rms); the choice is 2 % slower than the best one measured.
static int linear_choice(int M, int N, int K) {
  float least = 0.f;
  int best = 0;
  for (int t = 0; t < (int)(sizeof(kTiles) / sizeof(Tile)); ++t)
    for (int S = 1; S <= kMaxSlices && (S == 1 || K / BK / S >= 4); ++S) {
      const Tile& c = kTiles[t];
      const float groups = (float)((M + c.rows - 1) / c.rows) * ((N + c.cols - 1) / c.cols) * S;
      const float fullest = std::ceil(groups / 256.f);
      const int stages = (K / BK + S - 1) / S;
      const float a = fullest * c.stage * stages, b = 2e-6f / 8.4f * N * K * fullest * 256.f / std::max(128.f, groups);
      const float d = groups * (c.rows + c.cols) * 128.f * stages / 19e6f;
      float us = c.once + std::cbrt(a * a * a + b * b * b + d * d * d) + 2.6f * (std::ceil(groups / (256.f * c.each)) - 1);
      if (S > 1) us += 3.8f + 1.1e-6f * S * M * N;
      if (best == 0 || us < least) {
        least = us;
        best = t + 16 * S;
      }
    }
  return best;
}

}  // namespace

// How hds_linear_bf16 takes these rows, as tile + 16 x slices of K, or 0 where a library product is the faster one. N:
// columns of y; glu: of 2N rows of w. For callers to keep by size: the estimates take 3 us of the host.
HDS_EXPORT int hds_linear_plan(int M, int N, int K, int glu) {
  if (M < 9 || M > 1100 || N < 8 || K < 4 * BK || K % BK || N % 8 || K > 1 << 22 || N > 1 << 22) return 0;
  const int rows = glu ? 2 * N : N;
  const int64_t size = (int64_t)rows * K;
  if (size >= (int64_t)1 << 31) return 0;
  // Weights not in the caches, times as fast as the library (up to 16 rows as skinny_lines_kernel):
  // - up to 128 rows, which read the weights once at 6 TB/s and more: [28672, 4096] gated 24 / 64 / 128 rows 53 / 54 / 58 us
  //   -> 38 / 40 / 49, [32000, 4096] 59 / 56 / 59 -> 41 / 42 / 51, [10240, 8192] 1.0 - 1.8, [15360, 5120] 0.9 - 1.1; small
  //   matrices level as kernels ([2048, 2048], [3072, 2048] 0.8 - 1.05), but 10 us of host time instead of the library's 19,
  //   which is what bounds steps of short prompts (40 tokens, four layers of width 2048 663 -> 519 us, of 4096 656 -> 540).
  //   Up to 16 rows where the matrix is large and not sliced: [28672, 4096] 8 / 12 / 16 rows 38.8 / 42.6 / 45.1 -> 37.3 /
  //   37.3 / 37.5, [32000, 4096] 41.5 / 44.9 / 49.2 -> 40.0 / 40.4 / 40.4; smaller ones 0.6 - 1.03.
  const int choice = linear_choice(M, rows, K), S = choice / 16;
  if (M <= 16) return S == 1 && size >= 1 << 25 ? choice : 0;
  // 17 to 32 rows are decode steps, whose launches are recorded once, more often than prompts: smaller matrices are the
  // library's (18 / 24 / 32 sequences, four layers of width 2048, with all of them here 296 / 283 / 315 -> 321 / 309 / 337
  // us, two of 4096 299 / 300 / 358 -> 302 / 304 / 366; a prompt of 24 tokens 658 -> 513). From 33 on recorded steps are
  // level or faster here too (33 / 48 / 64 sequences, four layers of width 2048 382 / 418 / 433 -> 366 / 393 / 396, two of
  // 4096 352 / 376 / 381 -> 350 / 373 / 389, within the noise), although [2048, 2048] alone takes 8.6 / 10.4 us.
  if (M <= 32 && !glu && size < 3 << 23) return 0;
  bool take = M <= 128;
  // - up to 256 with a gated unit, whose kernel and pass it saves ([28672, 4096] 0.93 - 1.04, [11264, 2048] 1.2), or not much
  //   wider than deep ([6144, 4096] 0.87 - 1.35, [4096, 4096] 0.86 - 1.7, [8192, 8192] 1.2 - 1.6), as [32000, 4096] (0.95 -
  //   1.02) is (prompts of 137 / 170 / 200 / 256 tokens, four layers of width 4096, qkv and o 818 / 782 / 779 / 885 -> 777 /
  //   804 / 774 / 852);
  take = take || (M <= 256 && (glu || (K >= 4096 && 2 * rows <= 3 * K)));
  // - to 320 where the library's call is the longer half (0.8 - 1.1; two layers of width 2048, 310 tokens 452 -> 345 us);
  take = take || (M <= 320 && !glu && size <= 1 << 25);
  // - long reductions into few columns, whatever the rows: [4096, 14336] 1.0 - 2.3, [5120, 13824] 0.94 - 2.4. Beyond, the
  //   library's products are the faster ones (521 rows: [28672, 4096] 0.8, [11264, 2048] 0.85, [6144, 4096] 1.0).
  take = take || (K >= 8192 && 2 * rows <= K && size >= 1 << 24);
  return take ? choice : 0;
}

// x [M, ldx], w [N, K], bias [N] or null, y [M, ldy], plan: hds_linear_plan's, part: S x M x N floats where its slices S are
// more than one. glu: 0, or 1 + activation code (0 silu, 1 gelu_tanh, 2 relu): w [2N, K] is gate rows, then up rows, y =
// act(gate) up, and bias and part are of 2N columns. Rows of x and w begin at 16 bytes, of y at 8.
static int linear(const void* x, int64_t ldx, const void* w, const void* bias, void* y, int64_t ldy, float* part, int M, int N,
                  int K, int glu, int plan, const RowScale& scale, hipStream_t st) {
  const int S = plan / 16, tile = plan % 16;
  if (M < 1 || M > 1100 || N < 8 || K < 4 * BK || K % BK || N % 8 || K > 1 << 22 || N > 1 << 22 || glu < 0 || glu > 3 ||
      (int64_t)(glu ? 2 * N : N) * K >= (int64_t)1 << 31 || S < 1 || S > kMaxSlices || S > K / BK || tile < 0 ||
      tile >= (int)(sizeof(kTiles) / sizeof(Tile)) || (S > 1 && part == nullptr) || ldx < K || ldx % 8 || ldx > 1 << 22 || ldy < N ||
      ldy % 4 || ((uintptr_t)x | (uintptr_t)w) & 15 || (uintptr_t)y & 7)
    return hipErrorInvalidValue;
  const int rows = glu ? 2 * N : N, R = kTiles[tile].rows, W = kTiles[tile].cols;
  LinearArgs p{(const bf16*)x, (const bf16*)w, (const bf16*)bias, (bf16*)y, part, ldx, ldy, M, N, K, S, (M + R - 1) / R,
               (rows + W - 1) / W, glu - 1, 0, K % 2048 == 0, scale};
  if (glu) p.tn = (N + W / 2 - 1) / (W / 2);
  // Weights that one row of tiles reads go past the caches: [28672, 4096] 24 / 64 rows 43.5 / 44.7 -> 38.2 / 40.0 us. Not with
  // slices, whose walks are short ([4096, 14336], 128 rows 33.8 / 38.1), but in the smallest tile (24 rows 25.4 -> 24.0).
  p.nt = p.tm == 1 && (S == 1 || (R == 32 && p.apart));
  auto run = [&](auto kernel, int waves) {
    hipLaunchKernelGGL(kernel, dim3(p.tm * p.tn * S), dim3(64 * waves), 0, st, p);
  };
  if (scale.ssq != nullptr) {
    if (M > 16 || S > 1 || tile > 1) return hipErrorInvalidValue;
    if (tile == 0) glu ? run(linear_kernel<1, 2, 2, 2, 2, true, true>, 4) : run(linear_kernel<1, 2, 2, 2, 2, false, true>, 4);
    else glu ? run(linear_kernel<2, 2, 1, 4, 2, true, true>, 4) : run(linear_kernel<2, 2, 1, 4, 2, false, true>, 4);
    return hipGetLastError();
  }
#define HDS_LINEAR(id, RB, CB, WM, WN, OCC)                                     \
  case id:                                                                      \
    if (glu) run(linear_kernel<RB, CB, WM, WN, OCC, true>, WM * WN);            \
    else run(linear_kernel<RB, CB, WM, WN, OCC, false>, WM * WN);               \
    break
  switch (tile) {
    HDS_LINEAR(0, 1, 2, 2, 2, 2);
    HDS_LINEAR(1, 2, 2, 1, 4, 2);
    HDS_LINEAR(2, 2, 2, 2, 2, 1);
    HDS_LINEAR(3, 2, 2, 2, 4, 1);
    HDS_LINEAR(4, 4, 2, 2, 4, 1);
    HDS_LINEAR(5, 6, 4, 2, 2, 1);
    HDS_LINEAR(6, 4, 4, 4, 2, 1);
    HDS_LINEAR(7, 8, 4, 2, 4, 1);
  }
#undef HDS_LINEAR
  if (S > 1) {
    const dim3 grid((M * (N / 4) + 255) / 256);
    const SumArgs sum{part, p.bias, p.y, ldy, M, N, S, p.act};
    if (glu) hipLaunchKernelGGL(linear_sum_kernel<true>, grid, dim3(256), 0, st, sum);
    else hipLaunchKernelGGL(linear_sum_kernel<false>, grid, dim3(256), 0, st, sum);
  }
  return hipGetLastError();
}

HDS_EXPORT int hds_linear_bf16(const void* x, int64_t ldx, const void* w, const void* bias, void* y, int64_t ldy, float* part,
                               int M, int N, int K, int glu, int plan, hipStream_t st) {
  return linear(x, ldx, w, bias, y, ldy, part, M, N, K, glu, plan, RowScale{}, st);
}

// The same of up to 16 rows of K = 16 parts columns that are still to be scaled, from the sums of their squares ssq [parts][16]:
// plans of one slice and of the tiles of 32 rows
HDS_EXPORT int hds_linear_scaled_bf16(const void* x, const void* w, void* y, const float* ssq, float eps, int M, int N, int K,
                                      int glu, int plan, hipStream_t st) {
  if (ssq == nullptr) return hipErrorInvalidValue;
  return linear(x, K, w, nullptr, y, N, nullptr, M, N, K, glu, plan, RowScale{ssq, K / 16, eps}, st);
}
