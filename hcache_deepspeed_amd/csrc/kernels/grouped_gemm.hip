// Grouped (MoE) GEMM for gfx950: for every expert e, Y[o_e : o_{e+1}] = X[o_e : o_{e+1}] . W[e]^T
// with X [T, K] expert-contiguous rows (the permuted token order), W [E, N, K] (nn.Linear layout) and
// o = exclusive prefix of the per-expert row counts, kept ON THE DEVICE (no host sync on the routing).
//
// Reference parity: SURVEY.md §2.10 N15 / §2.11 K37 — the CUTLASS grouped MoE GEMM of
// inference/v2/kernels/cutlass_ops/moe_gemm (external libdeepspeedft). Not a translation: one launch covers
// every expert's ragged row block, no capacity padding (dropless), and the tile schedule is built on the GPU.
//
// Design (cdna_hip_programming.md §3/§5):
//   * a tiny planning kernel turns the device offsets into a tile list (expert, m0) and a tile count;
//     the GEMM grid is the host-side upper bound ceil(T/128)+E, blocks past the count exit at once;
//   * 128(N) x 128(tokens) block tile, BK = 128, 4 waves each owning a 64 x 64 quadrant = 2 x 2
//     v_mfma_f32_32x32x16_bf16 accumulators. Operand orientation D = W . X^T puts the token on the lane
//     and 4 consecutive output features in consecutive accumulator registers, so the epilogue writes
//     8-byte bf16x4 vectors of one output row;
//   * both operands are K-contiguous, staged by LDS-DMA (global_load_lds_dwordx4) into the XOR-swizzled
//     64 x 256 B tiles of attn_common.h (conflict-free ds_read_b128 A/B fragments), double-buffered:
//     the next K tile streams in while the current one feeds the MFMAs;
//   * options of the larger tiles (serving, hds_experts_gemm): X rows read through an index list instead of being permuted first; W = [gate;
//     up] with the activation silu(gate) * up or the clamped unit, optionally after a factor per row, in the epilogue -- a
//     wave then holds the accumulators of the same features of both halves; a tile list made elsewhere (experts.hip);
//   * blockIdx.x walks N tiles fastest so the (consecutively dispatched, XCD-round-robin) blocks of one
//     token tile share the X tile in L2 while W[e] streams.
#include <algorithm>

#include "attn_common.h"

using namespace hds;
using namespace hds::attn;

namespace {

constexpr int BM = 128;  // tokens per block tile
constexpr int BN = 128;  // output features per block tile
constexpr int BK = 128;  // reduction depth per stage (one 256-byte bf16 row per tile row)

template <int TM>
__global__ __launch_bounds__(64) void gg_plan_kernel(const int* __restrict__ offs, int E, int T,
                                                     int* __restrict__ tile_e, int* __restrict__ tile_m,
                                                     int* __restrict__ n_tiles, int max_tiles) {
  // single wave: serial prefix over experts (E <= a few hundred), lanes fill each expert's tiles
  const int lane = threadIdx.x;
  int base = 0;
  for (int e = 0; e < E; ++e) {
    const int lo = min(max(offs[e], 0), T), hi = min(max(offs[e + 1], lo), T);  // never trust offsets
    const int t = (hi - lo + TM - 1) / TM;
    for (int i = lane; i < t; i += 64) {
      if (base + i < max_tiles) {
        tile_e[base + i] = e;
        tile_m[base + i] = i * TM;
      }
    }
    base += t;
  }
  if (lane == 0) *n_tiles = base < max_tiles ? base : max_tiles;
}

// epilogue of gate | up products
struct GatedUnit {
  const float* weight;  // [rows] or null
  int clamped;
  float limit;
  __device__ __forceinline__ float factor(int row) const { return weight != nullptr ? weight[row] : 1.f; }
  __device__ __forceinline__ float operator()(float g, float u, float w) const {
    g *= w;
    u *= w;
    if (!clamped) return g / (1.f + __expf(-g)) * u;
    g = fminf(g, limit);
    return g / (1.f + __expf(-1.702f * g)) * (fminf(fmaxf(u, -limit), limit) + 1.f);
  }
};

__global__ __launch_bounds__(256) void gg_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                 bf16* __restrict__ y, const int* __restrict__ offs,
                                                 const int* __restrict__ tile_e, const int* __restrict__ tile_m,
                                                 const int* __restrict__ n_tiles, int T, int N, int K, int ldy) {
  const int t = blockIdx.y;
  if (t >= *n_tiles) return;  // block-uniform exit before any barrier
  const int e = tile_e[t];
  const int m0 = tile_m[t];
  const int row0 = min(max(offs[e], 0), T);
  const int rows = min(max(offs[e + 1], row0), T) - row0;  // >= 1: the plan only emits tiles of non-empty experts
  const int n0 = blockIdx.x * BN;

  __shared__ __attribute__((aligned(16))) char smem[2 * 65536];
  // buffer b: W tile halves at [b*64K, +16K, ...], X tile halves at [b*64K + 32K, +16K]
  const bf16* wb = w + (int64_t)e * N * K + (int64_t)n0 * K;
  const bf16* xb = x + (int64_t)row0 * K;
  auto wrow = [&](int half, int kt) {
    return [=](int r) { return wb + (int64_t)(64 * half + r) * K + (int64_t)kt * BK; };
  };
  auto xrow = [&](int half, int kt) {
    return [=](int r) {
      int m = m0 + 64 * half + r;
      m = m < rows ? m : rows - 1;
      return xb + (int64_t)m * K + (int64_t)kt * BK;
    };
  };
  auto stage = [&](int buf, int kt) {
    char* s = smem + buf * 65536;
    stage_tile64<4>(s, wrow(0, kt));
    stage_tile64<4>(s + 16384, wrow(1, kt));
    stage_tile64<4>(s + 32768, xrow(0, kt));
    stage_tile64<4>(s + 49152, xrow(1, kt));
  };

  const int wv = threadIdx.x >> 6;
  const int wn = wv & 1, wm = wv >> 1;
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};

  const int KT = K / BK;
  stage(0, 0);
  __syncthreads();
  for (int kt = 0; kt < KT; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < KT) stage(buf ^ 1, kt + 1);
    const char* Wt = smem + buf * 65536 + wn * 16384;
    const char* Xt = smem + buf * 65536 + 32768 + wm * 16384;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const bf16x8 a0 = read_rows(Wt, 0, ks), a1 = read_rows(Wt, 32, ks);
      const bf16x8 b0 = read_rows(Xt, 0, ks), b1 = read_rows(Xt, 32, ks);
      acc[0][0] = mfma(a0, b0, acc[0][0]);
      acc[0][1] = mfma(a0, b1, acc[0][1]);
      acc[1][0] = mfma(a1, b0, acc[1][0]);
      acc[1][1] = mfma(a1, b1, acc[1][1]);
    }
    __syncthreads();
  }

  // epilogue: lane = token, registers 4g..4g+3 = 4 consecutive output features
  const int lane = threadIdx.x & 63;
  const int h = lane >> 5;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int m = m0 + 64 * wm + 32 * j + (lane & 31);
    if (m >= rows) continue;
    bf16* yr = y + (int64_t)(row0 + m) * ldy + n0 + 64 * wn;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        bf16x4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = (bf16)acc[i][j][4 * g + q];
        *reinterpret_cast<bf16x4*>(yr + 32 * i + acc_row(4 * g, h)) = v;
      }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Large-expert variant: 256 x 256 block tile, BK = 64, 8 waves (2 along N x 4 along tokens, 128 x 64 per wave =
// 4 x 2 accumulators). The per-wave tile halves the LDS bytes per MFMA of the 128^2 kernel (6 ds_read_b128 per
// 8 MFMA instead of 4 per 4), which is what bounds the small tile. LDS: two buffers of (256 + 256) rows x 128 B
// = 128 KB; rows of 128 B use the XOR swizzle chunk ^ ((row >> 1) & 7): a 16-lane ds_read_b128 group reading 16
// consecutive rows at one logical chunk hits 16 distinct 16-B bank slots (row & 1 selects the half of the
// 256-B bank line). Staging is LDS-DMA (lane-linear destination, swizzle applied to the source address).
// Blocks are remapped so each XCD works on a contiguous range of (token tile, N tile) pairs, rastered in groups of
// 4 token tiles so co-resident blocks share X and W panels in the same L2.
// ---------------------------------------------------------------------------------------------------------------
constexpr int BM2 = 256, BN2 = 256, BK2 = 64;

__device__ __forceinline__ int off128(int row, int ch) { return row * 128 + 16 * (ch ^ ((row >> 1) & 7)); }

// stage `rows` x 128 B (rows % 64 == 0) with an NW-wave block: one wave-instruction fills 8 rows
template <int NW, int ROWS, typename RowPtr>
__device__ __forceinline__ void stage128(char* lds, RowPtr row_ptr) {
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  constexpr int PER = ROWS / 8 / NW;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int n = w * PER + i;
    const int row = 8 * n + (lane >> 3);
    const int ch = (lane & 7) ^ ((row >> 1) & 7);
    const char* src = (const char*)row_ptr(row) + ch * 16;
    __builtin_amdgcn_global_load_lds((gbl_void*)src, (lds_void*)(lds + n * 1024), 16, 0, 0);
  }
}

__device__ __forceinline__ bf16x8 frag128(const char* lds, int row0, int ks) {
  const int lane = threadIdx.x & 63;
  return *reinterpret_cast<const bf16x8*>(lds + off128(row0 + (lane & 31), 2 * ks + (lane >> 5)));
}

// GATHER: row r of the sorted order is x[src[r]] (n_src rows of x). GLU: w holds 2N rows per expert, gate then up.
template <bool GATHER, bool GLU>
__global__ __launch_bounds__(512) void gg_big_kernel(const bf16* __restrict__ x, int64_t ldx,
                                                     const int* __restrict__ src, int n_src,
                                                     const bf16* __restrict__ w, bf16* __restrict__ y, const int* __restrict__ offs,
                                                     const int* __restrict__ tile_e, const int* __restrict__ tile_m,
                                                     const int* __restrict__ n_tiles, int T, int N, int K, int ldy,
                                                     int ntn, GatedUnit unit) {
  // XCD-contiguous remap of the 1-D grid (bijective for any size)
  const int nwg = gridDim.x, orig = blockIdx.x;
  const int q = nwg / 8, r = nwg % 8, xcd = orig % 8;
  const int id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + orig / 8;
  // grouped raster: consecutive ids sweep GT token tiles before moving to the next N tile, so the ~32 blocks an
  // XCD runs at once cover a GT x (32/GT) rectangle and share both X and W K-slices in its L2
  constexpr int GT = 4;
  const int mt = gridDim.x / ntn;  // token-tile slots (host upper bound)
  const int grp = id / (GT * ntn), rem = id % (GT * ntn);
  const int gsz = min(GT, mt - grp * GT);
  const int t = grp * GT + rem % gsz;
  if (t >= *n_tiles) return;  // block-uniform exit before any barrier
  const int n0 = (rem / gsz) * (GLU ? BN2 / 2 : BN2);
  const int e = tile_e[t];
  const int m0 = tile_m[t];
  const int row0 = min(max(offs[e], 0), T);
  const int rows = min(max(offs[e + 1], row0), T) - row0;

  __shared__ __attribute__((aligned(16))) char smem[2 * 65536];  // [buf][W 32 KB | X 32 KB]
  __shared__ int s_src[GATHER ? BM2 : 1];
  const bf16* wb = w + (int64_t)e * (GLU ? 2 : 1) * N * K + (int64_t)n0 * K;
  const bf16* xb = x + (int64_t)row0 * ldx;
  if constexpr (GATHER) {
    if (threadIdx.x < BM2)
      s_src[threadIdx.x] = min(max(src[row0 + min(m0 + (int)threadIdx.x, rows - 1)], 0), n_src - 1);
    __syncthreads();
  }
  auto stage = [&](int buf, int kt) {
    char* s = smem + buf * 65536;
    const int64_t k0 = (int64_t)kt * BK2;
    const int* sp = s_src;
    // GLU: tile rows 0-127 are gate features, 128-255 the same features of the up half
    const int64_t up = GLU ? (int64_t)(N - 128) * K : 0;
    stage128<8, 256>(s, [=](int rr) { return wb + (int64_t)rr * K + k0 + (GLU && rr >= 128 ? up : 0); });
    stage128<8, 256>(s + 32768, [=](int rr) {
      if constexpr (GATHER) {
        return x + (int64_t)sp[rr] * ldx + k0;
      } else {
        int m = m0 + rr;
        m = m < rows ? m : rows - 1;
        return xb + (int64_t)m * ldx + k0;
      }
    });
  };

  const int wv = threadIdx.x >> 6;
  const int wn = wv & 1, wm = wv >> 1;  // 128 features x 64 tokens per wave
  f32x16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};

  const int KT = K / BK2;
  stage(0, 0);
  __syncthreads();
  for (int kt = 0; kt < KT; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < KT) stage(buf ^ 1, kt + 1);
    const char* Wt = smem + buf * 65536 + wn * (GLU ? 64 : 128) * 128;
    const char* Xt = smem + buf * 65536 + 32768 + wm * 64 * 128;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      bf16x8 a[4], b[2];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = frag128(Wt, GLU ? 32 * (i & 1) + 128 * (i >> 1) : 32 * i, ks);
#pragma unroll
      for (int j = 0; j < 2; ++j) b[j] = frag128(Xt, 32 * j, ks);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }

  const int lane = threadIdx.x & 63;
  const int h = lane >> 5;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int m = m0 + 64 * wm + 32 * j + (lane & 31);
    if (m >= rows) continue;
    bf16* yr = y + (int64_t)(row0 + m) * ldy + n0 + (GLU ? 64 : 128) * wn;
    if constexpr (GLU) {
      const float rw = unit.factor(row0 + m);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          bf16x4 v;
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = (bf16)unit(acc[i][j][4 * g + q], acc[i + 2][j][4 * g + q], rw);
          *reinterpret_cast<bf16x4*>(yr + 32 * i + acc_row(4 * g, h)) = v;
        }
      continue;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        bf16x4 v;
#pragma unroll
        for (int qq = 0; qq < 4; ++qq) v[qq] = (bf16)acc[i][j][4 * g + qq];
        *reinterpret_cast<bf16x4*>(yr + 32 * i + acc_row(4 * g, h)) = v;
      }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Many experts with few rows each (serving). Neither the weights from memory, nor the rows from L2, nor the products alone
// take the time (146 us; 131, 144 and 133 without one of them): what bounds it is how many cache lines a CU can have on the
// way, at about 20 bytes a cycle. So the tile is as large as the rounds over the CUs allow: all rows of an expert up to 256
// (64 NX of them are loaded and multiplied) x WR = 256, 128 or 64 weight rows. LDS is a ring of 20 chunks of 64 rows x 64 k: a
// step multiplies the chunks of 64 k, whose places are refilled one step later, so that R - 2 C to R - C chunks are on their
// way at any time, waited for with a count, one barrier a step. (Twelve or sixteen chunks are level, and so are fragments read
// a step ahead.) Waves: WR / 64 along the weight rows, the others along the tokens. Each XCD takes a contiguous range of the
// real tiles (expert after expert), so that the workgroups of one expert share its rows in one L2.
// 128 weight rows and three stages of 48 KB -> this, gate and up + down, us, weights not in the caches: 64 experts, 6 a token,
// 1024 x 2048, 66 / 700 / 1,600 / 3,000 tokens 125 + 54 / 125 + 63 / 153 + 85 / 247 + 141 -> 98 + 54 / 104 + 62 / 132 + 80 / 234 +
// 141; 64 experts, 4 a token, 2048 x 4096, 66 / 1,500 tokens 366 + 184 / 435 + 231 -> 351 + 183 / 394 + 216; 8 experts, 2 a token,
// 14336 x 4096, 66 / 500 / 1,000 tokens 332 + 165 / 450 + 214 / 760 + 473 -> 326 + 159 / 424 + 221 / 690 + 415; 5632 x 2048, 66 / 500 /
// 1,400 tokens 84 + 55 / 105 + 75 / 217 + 100 -> 78 + 43 / 109 + 60 / 195 + 104.
// ---------------------------------------------------------------------------------------------------------------
constexpr int kChunk = 64 * 128, kRing = 20;
// operand of s_waitcnt: no LDS access and at most n loads on their way
constexpr int flow_wait(int n) { return 0x70 | (n & 15) | n >> 4 << 14; }

template <int NX, int WR, bool GLU, bool NT>
__device__ __forceinline__ void gg_flow_tile(char* smem, const bf16* const (&wp)[WR / 64], const bf16* const (&xp)[4], int KT,
                                             int turn, f32x16 (&acc)[2][WR / 64]) {
  constexpr int CW = WR / 64, C = CW + NX, TG = 8 / CW, NB = (2 * NX + TG - 1) / TG;
  constexpr int R = kRing;
  const int w = threadIdx.x >> 6, wq = w % CW, tg = w / CW;  // wave-uniform
  auto issue = [&](int s, int i, int place) {  // chunk i of step s
    s += turn;
    const int64_t k0 = (int64_t)(s < KT ? s : s - KT) * BK2;
    const bf16* src = i < CW ? wp[i < CW ? i : 0] : xp[i < CW ? 0 : i - CW];
    char* to = smem + place * kChunk + w * 1024;
    if (NT && i < CW) __builtin_amdgcn_global_load_lds((gbl_void*)(src + k0), (lds_void*)to, 16, 0, 2);
    else __builtin_amdgcn_global_load_lds((gbl_void*)(src + k0), (lds_void*)to, 16, 0, 0);
  };
  auto wrap = [](int p) { return p < R ? p : p - R; };
#pragma unroll
  for (int c = 0; c < R - C; ++c)
    if (c < C * KT) issue(c / C, c % C, c);
  int base = 0;  // place of the step's first chunk
  for (int kt = 0; kt < KT; ++kt) {
    // This step's chunks have arrived for every wave, and every wave is done with the last step's: its reads have returned
    // (lgkmcnt), in one statement with the barrier, so that none can be moved between the two. The builtins in front tell
    // the compiler of the wait, which otherwise adds its own for all loads.
    if (C * (kt - 1) + R <= C * KT) {
      __builtin_amdgcn_s_waitcnt(flow_wait(R - 2 * C));
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(R - 2 * C) : "memory");
    } else {
      __builtin_amdgcn_s_waitcnt(flow_wait(0));
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
#pragma unroll
    for (int u = 0; u < C; ++u) {
      constexpr int first = R - C;
      const int s = kt + (first + u) / C;
      if (s < KT) issue(s, (first + u) % C, wrap(base + first + u));
    }
    const char *a0p, *a1p;
    if constexpr (GLU) {
      a0p = smem + wrap(base + (wq >> 1)) * kChunk + (wq & 1) * 4096;
      a1p = CW == 1 ? a0p + 4096 : smem + wrap(base + CW / 2 + (wq >> 1)) * kChunk + (wq & 1) * 4096;
    } else {
      a0p = smem + wrap(base + wq) * kChunk;
      a1p = a0p + 4096;
    }
    // all reads of the step on their way ahead of its products (waited for k by k: 516 us instead of 463 at 8 experts of
    // 14336 x 4096 and 500 tokens)
    constexpr bool some = 2 * NX % TG != 0;  // the last block is not every wave's
    const bool last = !some || tg + TG * (NB - 1) < 2 * NX;  // wave-uniform
    bf16x8 a0[4], a1[4], b[NB][4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      a0[ks] = frag128(a0p, 0, ks);
      a1[ks] = frag128(a1p, 0, ks);
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int blk = min(tg + TG * j, 2 * NX - 1);
      const char* bp = smem + wrap(base + CW + (blk >> 1)) * kChunk + (blk & 1) * 4096;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) b[j][ks] = frag128(bp, 0, ks);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if (some && j == NB - 1 && !last) break;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        acc[0][j] = mfma(a0[ks], b[j][ks], acc[0][j]);
        acc[1][j] = mfma(a1[ks], b[j][ks], acc[1][j]);
      }
    }
    base = wrap(base + C);
  }
}

template <bool GATHER, bool GLU, int WR, bool NT>
__global__ __launch_bounds__(512) void gg_flow_kernel(const bf16* __restrict__ x, int64_t ldx,
                                                      const int* __restrict__ src, int n_src,
                                                      const bf16* __restrict__ w, bf16* __restrict__ y,
                                                      const int* __restrict__ offs, const int* __restrict__ tile_e,
                                                      const int* __restrict__ tile_m, const int* __restrict__ n_tiles,
                                                      int T, int N, int K, int ldy, int ntn, GatedUnit unit, int apart) {
  constexpr int CW = WR / 64, TG = 8 / CW;
  __shared__ __attribute__((aligned(1024))) char smem[kRing * kChunk];
  const int nwg = *n_tiles * ntn, orig = blockIdx.x;
  if (orig >= nwg) return;  // block-uniform exit before any barrier
  const int q = nwg / 8, r = nwg % 8, xcd = orig % 8;
  const int id = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + orig / 8;
  const int t = id / ntn, n0 = (id % ntn) * (GLU ? WR / 2 : WR);
  const int e = tile_e[t], m0 = tile_m[t];
  const int row0 = min(max(offs[e], 0), T);
  const int rows = min(max(offs[e + 1], row0), T) - row0;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  // LDS-DMA sources: lane l fills 16 bytes of row l >> 3 of a group of 8, the piece that off128 keeps there
  const bf16* wp[CW];
  const bf16* xp[4];
  const bf16* wb = w + (int64_t)e * (GLU ? 2 : 1) * N * K + (int64_t)n0 * K;
#pragma unroll
  for (int i = 0; i < CW; ++i) {
    const int row = 64 * i + 8 * wv + (lane >> 3);
    wp[i] = wb + ((int64_t)row + (GLU && row >= WR / 2 ? N - WR / 2 : 0)) * K + 8 * ((lane & 7) ^ ((row >> 1) & 7));
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 64 * i + 8 * wv + (lane >> 3), m = min(m0 + row, rows - 1);
    int64_t at = row0 + m;
    if constexpr (GATHER) at = min(max(src[row0 + m], 0), n_src - 1);
    xp[i] = x + at * ldx + 8 * ((lane & 7) ^ ((row >> 1) & 7));
  }
  f32x16 acc[2][CW];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < CW; ++j) acc[i][j] = f32x16{};
  const int nx = (min(rows - m0, BM2) + 63) / 64, KT = K / BK2;
  const int turn = apart ? (int)__umulhi(blockIdx.x * 2654435769u, (unsigned)KT) : 0;
  if (nx <= 1) gg_flow_tile<1, WR, GLU, NT>(smem, wp, xp, KT, turn, acc);
  else if (nx == 2) gg_flow_tile<2, WR, GLU, NT>(smem, wp, xp, KT, turn, acc);
  else if (nx == 3) gg_flow_tile<3, WR, GLU, NT>(smem, wp, xp, KT, turn, acc);
  else gg_flow_tile<4, WR, GLU, NT>(smem, wp, xp, KT, turn, acc);

  // lane = token, registers 4g .. 4g + 3 = 4 consecutive output features
  const int h = lane >> 5, p = wv % CW, tg = wv / CW;
#pragma unroll
  for (int j = 0; j < CW; ++j) {
    const int m = m0 + 32 * (tg + TG * j) + (lane & 31);
    if (m >= rows) continue;
    bf16* yr = y + (int64_t)(row0 + m) * ldy + n0 + (GLU ? 32 : 64) * p;
    const float rw = GLU ? unit.factor(row0 + m) : 1.f;
#pragma unroll
    for (int i = 0; i < (GLU ? 1 : 2); ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        bf16x4 v;
#pragma unroll
        for (int qq = 0; qq < 4; ++qq)
          v[qq] = GLU ? (bf16)unit(acc[0][j][4 * g + qq], acc[1][j][4 * g + qq], rw) : (bf16)acc[i][j][4 * g + qq];
        *reinterpret_cast<bf16x4*>(yr + 32 * i + acc_row(4 * g, h)) = v;
      }
  }
}

}  // namespace

// Upper bound of the tile count for T rows over E experts (host-side grid size / scratch sizing).
HDS_EXPORT int hds_grouped_gemm_max_tiles(int T, int E) { return (T + BM - 1) / BM + E; }

// Y [T, ldy>=N] = per-expert X . W[e]^T.  x [T, K], w [E, N, K], offs [E+1] (device, int32),
// work = int32 scratch of 2*hds_grouped_gemm_max_tiles(T, E) + 1 elements. Requires N % 128 == 0, K % 128 == 0.
// variant: 0 = auto (256^2 tiles when N % 256 == 0 and the average expert has >= 256 rows), 1 = 128^2, 2 = 256^2.
HDS_EXPORT int hds_grouped_gemm(const void* x, const void* w, void* y, const int* offs, int* work, int T, int N, int K,
                                int E, int ldy, int variant, hipStream_t st) {
  if (T <= 0 || E <= 0) return 0;
  if (N % BN || K % BK || ldy < N || ldy % 8) return hipErrorInvalidValue;
  bool big = variant == 2 || (variant == 0 && N % BN2 == 0 && T >= BM2 * E);
  if (big && N % BN2) return hipErrorInvalidValue;
  const int cap = hds_grouped_gemm_max_tiles(T, E);
  int* tile_e = work;
  int* tile_m = work + cap;
  int* n_tiles = work + 2 * cap;
  if (big) {
    const int max_tiles = (T + BM2 - 1) / BM2 + E;  // <= cap
    const int ntn = N / BN2;
    hipLaunchKernelGGL(gg_plan_kernel<BM2>, dim3(1), dim3(64), 0, st, offs, E, T, tile_e, tile_m, n_tiles, max_tiles);
    hipLaunchKernelGGL((gg_big_kernel<false, false>), dim3(ntn * max_tiles), dim3(512), 0, st, (const bf16*)x, K,
                       (const int*)nullptr, 0, (const bf16*)w, (bf16*)y, offs, tile_e, tile_m, n_tiles, T, N, K, ldy, ntn,
                       GatedUnit{});
  } else {
    hipLaunchKernelGGL(gg_plan_kernel<BM>, dim3(1), dim3(64), 0, st, offs, E, T, tile_e, tile_m, n_tiles, cap);
    hipLaunchKernelGGL(gg_kernel, dim3(N / BN, cap), dim3(256), 0, st, (const bf16*)x, (const bf16*)w, (bf16*)y, offs, tile_e,
                       tile_m, n_tiles, T, N, K, ldy);
  }
  return hipGetLastError();
}

// Rows of a tile of hds_experts_gemm's tile list
HDS_EXPORT int hds_experts_gemm_tile() { return BM2; }

// gg_flow_kernel's weight rows a tile, and whether its workgroups' walks along K begin apart
struct FlowTile {
  int rows, apart;
};
static FlowTile flow_tile(int T, int N, int K, int E, int glu) {
  // The tile of weight rows with which the rounds over the CUs take least; a round of 64, 128 and 256 weight rows
  // takes about 3, 4 and 6 parts (one round of [2048, 5632]: 41.5 / 44.7 / 57 us at 66 tokens, 60 / 77 / 118 at 500), the last 7
  // where an expert has few or very many rows (16 experts, 4 a token, 6400 x 4096, 66 tokens: 322 us with 256, 308 with 128; one
  // round of [3072, 8192], 1,000 tokens 238 / 147). Experts are taken to be alike within 20 rows: near 256 only some have a
  // second tile (6400 x 4096, 1,000 tokens, down: 386 / 353). One that has it costs 64 weight rows, which fill the chip
  // without room, a whole round (8 experts, 2 a token, 5632 x 2048, 900 tokens, down: 73 us without one, 128 with; 128 weight rows
  // 91 and 92).
  const int cols_of = glu ? 2 : 1, avg = (int)(((int64_t)T + E - 1) / E);
  int part = 40;  // tiles of an expert, in 40ths
  for (int m = BM2; m < avg + 20; m += BM2) part += std::min(40, avg + 20 - m);
  const int64_t tiles = (int64_t)std::min(E, T) * part / 40;
  int wr = 64;
  int64_t least = 0;
  for (int r = 64; r <= 256; r *= 2) {
    const int64_t groups = (tiles + (r == 64 && avg > 216)) * (N / (r / cols_of));
    const int64_t cost = (groups + 255) / 256 * (r == 256 && (avg <= 64 || avg > 192) ? 7 : r / 64 + 2);
    if (N % (r / cols_of) == 0 && (r == 64 || cost < least)) {
      wr = r;
      least = cost;
    }
  }
  // Weight rows a multiple of 4 KB apart lie alike in the memory's channels, and workgroups that walk them side by side
  // meet in the same ones: there each begins its walk along K somewhere else. It helps single rounds, whose workgroups stay in
  // step ([4096, 14336], 66 tokens 184 -> 161 us, [4096, 4096] of 16 experts 121 -> 91, 1,000 tokens 136 -> 120, gate and up
  // of 4 experts, 8192 x 4096 130 -> 103), and gate and up rows of an odd number of 4 KB, which are two such walks a workgroup (1024
  // x 2048, 66 tokens 123 -> 96, 1,600 147 -> 135). Several rounds or many rows share in L2 what it takes apart: there only
  // down rows of few tokens ([4096, 2048] of 64 experts, 200 tokens 193 -> 186; of 32, K = 4096, 300 tokens 196 -> 186) and gate
  // and up in 128 weight rows (14336 x 4096, 66 tokens 328 -> 323) gain, others lose ([28672, 4096] 351 -> 386, 1024 x 2048, 3,000 tokens 244
  // -> 275, [4096, 8192], 1,000 tokens 219 -> 236).
  const int64_t rounds = (tiles * (N / (wr / cols_of)) + 255) / 256;
  const bool one = rounds == 1 && avg <= (K % 8192 ? 192 : 96);
  const bool more = glu ? (K / 2048 % 2 && avg <= 192) || (wr == 128 && avg <= 64) : avg <= 64;
  return {wr, K % 2048 == 0 && (one || more)};
}
// the same as one number, rows + apart
HDS_EXPORT int hds_experts_gemm_rows(int T, int N, int K, int E, int glu) {
  if (T <= 0 || E <= 0) return 0;
  const FlowTile t = flow_tile(T, N, K, E, glu);
  return t.rows + t.apart;
}

// Grouped product of sorted rows with a ready tile list (hds_experts_gemm_tile rows a tile; at most
// max_tiles entries, the number on the device). src: row of x [n_src, ldx] for every sorted row, or null: x is sorted.
// glu: w [E, 2N, K] is gate rows then up rows and y = silu(gate) * up, or the clamped unit with its limit (act 5); weight [T]
// or null multiplies the sorted rows' products in front of it. T: upper bound of the rows. K % 128 == 0; N a
// multiple of 128, with glu of 64.
HDS_EXPORT int hds_experts_gemm(const void* x, int64_t ldx, const int* src, int n_src, const void* w, void* y, int ldy,
                                const int* offs, const int* tile_e, const int* tile_m, const int* n_tiles,
                                int max_tiles, int T, int N, int K, int E, int glu, int act, float limit,
                                const float* weight, hipStream_t st) {
  if (T <= 0 || E <= 0) return 0;
  const GatedUnit unit{weight, act == 5, limit};
  const int big_cols = BN2 / (glu ? 2 : 1);
  // 256 x 256 tiles, which read the rows half as often and the weights once per 256 of them, from 512 rows an expert on: 8
  // experts, 2 a token, 14336 x 4096: 1,500 tokens 1,774 us against 1,534 here, 2,000 2,063 / 2,054, 2,700 2,390 / 2,488; 64
  // experts, 6 a token, 1024 x 2048: 3,000 540 / 427, 6,000 786 / 733, 12,000 1,262 / 1,315.
  const bool big = N % big_cols == 0 && T >= 2 * BM2 * E;
  // otherwise gg_flow_kernel's tiles
  const FlowTile flow = flow_tile(T, N, K, E, glu);
  const int wr = flow.rows, apart = flow.apart;
  const int cols = big ? big_cols : wr / (glu ? 2 : 1);
  if (N % cols || K % BK || ldx < K || ldx % 8 || ldy < N || ldy % 8 || max_tiles < 1 || max_tiles > 65535 ||
      (src != nullptr && n_src < 1) || (act != 0 && act != 5) || (int64_t)(N / cols) * max_tiles > INT32_MAX)
    return hipErrorInvalidValue;
  auto run = [&](auto kernel, auto... more) {
    hipLaunchKernelGGL(kernel, dim3(N / cols * max_tiles), dim3(512), 0, st, (const bf16*)x, ldx, src, n_src, (const bf16*)w,
                       (bf16*)y, offs, tile_e, tile_m, n_tiles, T, N, K, ldy, N / cols, unit, more...);
  };
  // Weights that one tile of rows reads go past the caches: 66 tokens, gate and up + down, 64 experts of 1024 x 2048
  // 98.5 + 53.8 -> 87 + 46 us, 8 of 14336 x 4096 325 + 160 -> 297 + 140, 16 of 4096 x 4096 199 + 92 -> 180 + 80; 1,600 tokens of
  // the first 131 + 80 -> 128 + 74. Tiles of one expert find them in L2 or the memory-side cache (past it 3,000 tokens of the first,
  // gate and up 235 / 252, 1,400 of 8 of 5632 x 2048 191 / 202), unless an expert's are too many (2,090 choices of 8 of
  // 14336 x 4096, 117 and 235 MB, a layer 1,470 -> 1,333).
  const bool once = T <= BM2 * E || (int64_t)(glu ? 2 : 1) * N * K >= 1 << 25;
#define HDS_FLOW(GA, GL, NT)                                               \
  do {                                                                     \
    if (wr == 256) run(gg_flow_kernel<GA, GL, 256, NT>, apart);            \
    else if (wr == 128) run(gg_flow_kernel<GA, GL, 128, NT>, apart);       \
    else run(gg_flow_kernel<GA, GL, 64, NT>, apart);                       \
  } while (0)
#define HDS_EG(GA, GL)                                                     \
  do {                                                                     \
    if (big) run(gg_big_kernel<GA, GL>);                                   \
    else if (once) HDS_FLOW(GA, GL, true);                                 \
    else HDS_FLOW(GA, GL, false);                                          \
  } while (0)
  if (src != nullptr) {
    if (glu) HDS_EG(true, true); else HDS_EG(true, false);
  } else {
    if (glu) HDS_EG(false, true); else HDS_EG(false, false);
  }
#undef HDS_EG
#undef HDS_FLOW
  return hipGetLastError();
}
