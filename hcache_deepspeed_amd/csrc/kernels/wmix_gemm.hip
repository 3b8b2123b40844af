// Mixed-input GEMM on the gfx950 matrix cores: C[M, N] = A[M, K] (bf16) x dequant(W)[N, K]^T for weight-only
// quantized W (symmetric group INT8, INT4, or FP6 e3m2 / e2m3 with fp32 group scales along k), bf16 out.
//
// Reference parity: the CUTLASS mixed-input GEMM (inference/v2 mixed_gemm) and the
// FP6-LLM tensor-core kernel (N12 / K29, inference/v2/kernels/core_ops/cuda_linear). Those decode packed weights
// in the mainloop so the weight stream stays at 8 / 6 / 4 bits; this kernel does the same on MFMA.
//
// Regime: 8 < M <= a few hundred rows (batched decode, chunked prefill) where a bf16 GEMM is bound by the 16-bit
// weight stream. Decode-sized M (<= 8) runs the GEMVs (quant.hip / fpq.hip); prefill-sized M dequantizes once and
// runs hipBLASLt (compute-bound there, so the weight bytes no longer matter).
//
// Structure: workgroup = 4 waves = 512 weight rows (wave = 4 fragments of 32 rows, the weight row on the MFMA lane)
// x 32*MB activation rows, over one K split. Per 64-k chunk a lane reads 32 consecutive k of each of its 4 weight
// rows (32 B int8, 16 B int4, 24 B fp6), applies the group scale and converts to bf16x8 B fragments; the
// contraction order inside a chunk is permuted (half h of the lane group takes k = 32h .. 32h + 31, fragment j = 8
// of them) and the A fragments are read with the same permutation, so the sum is unchanged. The A chunk is staged
// once per workgroup in LDS (padded rows, conflict-free ds_read_b128) and every A fragment feeds 4 MFMAs: a first
// version that read A per 32-row wave from L2 moved 2x (M = 16) to 30x (M = 256) more A bytes than weight bytes
// and ran at 0.2-0.8x the bf16 GEMM. The next chunk's weights and A are loaded before the current chunk's MFMAs.
// K splits (grid.z) write fp32 partials reduced by wmix_reduce_kernel.
#include "hds_common.h"

namespace {
using namespace hds;

__device__ __forceinline__ f32x16 mma(const bf16x8& a, const bf16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int acc_row(int r, int h) { return (r & 3) + 8 * (r >> 2) + 4 * h; }

enum WFmt : int { kInt8 = 0, kInt4 = 1, kFp6 = 2 };

template <int FMT> struct WRaw;
template <> struct WRaw<kInt8> { uint4 a, b; };
template <> struct WRaw<kInt4> { uint4 a; };
template <> struct WRaw<kFp6> { uint2 a, b, c; };

// raw bytes of the 32 weights k = ks .. ks + 31 of row n
template <int FMT>
__device__ __forceinline__ WRaw<FMT> load_w(const uint8_t* __restrict__ w, int64_t n, int K, int ks) {
  WRaw<FMT> r;
  if constexpr (FMT == kInt8) {
    const uint4* p = reinterpret_cast<const uint4*>(w + n * K + ks);
    r.a = p[0];
    r.b = p[1];
  } else if constexpr (FMT == kInt4) {
    r.a = *reinterpret_cast<const uint4*>(w + (n * K + ks) / 2);
  } else {
    const uint2* p = reinterpret_cast<const uint2*>(w + (n * K + ks) * 3 / 4);
    r.a = p[0];
    r.b = p[1];
    r.c = p[2];
  }
  return r;
}

// FP6 magnitude (E exponent bits, M mantissa bits, no inf/nan) -> float, without ldexp:
// normal codes become an fp32 bit pattern directly; subnormals (e == 0) are m * 2^(1 - bias - M)
template <int E, int M>
__device__ __forceinline__ float fp6_val(uint32_t c) {
  constexpr int bias = (1 << (E - 1)) - 1;
  const uint32_t e = (c >> M) & ((1u << E) - 1), m = c & ((1u << M) - 1);
  const float nrm = __uint_as_float(((e + 127 - bias) << 23) | (m << (23 - M)));
  const float sub = (float)m * __uint_as_float((uint32_t)(127 + 1 - bias - M) << 23);
  const float v = e ? nrm : sub;
  return (c >> (E + M)) & 1u ? -v : v;
}

// fragment j (weights 8j .. 8j+7 of the lane's 32) scaled by s, as bf16
template <int FMT, int E>
__device__ __forceinline__ bf16x8 frag(const WRaw<FMT>& r, int j, float s) {
  bf16x8 out;
  if constexpr (FMT == kInt8) {
    const uint32_t dw[8] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w};
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int e = 8 * j + t;
      out[t] = (bf16)((float)(int8_t)((dw[e >> 2] >> (8 * (e & 3))) & 0xff) * s);
    }
  } else if constexpr (FMT == kInt4) {
    const uint32_t dw[4] = {r.a.x, r.a.y, r.a.z, r.a.w};
#pragma unroll
    for (int t = 0; t < 8; ++t) out[t] = (bf16)((float)((int)((dw[j] >> (4 * t)) & 0xf) ^ 8) - 8.f) * s;
  } else {
    const uint64_t q[3] = {((uint64_t)r.a.y << 32) | r.a.x, ((uint64_t)r.b.y << 32) | r.b.x,
                           ((uint64_t)r.c.y << 32) | r.c.x};
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int b = 6 * (8 * j + t), wi = b >> 6, o = b & 63;
      uint64_t v = q[wi] >> o;
      if (o > 58) v |= q[wi + 1] << (64 - o);
      out[t] = (bf16)(fp6_val<E, 5 - E>((uint32_t)v & 63u) * s);
    }
  }
  return out;
}

constexpr int kArow = 144;             // LDS bytes per A row of a 64-k chunk (128 + 16 pad: conflict-free b128 reads)

template <int FMT, int MB, int E, int kNF>
__global__ __launch_bounds__(256) void wmix_gemm_kernel(const bf16* __restrict__ A, const uint8_t* __restrict__ W,
                                                        const float* __restrict__ scales,
                                                        const bf16* __restrict__ bias, bf16* __restrict__ C,
                                                        float* __restrict__ part, int M, int N, int K, int G,
                                                        int kc) {
  constexpr int BM = 32 * MB;
  constexpr int kBN = 4 * 32 * kNF;  // weight rows per workgroup
  __shared__ __attribute__((aligned(16))) char As[2][BM * kArow];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, h = lane >> 5;
  const int nb = blockIdx.x * kBN + 32 * kNF * w + (lane & 31);  // row of fragment f: nb + 32 f
  const int m0 = blockIdx.y * BM;
  const int k_begin = blockIdx.z * kc, k_end = min(K, k_begin + kc);
  int nr[kNF];
#pragma unroll
  for (int f = 0; f < kNF; ++f) nr[f] = min(nb + 32 * f, N - 1);
  // A staging: thread -> (row, 16-B piece) of the chunk, MB rows of 32 apart
  const int ar = tid >> 3, ap = tid & 7;
  const bf16* asrc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) asrc[mb] = A + (int64_t)min(m0 + 32 * mb + ar, M - 1) * K + 8 * ap;

  f32x16 acc[MB][kNF];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int f = 0; f < kNF; ++f) acc[mb][f] = f32x16{};

  WRaw<FMT> wc[kNF], wn[kNF];
  float sc[kNF], sn[kNF];
  auto load_wf = [&](WRaw<FMT> (&wr)[kNF], float (&sr)[kNF], int k0) {
#pragma unroll
    for (int f = 0; f < kNF; ++f) {
      wr[f] = load_w<FMT>(W, nr[f], K, k0 + 32 * h);
      sr[f] = scales[(int64_t)nr[f] * (K / G) + (k0 + 32 * h) / G];
    }
  };
  bf16x8 ag[MB];
  auto load_ag = [&](int k0) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) ag[mb] = *reinterpret_cast<const bf16x8*>(asrc[mb] + k0);
  };
  auto store_ag = [&](int buf) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) *reinterpret_cast<bf16x8*>(&As[buf][(32 * mb + ar) * kArow + 16 * ap]) = ag[mb];
  };

  load_wf(wc, sc, k_begin);
  load_ag(k_begin);
  store_ag(0);
  __syncthreads();
  int buf = 0;
  for (int k0 = k_begin; k0 < k_end; k0 += 64) {
    const bool more = k0 + 64 < k_end;
    if (more) {
      load_wf(wn, sn, k0 + 64);
      load_ag(k0 + 64);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      bf16x8 af[MB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        af[mb] = *reinterpret_cast<const bf16x8*>(&As[buf][(32 * mb + (lane & 31)) * kArow + 64 * h + 16 * j]);
#pragma unroll
      for (int f = 0; f < kNF; ++f) {
        const bf16x8 b = frag<FMT, E>(wc[f], j, sc[f]);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[mb][f] = mma(af[mb], b, acc[mb][f]);
      }
    }
    if (more) {
      store_ag(buf ^ 1);
#pragma unroll
      for (int f = 0; f < kNF; ++f) {
        wc[f] = wn[f];
        sc[f] = sn[f];
      }
    }
    __syncthreads();
    buf ^= 1;
  }
#pragma unroll
  for (int f = 0; f < kNF; ++f) {
    const int n = nb + 32 * f;
    if (n >= N) continue;
    if (part == nullptr) {
      const float bv = bias ? (float)bias[n] : 0.f;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = m0 + 32 * mb + acc_row(r, h);
          if (m < M) C[(int64_t)m * N + n] = (bf16)(acc[mb][f][r] + bv);
        }
    } else {
      float* P = part + (int64_t)blockIdx.z * M * N;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = m0 + 32 * mb + acc_row(r, h);
          if (m < M) P[(int64_t)m * N + n] = acc[mb][f][r];
        }
    }
  }
}

// C = sum_z part[z] (+ bias): 4 outputs per thread
__global__ __launch_bounds__(256) void wmix_reduce_kernel(const float* __restrict__ part,
                                                          const bf16* __restrict__ bias, bf16* __restrict__ C, int M,
                                                          int N, int splits) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const int64_t MN = (int64_t)M * N;
  if (i >= MN) return;
  f32x4 a = *reinterpret_cast<const f32x4*>(part + i);
  for (int z = 1; z < splits; ++z) a += *reinterpret_cast<const f32x4*>(part + z * MN + i);
  const int n = (int)(i % N);
  bf16x4 o;
#pragma unroll
  for (int t = 0; t < 4; ++t) o[t] = (bf16)(a[t] + (bias ? (float)bias[n + t] : 0.f));
  *reinterpret_cast<bf16x4*>(C + i) = o;
}

// ---------------------------------------------------------------------------------------------------------------
// Few rows (decode): a stream of packed weights
// ---------------------------------------------------------------------------------------------------------------
// A workgroup owns 16 NT weight rows, its NW waves take runs of 512 k in turn. In a run a lane holds 32 consecutive k
// of a weight row for each of four chunks of 128 (24 bytes fp6, 32 int8, 16 int4: all loads of the run are in flight
// together), and mfma_f32_16x16x32_bf16 contracts elements 8 j .. 8 j + 7 of the four lane groups with the same k of up
// to 16 MT rows of A. The operand is the weight's CODE, which bf16 holds exactly; the group's scale multiplies the 32-bit
// sum of each group (every chunk lies in one group), so no weight is rounded. fp6 codes become bf16 in one instruction
// for 32 of them. Measured at 8 rows, [28672, 4096] / [4096, 14336]: fp6 38 / 22 us (92 / 46 MB; the GEMV that decodes and
// multiplies on the VALU 112 / 77; 27 us with A resident, below), int8 39 / 20 us (121 / 61 MB; the tile kernel above 45 / 28), int4 29 / 16 us (41 /
// 29). A third of the time at 8 rows goes to reading A again from L2 in every workgroup.
typedef uint32_t u32x6 __attribute__((ext_vector_type(6)));
typedef __bf16 bf16x32 __attribute__((ext_vector_type(32)));

template <int FMT, int E>
__device__ __forceinline__ void codes(const WRaw<FMT>& r, bf16x8 (&f)[4]) {
  if constexpr (FMT == kFp6) {
    const u32x6 q = {r.a.x, r.a.y, r.b.x, r.b.y, r.c.x, r.c.y};
    bf16x32 v;
    if constexpr (E == 3) v = __builtin_amdgcn_cvt_scalef32_pk32_bf16_bf6(q, 1.f);  // "bf6" is e3m2
    else v = __builtin_amdgcn_cvt_scalef32_pk32_bf16_fp6(q, 1.f);
    f[0] = __builtin_shufflevector(v, v, 0, 1, 2, 3, 4, 5, 6, 7);
    f[1] = __builtin_shufflevector(v, v, 8, 9, 10, 11, 12, 13, 14, 15);
    f[2] = __builtin_shufflevector(v, v, 16, 17, 18, 19, 20, 21, 22, 23);
    f[3] = __builtin_shufflevector(v, v, 24, 25, 26, 27, 28, 29, 30, 31);
  } else if constexpr (FMT == kInt8) {
    const uint32_t dw[8] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t u = dw[i] ^ 0x80808080u;  // unsigned bytes, 128 too large
#pragma unroll
      for (int t = 0; t < 4; ++t) f[i >> 1][4 * (i & 1) + t] = (bf16)((float)((u >> (8 * t)) & 0xff) - 128.f);
    }
  } else {
    const uint32_t dw[4] = {r.a.x, r.a.y, r.a.z, r.a.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t lo = (dw[i] & 0x0f0f0f0fu) ^ 0x08080808u, hi = ((dw[i] >> 4) & 0x0f0f0f0fu) ^ 0x08080808u;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        f[i][2 * t] = (bf16)((float)((lo >> (8 * t)) & 0xff) - 8.f);
        f[i][2 * t + 1] = (bf16)((float)((hi >> (8 * t)) & 0xff) - 8.f);
      }
    }
  }
}

// GLU: W is [gate; up] of 2 N rows, a tile of 16 weight rows holds 8 gate rows and their 8 up rows (as many workgroups as
// without), and the result is bf16(act(bf16(gate)) * bf16(up)) [M, N].
template <bool GLU>
__device__ __forceinline__ int wmix_row(int tile, int r, int N) {
  if constexpr (GLU) {
    const int n = min(tile * 8 + (r & 7), N - 1);
    return r < 8 ? n : N + n;
  }
  return min(tile * 16 + r, N - 1);
}

__device__ __forceinline__ float wmix_act(float v, int act) {  // codes of act.hip
  if (act == 2) return fmaxf(v, 0.f);
  if (act == 1) return 0.5f * v * (1.f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
  return v * __builtin_amdgcn_rcpf(1.f + __expf(-v));
}

// a tile's sums: lane = A row r | 16 g, weight rows 4 g .. 4 g + 3
template <bool GLU>
__device__ __forceinline__ void wmix_store(f32x4 s, int tile, int row, int g, int lane, const bf16* bias, bf16* C, int M,
                                           int N, int act) {
  if constexpr (GLU) {  // lanes of the upper half hold the up rows of those 32 below
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = tile * 8 + 4 * (g & 1) + i;
      const float up = __shfl_down(s[i], 32, 64);
      if (lane < 32 && row < M && n < N) C[(int64_t)row * N + n] = (bf16)(wmix_act((float)(bf16)s[i], act) * (float)(bf16)up);
    }
  } else if (row < M) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = tile * 16 + 4 * g + i;
      if (n < N) C[(int64_t)row * N + n] = (bf16)(s[i] + (bias ? (float)bias[n] : 0.f));
    }
  }
}

// MW: waves a SIMD that the registers have to leave room for
template <int FMT, int E, int NT, int MT, int NW, int MW, bool GLU>
__global__ __launch_bounds__(64 * NW, MW) void wmix_skinny_kernel(const bf16* __restrict__ A,
                                                                  const uint8_t* __restrict__ W,
                                                                  const float* __restrict__ scales,
                                                                  const bf16* __restrict__ bias, bf16* __restrict__ C,
                                                                  int M, int N, int K, int G, int act) {
  __shared__ f32x4 red[NW - 1][NT][MT][64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const int tile0 = blockIdx.x * NT, groups = K / G;
  f32x4 acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{};
  const bf16* xp[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) xp[m] = A + (int64_t)min(16 * m + r, M - 1) * K + 32 * g;

  for (int run = wid; run * 512 < K; run += NW) {
    WRaw<FMT> raw[4][NT];
    f32x4 sc[NT][4];  // of the lane's four sums, chunks 0 .. 3
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int k = min(512 * run + 128 * c, K - 128);
#pragma unroll
      for (int t = 0; t < NT; ++t) raw[c][t] = load_w<FMT>(W, wmix_row<GLU>(tile0 + t, r, N), K, k + 32 * g);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float* s = scales + (int64_t)wmix_row<GLU>(tile0 + t, 4 * g + i, N) * groups;
        if (G == 128 && groups % 4 == 0) {
          sc[t][i] = *reinterpret_cast<const f32x4*>(s + 4 * run);
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c) sc[t][i][c] = s[min(512 * run + 128 * c, K - 128) / G];
        }
      }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int k = 512 * run + 128 * c;
      if (k >= K) break;  // wave-uniform
      bf16x8 x[MT][4];
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j) x[m][j] = *reinterpret_cast<const bf16x8*>(xp[m] + k + 8 * j);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        bf16x8 f[4];
        codes<FMT, E>(raw[c][t], f);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          f32x4 s{};
#pragma unroll
          for (int j = 0; j < 4; ++j) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[j], x[m][j], s, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[t][m][i] += s[i] * sc[t][i][c];
        }
      }
    }
  }
  if (wid > 0) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) red[wid - 1][t][m][lane] = acc[t][m];
  }
  __syncthreads();
  if (wid > 0) return;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
      for (int v = 0; v < NW - 1; ++v) acc[t][m] += red[v][t][m][lane];
      wmix_store<GLU>(acc[t][m], tile0 + t, 16 * m + r, g, lane, bias, C, M, N, act);
    }
}

// The same for fp6 and many weight rows, with A resident. At 8 rows A is more bytes of loads than the packed weights (2
// against 0.75 a code), and every workgroup above loads all of it: [28672, 4096] 37.4 us, 2.5 TB/s. Here a workgroup of 16
// waves stays on its CU: A lies in LDS in the order of the products (MP = its rows rounded up to 4, 8 or 16), RW waves
// share a tile's K in runs of 512, and while a tile's sums are reduced the other waves' next runs are on their way. 2 / 8 /
// 16 rows: 30.3 / 37.6 / 40.3 -> 25.2 / 26.6 / 28.9 us (3.5 TB/s). int8 and int4 are bound by turning codes into bf16 and
// gain nothing (8 rows: 38.8 -> 37.8, 27.9 -> 30.2).
constexpr int kResWaves = 16;
constexpr int kResTiles = 1024;

template <int FMT, int E, int RW, bool GLU>
__global__ __launch_bounds__(64 * kResWaves) void wmix_resident_kernel(const bf16* __restrict__ A,
                                                                       const uint8_t* __restrict__ W,
                                                                       const float* __restrict__ scales,
                                                                       const bf16* __restrict__ bias,
                                                                       bf16* __restrict__ C, int M, int N, int K, int G,
                                                                       int act, int tiles, int MP) {
  extern __shared__ __attribute__((aligned(16))) char sm[];  // A: K * MP * 2, sums: [2][waves][64] of 16 bytes
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  constexpr int TG = kResWaves / RW;
  const int tg = wid / RW, w = wid % RW;
  const int runs = (K + 511) / 512, groups = K / G;
  f32x4* red = reinterpret_cast<f32x4*>(sm + (int64_t)K * MP * 2);
  const int t0 = blockIdx.x * TG, dt = gridDim.x * TG;
  const int rounds = (tiles - t0 + dt - 1) / dt;  // the same for all waves: every round has one barrier
  WRaw<FMT> raw[4];
  f32x4 sc[4];
  int lt = t0 + tg, lrun = w;  // the wave's next run to load
  auto load = [&]() {
    if (lt >= tiles || lrun >= runs) return;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      raw[c] = load_w<FMT>(W, wmix_row<GLU>(lt, r, N), K, min(512 * lrun + 128 * c, K - 128) + 32 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* s = scales + (int64_t)wmix_row<GLU>(lt, 4 * g + i, N) * groups;
      if (G == 128 && groups % 4 == 0) {
        sc[i] = *reinterpret_cast<const f32x4*>(s + 4 * lrun);
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) sc[i][c] = s[min(512 * lrun + 128 * c, K - 128) / G];
      }
    }
    lrun += RW;
    if (lrun >= runs) {
      lrun = w;
      lt += dt;
    }
  };
  load();
  // piece p of A: row p % MP, 8 columns of lane group (p / MP) % 4 for product (p / 4 MP) % 4 of 128-chunk p / 16 MP
  for (int i = wid; i < K * MP / 512; i += kResWaves) {
    const int p = 64 * i + lane, k = 128 * (p / (16 * MP)) + 32 * ((p / MP) & 3) + 8 * ((p / (4 * MP)) & 3);
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) void*)(A + (int64_t)min(p % MP, M - 1) * K + k),
        (__attribute__((address_space(3))) void*)(sm + i * 1024), 16, 0, 0);
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  __syncthreads();
  const char* xs = sm + (g * MP + (r & (MP - 1))) * 16;
  for (int round = 0, t = t0 + tg; round < rounds; ++round, t += dt) {
    f32x4 acc{};
    if (t < tiles) {
      for (int run = w; run < runs; run += RW) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          if (512 * run + 128 * c >= K) break;  // wave-uniform
          bf16x8 f[4];
          codes<FMT, E>(raw[c], f);
          f32x4 s{};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const bf16x8 x = *reinterpret_cast<const bf16x8*>(xs + (16 * (4 * run + c) + 4 * j) * MP * 16);
            s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[j], x, s, 0, 0, 0);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[i] += s[i] * sc[i][c];
        }
        load();
      }
    }
    f32x4* rb = red + (round & 1) * kResWaves * 64;
    rb[wid * 64 + lane] = acc;
    __syncthreads();
    if (t < tiles && w == round % RW) {
      f32x4 s = rb[tg * RW * 64 + lane];
#pragma unroll
      for (int v = 1; v < RW; ++v) s += rb[(tg * RW + v) * 64 + lane];
      wmix_store<GLU>(s, t, r, g, lane, bias, C, M, N, act);
    }
  }
}

// rows of A the resident kernel makes room for, and its LDS (0: it does not take the size)
int resident_rows(int M) { return M <= 4 ? 4 : (M <= 8 ? 8 : 16); }
size_t resident_bytes(int M, int K) {
  const size_t b = (size_t)K * resident_rows(M) * 2 + 2 * kResWaves * 1024;
  return M <= 16 && b <= 160 * 1024 ? b : 0;
}

int pick_mb(int M) { return M <= 32 ? 1 : 2; }
// weight fragments per wave: 1 at small M (more workgroups in flight for the weight stream), 4 once the A chunk
// re-reads and the per-fragment MFMA chain matter (measured, profiles/wmix_bench_r2.log)
int pick_nf(int M) { return M <= 64 ? 1 : 4; }

}  // namespace

// number of K splits (grid.z) for a problem; the caller provides an fp32 workspace of splits * M * N when > 1
HDS_EXPORT int hds_wmix_splits(int M, int N, int K) {
  const int mb = pick_mb(M), kBN = 128 * pick_nf(M);
  const int base = ((N + kBN - 1) / kBN) * ((M + 32 * mb - 1) / (32 * mb));
  int splits = (512 + base - 1) / base;
  const int max_splits = K / 256 > 1 ? K / 256 : 1;  // >= 4 chunks of 64 k per split
  if (splits > max_splits) splits = max_splits;
  if (splits > 16) splits = 16;
  if (splits < 1) splits = 1;
  const int kc = ((K / 64 + splits - 1) / splits) * 64;
  return (K + kc - 1) / kc;
}

HDS_EXPORT int hds_wmix_supported(int M, int N, int K, int G) {
  return M > 0 && N % 4 == 0 && K % 64 == 0 && G % 32 == 0 && K % G == 0;
}

// fmt: 0 int8, 1 int4, 2 fp6 (ebits 3 -> e3m2, ebits 2 -> e2m3). A [M, K] bf16 row-major, W packed [N, K], scales
// [N, K / G] fp32, bias [N] bf16 or null, C [M, N] bf16, ws fp32 [splits, M, N] (null when splits == 1)
HDS_EXPORT int hds_wmix_gemm(const void* A, const void* W, const float* scales, const void* bias, void* C, float* ws,
                             int M, int N, int K, int G, int fmt, int ebits, hipStream_t st) {
  if (!hds_wmix_supported(M, N, K, G)) return hipErrorInvalidValue;
  const int splits = hds_wmix_splits(M, N, K);
  if (splits > 1 && ws == nullptr) return hipErrorInvalidValue;
  const int kc = ((K / 64 + splits - 1) / splits) * 64;
  const int mb = pick_mb(M), nf = pick_nf(M), kBN = 128 * nf;
  dim3 grid((N + kBN - 1) / kBN, (M + 32 * mb - 1) / (32 * mb), splits);
  float* part = splits > 1 ? ws : nullptr;
  auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, (const bf16*)A, (const uint8_t*)W, scales, (const bf16*)bias,
                       (bf16*)C, part, M, N, K, G, kc);
  };
#define HDS_WMIX(F, E)                                                 \
  do {                                                                 \
    if (mb == 1 && nf == 1) launch(wmix_gemm_kernel<F, 1, E, 1>);      \
    else if (mb == 1) launch(wmix_gemm_kernel<F, 1, E, 4>);            \
    else if (nf == 1) launch(wmix_gemm_kernel<F, 2, E, 1>);            \
    else launch(wmix_gemm_kernel<F, 2, E, 4>);                         \
  } while (0)
  if (fmt == 0) HDS_WMIX(kInt8, 0);
  else if (fmt == 1) HDS_WMIX(kInt4, 0);
  else if (fmt == 2 && ebits == 3) HDS_WMIX(kFp6, 3);
  else if (fmt == 2 && ebits == 2) HDS_WMIX(kFp6, 2);
  else return hipErrorInvalidValue;
#undef HDS_WMIX
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || splits == 1) return e;
  const int64_t MN = (int64_t)M * N;
  hipLaunchKernelGGL(wmix_reduce_kernel, dim3((unsigned)((MN / 4 + 255) / 256)), dim3(256), 0, st, ws,
                     (const bf16*)bias, (bf16*)C, M, N, splits);
  return hipGetLastError();
}

// The same product for few rows as a stream of packed weights (wmix_skinny_kernel, wmix_resident_kernel): 1 <= M <= 16, fp6
// up to 32. K and G multiples of 128, A 16-byte aligned. glu: 0, or 1 + activation code (0 silu, 1 gelu_tanh, 2 relu) for
// W = [gate; up] of 2 N rows (M <= 16, no bias).
HDS_EXPORT int hds_wmix_skinny(const void* A, const void* W, const float* scales, const void* bias, void* C, int M, int N,
                               int K, int G, int fmt, int ebits, int glu, hipStream_t st) {
  if (M < 1 || M > (fmt == 2 && !glu ? 32 : 16) || N < 1 || K < 128 || K % 128 || G < 128 || G % 128 || K % G || glu < 0 ||
      glu > 3 || (glu && bias) || (glu && N > (1 << 29)))
    return hipErrorInvalidValue;
  const int tiles = (N + (glu ? 7 : 15)) / (glu ? 8 : 16);
  auto launch = [&](auto kern, int nt, int waves) {
    hipLaunchKernelGGL(kern, dim3((tiles + nt - 1) / nt), dim3(64 * waves), 0, st, (const bf16*)A, (const uint8_t*)W,
                       scales, (const bf16*)bias, (bf16*)C, M, N, K, G, glu - 1);
    return hipGetLastError();
  };
  auto resident = [&](auto kern, int rw) {
    const int wg = (tiles + kResWaves / rw - 1) / (kResWaves / rw);
    const size_t lds = resident_bytes(M, K);
    const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(wg < 256 ? wg : 256), dim3(64 * kResWaves), lds, st, (const bf16*)A, (const uint8_t*)W,
                       scales, (const bf16*)bias, (bf16*)C, M, N, K, G, glu - 1, tiles, resident_rows(M));
    return hipGetLastError();
  };
  // A resident from four tiles a CU on, where it fits: [16384, 4096], 8 rows 20.8 -> 16.8 us, [32768, 2048] 21.2 -> 15.8,
  // [27648, 5120] 53 -> 33, [16384, 7168] 37.5 -> 25.6; at [12288, 4096] 2 / 8 / 16 rows 13.8 / 16.2 / 21.0 -> 15.0 / 16.3
  // / 18.5, at [8192, 4096] level: the last round of tiles and the way of A into LDS.
  const bool res = fmt == 2 && resident_bytes(M, K) != 0 && tiles >= kResTiles;
  // From nine rows on two tiles of weight rows share what is read of A ([28672, 4096], 16 rows: fp6 48 -> 41 us), where
  // enough workgroups remain. Short sums on many rows: four waves a workgroup, otherwise eight ([4096, 14336] fp6, 8 rows 27
  // -> 22 us).
#define HDS_WS(F, E, GL)                                                                                            \
  do {                                                                                                              \
    if constexpr (F == kFp6) {                                                                                      \
      if (res && (K + 511) / 512 % 8 == 0) return resident(wmix_resident_kernel<F, E, 8, GL>, 8);                   \
      if (res) return resident(wmix_resident_kernel<F, E, 4, GL>, 4);                                               \
    }                                                                                                               \
    if (M > 8 && M <= 16 && tiles >= 2 * 512) return launch(wmix_skinny_kernel<F, E, 2, 1, 4, 3, GL>, 2, 4);        \
    if (M <= 16 && K <= 4096 && tiles >= 384) return launch(wmix_skinny_kernel<F, E, 1, 1, 4, 1, GL>, 1, 4);        \
    if (M <= 16) return launch(wmix_skinny_kernel<F, E, 1, 1, 8, 1, GL>, 1, 8);                                     \
    if constexpr (F == kFp6 && !GL) return launch(wmix_skinny_kernel<F, E, 1, 2, 8, 1, false>, 1, 8);               \
    return hipErrorInvalidValue;                                                                                    \
  } while (0)
#define HDS_WSG(F, E)          \
  do {                         \
    if (glu) HDS_WS(F, E, true); \
    HDS_WS(F, E, false);       \
  } while (0)
  if (fmt == 0) HDS_WSG(kInt8, 0);
  if (fmt == 1) HDS_WSG(kInt4, 0);
  if (fmt == 2 && ebits == 3) HDS_WSG(kFp6, 3);
  if (fmt == 2 && ebits == 2) HDS_WSG(kFp6, 2);
#undef HDS_WSG
#undef HDS_WS
  return hipErrorInvalidValue;
}
