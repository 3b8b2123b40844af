// Mixed-input GEMM on the gfx950 matrix cores: C[M, N] = A[M, K] (bf16) x dequant(W)[N, K]^T for weight-only
// quantized W (symmetric group INT8, INT4, or FP6 e3m2 / e2m3 with fp32 group scales along k), bf16 out.
//
// Reference parity: the CUTLASS mixed-input GEMM (inference/v2 mixed_gemm) and the
// FP6-LLM tensor-core kernel (N12 / K29, inference/v2/kernels/core_ops/cuda_linear). Those decode packed weights
// in the mainloop so the weight stream stays at 8 / 6 / 4 bits; this kernel does the same on MFMA.
//
// Regime: 8 < M <= a few hundred rows (batched decode, chunked prefill) where a bf16 GEMM is bound by the 16-bit
// weight stream, and groups or rows that linear_packed.hip does not take (it is 1.2 to 3 times as fast). Decode-sized M (<= 8)
// runs the GEMVs (quant.hip / fpq.hip); prefill-sized M dequantizes once and runs hipBLASLt (compute-bound there, so the weight
// bytes no longer matter).
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
#include "packed_codes.h"
#include "row_norm.h"

namespace {
using namespace hds;

__device__ __forceinline__ f32x16 mma(const bf16x8& a, const bf16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int acc_row(int r, int h) { return (r & 3) + 8 * (r >> 2) + 4 * h; }

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
// for 32 of them, int8 and int4 in one and a half and two a code (int4, [11264, 2048] gated, 2 rows: 8.0 us with the offset
// of unsigned nibbles subtracted, 7.1 without). Measured at 8 rows, [28672, 4096] / [4096, 14336]: fp6 38 / 22 us (92 / 46 MB;
// the GEMV that decodes and multiplies on the VALU 112 / 77), int8 39 / 20 (121 / 61 MB; the tile kernel above 45 / 28), int4
// 29 / 16 (41 / 29). What is left to it are the sizes that the two kernels below do not gain on.
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

struct WmixOut {
  const bf16* bias;
  bf16* C;  // [M, N]
  int M, N, act;
  RowScale scale;  // A's rows are still to be scaled (row_norm.h); M <= 16
  RowNorm norm;    // what becomes of the sums is a stream to be scaled; M <= 16, N % 16 == 0, no gated unit, no bias
};

// what a tile's norm reads beside its sums
struct NormIn {
  bf16x4 res, gamma;
  __device__ __forceinline__ void load(const WmixOut& o, int tile, int row, int g) {
    const int n = tile * 16 + 4 * g;
    if (o.norm.res == nullptr || n >= o.N) return;  // (with two tiles a workgroup the last may not be there)
    res = *reinterpret_cast<const bf16x4*>(o.norm.res + (int64_t)min(row, o.M - 1) * o.N + n);
    gamma = *reinterpret_cast<const bf16x4*>(o.norm.gamma + n);
  }
};

// a tile's sums: lane = A row r | 16 g, weight rows 4 g .. 4 g + 3
template <bool GLU>
__device__ __forceinline__ void wmix_store(f32x4 s, int tile, int row, int g, int lane, const WmixOut& o, const NormIn& in) {
  if constexpr (GLU) {  // lanes of the upper half hold the up rows of those 32 below
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = tile * 8 + 4 * (g & 1) + i;
      const float up = __shfl_down(s[i], 32, 64);
      if (lane < 32 && row < o.M && n < o.N)
        o.C[(int64_t)row * o.N + n] = (bf16)(wmix_act((float)(bf16)s[i], o.act) * (float)(bf16)up);
    }
  } else if (o.norm.res != nullptr) {
    if (tile * 16 < o.N)  // (whole tiles)
      store_normed(o.norm, o.C, (int64_t)row * o.N + tile * 16 + 4 * g, s, in.res, in.gamma, tile, lane, row < o.M);
  } else if (row < o.M) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = tile * 16 + 4 * g + i;
      if (n < o.N) o.C[(int64_t)row * o.N + n] = (bf16)(s[i] + (o.bias ? (float)o.bias[n] : 0.f));
    }
  }
}

// MW: waves a SIMD that the registers have to leave room for
template <int FMT, int E, int NT, int MT, int NW, int MW, bool GLU>
__global__ __launch_bounds__(64 * NW, MW) void wmix_skinny_kernel(const bf16* __restrict__ A,
                                                                  const uint8_t* __restrict__ W,
                                                                  const float* __restrict__ scales, WmixOut out,
                                                                  int K, int G) {
  __shared__ f32x4 red[NW - 1][NT][MT][64];
  __shared__ __attribute__((aligned(16))) float rows[NW * 16];
  const int M = out.M, N = out.N;
  RowSums<64 * NW> sums;
  if (out.scale.ssq != nullptr) sums.load(out.scale);
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
          for (int i = 0; i < 4; ++i) acc[t][m][i] += s[i] * (kUnit<FMT> * sc[t][i][c]);
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
  if (out.scale.ssq != nullptr) sums.add(out.scale, rows);
  __syncthreads();
  if (wid > 0) return;
  const float rstd = out.scale.ssq != nullptr ? RowSums<64 * NW>::rstd(out.scale, rows, r) : 1.f;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
      for (int v = 0; v < NW - 1; ++v) acc[t][m] += red[v][t][m][lane];
      NormIn in{};
      if constexpr (!GLU) in.load(out, tile0 + t, 16 * m + r, g);
      wmix_store<GLU>(acc[t][m] * rstd, tile0 + t, 16 * m + r, g, lane, out, in);
    }
}

// With whole cache lines: a load above asks for 8 to 16 bytes a lane of 16 weight rows, and for 16-byte pieces of A. Here
// a wave loads its run of 512 k of 16 rows in 16-byte pieces side by side, which pass through its piece of LDS into the
// operand's layout (rows 16 bytes apart beyond their length: pieces of 16 rows lie in different banks).
template <int FMT>
struct Lines {
  static constexpr int RB = FMT == kFp6 ? 384 : FMT == kInt8 ? 512 : 256;  // bytes of a run of a row
  static constexpr int PR = RB / 16, NL = PR / 4;                          // its pieces; loads of a lane
  static constexpr int ST = RB + 16, WB = 16 * ST;
  static __device__ __forceinline__ u32x4 piece(const uint8_t* p) {
    typedef u32x4 __attribute__((aligned(8))) v4;
    return __builtin_nontemporal_load(reinterpret_cast<const v4*>(p));
  }
  static __device__ __forceinline__ int place(int x) { return x / PR * ST + 16 * (x % PR); }
  // k = 128 c + 32 g .. + 31 of row r
  static __device__ __forceinline__ WRaw<FMT> raw(const char* wl, int r, int g, int c) {
    const char* q = wl + r * ST + (RB / 4) * c + (RB / 16) * g;
    WRaw<FMT> v;
    if constexpr (FMT == kInt8) {
      v.a = *reinterpret_cast<const uint4*>(q);
      v.b = *reinterpret_cast<const uint4*>(q + 16);
    } else if constexpr (FMT == kInt4) {
      v.a = *reinterpret_cast<const uint4*>(q);
    } else {
      v.a = *reinterpret_cast<const uint2*>(q);
      v.b = *reinterpret_cast<const uint2*>(q + 8);
      v.c = *reinterpret_cast<const uint2*>(q + 16);
    }
    return v;
  }
};

// a row's scales of the four chunks of a run
__device__ __forceinline__ f32x4 run_scales(const float* s, int run, int K, int G, int groups) {
  if (G == 128 && groups % 4 == 0) return *reinterpret_cast<const f32x4*>(s + 4 * run);
  f32x4 v;
#pragma unroll
  for (int c = 0; c < 4; ++c) v[c] = s[min(512 * run + 128 * c, K - 128) / G];
  return v;
}

// Up to MR (8 or 16) rows: A in the same way, 1 KB of each row a run; the next run's loads are on their way meanwhile.
template <int FMT, int E, int MR, int NW, bool GLU>
__global__ __launch_bounds__(64 * NW) void wmix_lines_kernel(const bf16* __restrict__ A, const uint8_t* __restrict__ W,
                                                             const float* __restrict__ scales, WmixOut out, int K, int G) {
  using L = Lines<FMT>;
  __shared__ __attribute__((aligned(16))) char buf[NW][L::WB + 1024 * MR];
  __shared__ __attribute__((aligned(16))) float rows[NW * 16];
  const int M = out.M, N = out.N;
  RowSums<64 * NW> sums;
  if (out.scale.ssq != nullptr) sums.load(out.scale);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, r = lane & 15, g = lane >> 4, groups = K / G;
  NormIn in{};
  if constexpr (!GLU)
    if (wid == 0) in.load(out, blockIdx.x, r, g);
  const int row_bytes = K / 512 * L::RB + K % 512 * L::RB / 512, runs = (K + 511) / 512;
  char *wl = buf[wid], *al = wl + L::WB;
  const uint8_t* wp[L::NL];
#pragma unroll
  for (int i = 0; i < L::NL; ++i) wp[i] = W + (int64_t)wmix_row<GLU>(blockIdx.x, (64 * i + lane) / L::PR, N) * row_bytes;
  const float* sp[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) sp[i] = scales + (int64_t)wmix_row<GLU>(blockIdx.x, 4 * g + i, N) * groups;
  u32x4 wr[L::NL], ar[MR];
  f32x4 sn[4];
  auto load = [&](int run) {
#pragma unroll
    for (int i = 0; i < L::NL; ++i)  // (past the row's end: its last piece, unused)
      wr[i] = L::piece(wp[i] + min(run * L::RB + 16 * ((64 * i + lane) % L::PR), row_bytes - 16));
    const int k = min(512 * run + 8 * lane, K - 8);
#pragma unroll
    for (int m = 0; m < MR; ++m)
      if (m < M) ar[m] = *reinterpret_cast<const u32x4*>(A + (int64_t)m * K + k);
#pragma unroll
    for (int i = 0; i < 4; ++i) sn[i] = run_scales(sp[i], run, K, G, groups);
  };
  f32x4 acc{};
  if (wid < runs) load(wid);
  for (int run = wid; run < runs; run += NW) {
#pragma unroll
    for (int i = 0; i < L::NL; ++i) *reinterpret_cast<u32x4*>(wl + L::place(64 * i + lane)) = wr[i];
#pragma unroll
    for (int m = 0; m < MR; ++m)
      if (m < M) *reinterpret_cast<u32x4*>(al + 1024 * m + 16 * (lane ^ m)) = ar[m];
    f32x4 sc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) sc[i] = sn[i];
    if (run + NW < runs) load(run + NW);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (512 * run + 128 * c >= K) break;  // wave-uniform
      bf16x8 x[4], f[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        x[j] = *reinterpret_cast<const bf16x8*>(al + 1024 * (r & (MR - 1)) + 16 * ((16 * c + 4 * g + j) ^ (r & (MR - 1))));
      codes<FMT, E>(L::raw(wl, r, g, c), f);
      f32x4 s{};
#pragma unroll
      for (int j = 0; j < 4; ++j) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[j], x[j], s, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] += s[i] * (kUnit<FMT> * sc[i][c]);
    }
  }
  reinterpret_cast<f32x4*>(wl)[lane] = acc;
  if (out.scale.ssq != nullptr) sums.add(out.scale, rows);
  __syncthreads();
  if (wid > 0) return;
#pragma unroll
  for (int v = 1; v < NW; ++v) acc += reinterpret_cast<const f32x4*>(buf[v])[lane];
  if (out.scale.ssq != nullptr) acc *= RowSums<64 * NW>::rstd(out.scale, rows, r);
  wmix_store<GLU>(acc, blockIdx.x, r, g, lane, out, in);
}

// Many weight rows of up to 4,096 k: workgroups that stay on their CU. Wave w of RW holds run w of A in registers, in the
// operands' layout, and walks over the workgroup's tiles; it loads whole lines as above, a tile ahead.
constexpr int kResWaves = 8;

template <int FMT, int E, int RW, bool GLU>
__global__ __launch_bounds__(64 * kResWaves, 2) void wmix_resident_kernel(const bf16* __restrict__ A,
                                                                          const uint8_t* __restrict__ W,
                                                                          const float* __restrict__ scales, WmixOut out, int K,
                                                                          int G, int tiles) {
  constexpr int TG = kResWaves / RW;
  const int M = out.M, N = out.N;
  using L = Lines<FMT>;
  __shared__ __attribute__((aligned(16))) char buf[kResWaves][L::WB];
  __shared__ f32x4 red[2][4][kResWaves][64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, r = lane & 15, g = lane >> 4, groups = K / G;
  const int row_bytes = K / 512 * L::RB + K % 512 * L::RB / 512;
  const int tg = wid / RW, w = wid % RW, t0 = blockIdx.x * TG + tg, dt = gridDim.x * TG;
  const int rounds = (tiles - (int)blockIdx.x * TG + dt - 1) / dt;  // the same for all waves: every round has one barrier
  const bool on = 512 * w < K;
  const int wr = on ? w : 0;
  char* wl = buf[wid];
  struct Run {
    u32x4 wr[L::NL];
    f32x4 sc[4];
  } ahead;
  // Unconditional: past the end a tile that has just been read. Behind a branch the compiler, which counts loads that are
  // on their way, would have every run wait for the one after it
  auto load = [&](int t, Run& n) {
    t = min(t, tiles - 1);
#pragma unroll
    for (int i = 0; i < L::NL; ++i) {
      const int x = 64 * i + lane;  // (past the row's end: its last piece, unused)
      n.wr[i] = L::piece(W + (int64_t)wmix_row<GLU>(t, x / L::PR, N) * row_bytes +
                         min(wr * L::RB + 16 * (x % L::PR), row_bytes - 16));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      n.sc[i] = run_scales(scales + (int64_t)wmix_row<GLU>(t, 4 * g + i, N) * groups, wr, K, G, groups);
  };
  RowSums<64 * kResWaves> sums;
  if (out.scale.ssq != nullptr) sums.load(out.scale);
  load(t0, ahead);
  float rstd = 1.f;
  if (out.scale.ssq != nullptr) {  // (before the tiles: what its loads were ahead of is still on its way)
    float* rows = reinterpret_cast<float*>(red[1]);
    sums.add(out.scale, rows);
    __syncthreads();
    rstd = RowSums<64 * kResWaves>::rstd(out.scale, rows, r);
  }
  bf16x8 x[4][4];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      x[c][j] = *reinterpret_cast<const bf16x8*>(A + (int64_t)min(r, M - 1) * K + min(512 * w + 128 * c, K - 128) + 32 * g + 8 * j);
  auto step = [&](int round, f32x4 (*rb)[64], Run& cur) {
    const int t = t0 + round * dt;
    f32x4 acc{};
#pragma unroll
    for (int i = 0; i < L::NL; ++i) *reinterpret_cast<u32x4*>(wl + L::place(64 * i + lane)) = cur.wr[i];
    f32x4 sc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) sc[i] = cur.sc[i];
    load(t + dt, cur);
    __builtin_amdgcn_sched_barrier(0);
    if (t < tiles && on) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (512 * w + 128 * c >= K) break;  // wave-uniform
        bf16x8 f[4];
        codes<FMT, E>(L::raw(wl, r, g, c), f);
        f32x4 s{};
#pragma unroll
        for (int j = 0; j < 4; ++j) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[j], x[c][j], s, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += s[i] * (kUnit<FMT> * sc[i][c]);
      }
    }
    rb[wid][lane] = acc;
  };
  for (int round = 0; round < rounds; round += 4) {
    auto* rb = red[round >> 2 & 1];
#pragma unroll
    for (int i = 0; i < 4; ++i) step(round + i, rb[i], ahead);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = t0 + (round + i) * dt;
      if (t >= tiles || w != i) continue;
      f32x4 s = rb[i][tg * RW][lane];
#pragma unroll
      for (int v = 1; v < RW; ++v) s += rb[i][tg * RW + v][lane];
      NormIn in{};
      if constexpr (!GLU) in.load(out, t, r, g);
      wmix_store<GLU>(s * rstd, t, r, g, lane, out, in);
    }
  }
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

// Does wmix_resident_kernel take M rows by [N, K] (N: weight rows, gate and up rows together)? From four tiles a CU on: the
// barriers and a last round that is not full cost more than what is saved below (8 rows, fp6 [11264, 2048] gated 10.8 us
// against 10.1, [12288, 4096] 16.3 with A resident in LDS against 15.5 of whole lines). With up to 2,048 k two tiles are at
// work at a time.
HDS_EXPORT int hds_wmix_resident(int M, int N, int K) {
  return M <= 16 && K <= 4096 && (N + 15) / 16 >= (K > 2048 ? 1024 : 2048);
}

// The same product for few rows as a stream of packed weights (wmix_skinny_kernel, wmix_lines_kernel,
// wmix_resident_kernel): 1 <= M <= 16, fp6 up to 32. K and G multiples of 128, A 16-byte aligned. glu: 0, or 1 + activation code (0 silu, 1 gelu_tanh, 2 relu) for
// W = [gate; up] of 2 N rows (M <= 16, no bias).
static int wmix_skinny(const void* A, const void* W, const float* scales, const WmixOut& o, int K, int G, int fmt, int ebits,
                       int glu, hipStream_t st) {
  const int M = o.M, N = o.N;
  const bf16* bias = o.bias;
  if (M < 1 || M > (fmt == 2 && !glu ? 32 : 16) || N < 1 || K < 128 || K % 128 || G < 128 || G % 128 || K % G || glu < 0 ||
      glu > 3 || (glu && bias) || (glu && N > (1 << 29)))
    return hipErrorInvalidValue;
  const int tiles = (N + (glu ? 7 : 15)) / (glu ? 8 : 16);
  auto launch = [&](auto kern, int nt, int waves) {
    hipLaunchKernelGGL(kern, dim3((tiles + nt - 1) / nt), dim3(64 * waves), 0, st, (const bf16*)A, (const uint8_t*)W,
                       scales, o, K, G);
    return hipGetLastError();
  };
  auto resident = [&](auto kern, int rw) {
    const int wg = (tiles + kResWaves / rw - 1) / (kResWaves / rw);
    hipLaunchKernelGGL(kern, dim3(wg < 256 ? wg : 256), dim3(64 * kResWaves), 0, st, (const bf16*)A, (const uint8_t*)W,
                       scales, o, K, G, tiles);
    return hipGetLastError();
  };
  const bool res = hds_wmix_resident(M, glu ? 2 * N : N, K);
  // Whole lines pay where a wave walks far: 8 rows, fp6 [2048, 2048] 4.8 us against 4.9, [11264, 2048] gated 10.3 / 10.1,
  // [16384, 7168] 26.3 (with A resident in LDS 27.5), [27648, 5120] gated 35.1 (34.6); int8 [4096, 4096] 8.7 / 8.6, [6144, 4096]
  // 12.1 / 12.5, [2048, 5632] 8.2 / 8.7; int4 [4096, 4096] 6.5 / 6.2, [2048, 5632] 7.3 / 7.1, [4096, 14336] 14.3 / 15.7, and with
  // many weight rows from 4,096 k on ([20480, 5120], 4 / 8 rows 25.0 / 27.1, without 26.5 / 29.6; 2 rows [18432, 7168] 28.9 / 26.9).
  const bool lines = K > (fmt == 2 ? 2048 : fmt == 0 ? 4096 : 8192) || (fmt == 1 && K > 4096 && tiles >= 1024 && M > 2);
  // From nine rows on the wider codes lose (int8 [4096, 14336], 16 rows, 24.7 / 23.8) and fp6 gains where a CU's one workgroup
  // is not followed by another or is long ([6144, 4096] 14.8 / 14.6, [5120, 13824] 37.9 / 47.2), but up to 6,144 k of many
  // weight rows the last round has to be full ([22016, 6144] gated 51.1 / 47.3, [20480, 5120] 37.4 / 40.7).
  const int rounds = (tiles + 255) / 256;
  const bool lines16 = lines && (tiles <= 256 || K > 6144 || (K > 4096 && (tiles < 1024 || tiles >= 240 * rounds)));
  // From nine rows on two tiles of weight rows share what is read of A ([28672, 4096], 16 rows: fp6 48 -> 41 us), where
  // enough workgroups remain. int4 with the registers of two waves a SIMD where a third would save no round ([27648, 5120]
  // gated, 12 / 16 rows 41.6 / 44.4 -> 37.2 / 39.5; [22016, 6144] gated 30.9 / 34.6). Short sums on many rows: four waves a
  // workgroup, otherwise eight ([4096, 14336] fp6, 8 rows 27 -> 22 us).
  const bool two = ((tiles + 1) / 2 + 511) / 512 == ((tiles + 1) / 2 + 767) / 768;
#define HDS_WS(F, E, GL)                                                                                            \
  do {                                                                                                              \
    if (res && K > 2048) return resident(wmix_resident_kernel<F, E, 8, GL>, 8);                                     \
    if (res) return resident(wmix_resident_kernel<F, E, 4, GL>, 4);                                                 \
    if (lines && M <= 8 && tiles > 256) return launch(wmix_lines_kernel<F, E, 8, 4, GL>, 1, 4);                     \
    if (lines && M <= 8) return launch(wmix_lines_kernel<F, E, 8, 8, GL>, 1, 8);                                    \
    if constexpr (F == kFp6)                                                                                        \
      if (lines16 && M <= 16) return launch(wmix_lines_kernel<F, E, 16, 6, GL>, 1, 6);                              \
    if constexpr (F == kInt4)                                                                                       \
      if (M > 8 && tiles >= 2 * 512 && two) return launch(wmix_skinny_kernel<F, E, 2, 1, 4, 2, GL>, 2, 4);          \
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

HDS_EXPORT int hds_wmix_skinny(const void* A, const void* W, const float* scales, const void* bias, void* C, int M, int N,
                               int K, int G, int fmt, int ebits, int glu, hipStream_t st) {
  return wmix_skinny(A, W, scales, WmixOut{(const bf16*)bias, (bf16*)C, M, N, glu - 1, {}, {}}, K, G, fmt, ebits, glu, st);
}

// The same of up to 16 rows with a norm on either side, as hds_skinny_norm_bf16 (gemv.hip)
HDS_EXPORT int hds_wmix_norm(const void* A, const void* W, const float* scales, void* C, const float* ssq, float eps,
                             const void* res, const void* gamma, void* r, float* ssq_out, int M, int N, int K, int G, int fmt,
                             int ebits, int glu, hipStream_t st) {
  if (M > 16 || (ssq == nullptr) == (res == nullptr) || (res != nullptr && (glu || N % 16 || !gamma || !r || !ssq_out)))
    return hipErrorInvalidValue;
  return wmix_skinny(A, W, scales, WmixOut{nullptr, (bf16*)C, M, N, glu - 1, {ssq, K / 16, eps},
                                           {(const bf16*)res, (const bf16*)gamma, (bf16*)r, ssq_out}}, K, G, fmt, ebits, glu, st);
}
