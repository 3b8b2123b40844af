// Decode-sized bf16 linear: y[M, N] = x[M, K] . W[N, K]^T (+ bias) for M <= 8 token rows.
//
// Capability parity: the reference's inference kernels run decode projections through cuBLAS GEMV-shaped GEMMs
// (csrc/transformer/inference/csrc/pt_binding.cpp qkv_gemm / vector_matmul). At M <= 8 the
// product is a pure weight stream (N * K * 2 bytes); hipBLASLt reaches 6+ TB/s on the wide projections but
// only ~2.7 TB/s on the narrow ones (Llama-3-8B qkv 6144 x 4096: 18.9 us for 50 MB), where a few hundred
// workgroups cannot cover its launch / tail latency (profiles/int_gemv_bench_r1.log).
//
// Structure: a wave owns R consecutive weight rows; each lane streams 16-B chunks (8 bf16) of those rows, two
// k-chunks per iteration so 2R loads are in flight per lane, and contracts them with the matching x chunks
// (x is tiny and L2/L1-resident) by v_dot2_f32_bf16 (4 per chunk per token row). The per-(row, token) partial
// sums are reduced across the wave once at the end. Here and below the weights are loaded past the caches (load_nt), whole
// lines by one instruction: temporal -> not, 1 row [32000, 2048] 23.5 -> 21.7 us, [28672, 4096] 40.4 -> 37.2 (6.3 TB/s), with norm and
// GLU 43.6 -> 39.9; 8 rows [28672, 4096] 45.3 -> 40.5, [4096, 14336] 24.5 -> 22.5; 16 rows 51.8 -> 47.9, 28.1 -> 27.0.
// Weights that the memory-side cache would hold from one step to the next lose by it (all of them under 256 MB: [2048, 5632], 1
// / 4 rows 6.3 / 6.9 -> 6.6 / 9.4 us).
#include "hds_common.h"
#include "row_norm.h"

namespace {
using namespace hds;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float dot8(const bf16x8& a, const bf16x8& b, float c) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const bf16x2 a2 = {a[2 * j], a[2 * j + 1]}, b2 = {b[2 * j], b[2 * j + 1]};
    c = __builtin_amdgcn_fdot2_f32_bf16(a2, b2, c, false);
  }
  return c;
}

__device__ __forceinline__ float gate_f(float v, int act);

// Optional last step of the kernels below (GATHER): y[m, n] = act(y[m, n]) * table[ids[m], n]
struct Gather {
  const bf16* table;  // [vocab, ld]
  int64_t ld;
  const int64_t* ids;
  int vocab, act;
  __device__ __forceinline__ float operator()(float v, int m, int n) const {
    const int64_t id = min(max(ids[m], (int64_t)0), (int64_t)vocab - 1);
    return gate_f((float)(bf16)v, act) * (float)table[id * ld + n];  // (the product rounded, as the separate kernel reads it)
  }
};

template <int MAXM, int R>
__global__ __launch_bounds__(256) void gemv_bf16_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                        const bf16* __restrict__ bias, bf16* __restrict__ y, int M,
                                                        int N, int K, int64_t ldx, int64_t ldy) {
  const int lane = threadIdx.x & 63;
  const int n0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * R;
  if (n0 >= N) return;
  float acc[R][MAXM];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int m = 0; m < MAXM; ++m) acc[r][m] = 0.f;
  const bf16* wr[R];
#pragma unroll
  for (int r = 0; r < R; ++r) wr[r] = w + (int64_t)min(n0 + r, N - 1) * K;  // tail rows re-read row N-1 (unused)
  int k0 = 8 * lane;
  for (; k0 + 512 < K; k0 += 1024) {
    bf16x8 wa[R], wb[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      wa[r] = load_nt(reinterpret_cast<const bf16x8*>(wr[r] + k0));
      wb[r] = load_nt(reinterpret_cast<const bf16x8*>(wr[r] + k0 + 512));
    }
#pragma unroll
    for (int m = 0; m < MAXM; ++m) {
      if (m < M) {
        const bf16x8 xa = *reinterpret_cast<const bf16x8*>(x + m * ldx + k0);
        const bf16x8 xb = *reinterpret_cast<const bf16x8*>(x + m * ldx + k0 + 512);
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r][m] = dot8(xb, wb[r], dot8(xa, wa[r], acc[r][m]));
      }
    }
  }
  if (k0 < K) {  // K / 8 not a multiple of 128 chunks: one last single chunk per lane
    bf16x8 wa[R];
#pragma unroll
    for (int r = 0; r < R; ++r) wa[r] = load_nt(reinterpret_cast<const bf16x8*>(wr[r] + k0));
#pragma unroll
    for (int m = 0; m < MAXM; ++m) {
      if (m < M) {
        const bf16x8 xa = *reinterpret_cast<const bf16x8*>(x + m * ldx + k0);
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r][m] = dot8(xa, wa[r], acc[r][m]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int m = 0; m < MAXM; ++m) {
      if (m < M && n0 + r < N) {
        float v = wave_sum(acc[r][m]);
        if (lane == 0) {
          if (bias) v += (float)bias[n0 + r];
          y[m * ldy + n0 + r] = (bf16)v;
        }
      }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// Fused decode GEMV: the pre-norm and the gated activation of a decoder layer folded into its projection GEMVs, so a
// decode step launches neither the RMSNorm nor the GLU kernel (each ~4-5 us per call in a decode graph, i.e. about a
// tenth of a Llama-3-8B B = 1 step, for kernels that move a few KB).
//
// NORM: the input rows are x = bf16(r * rstd * gamma), r = bf16(h + res) (or h without a residual) -- the arithmetic
// of norm.hip's RMSNorm forward. rstd is one scalar per row, so x . w = rstd * (bf16(r * gamma) . w): a wave streams
// its weight rows against bf16(r * gamma) chunks built on the fly (r and gamma are L2-resident, K * 2 bytes) and, since
// its 64 lanes together walk the whole row, accumulates sum(r^2) in the same loop; rstd scales the reduced dot
// products at the end. No workgroup-wide prologue (row reduction, LDS, barriers) sits ahead of the weight stream: that
// serial prologue cost what a separate RMSNorm launch did (fused qkv 15.4 us vs 10.9 us plain GEMV + 4.6 us norm).
// Workgroup 0 also writes r (the new residual stream) and, when asked, x (the normed rows: HCache's hidden-state
// latents) once its waves know rstd.
// GLU: the weight is [gate; up] ([2I, K]) and the output y[M, I] = bf16(act(bf16(x.g_j)) * bf16(x.u_j)): a wave
// owns R output columns and streams their gate AND up rows, so the [M, 2I] intermediate never exists.
__device__ __forceinline__ float silu_f(float v) { return v * __builtin_amdgcn_rcpf(1.f + __expf(-v)); }
// gated unit, by the codes of act.hip: 0 silu, 1 gelu_tanh, 2 relu, 5 the clamped form with its limit
__device__ __forceinline__ float gate_f(float v, int act) {
  if (act == 2) return fmaxf(v, 0.f);
  if (act == 1) return 0.5f * v * (1.f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
  return silu_f(v);
}
__device__ __forceinline__ float gated_f(float g, float u, int act, float limit) {
  if (act != 5) return gate_f(g, act) * u;
  g = fminf(g, limit);
  return g * __builtin_amdgcn_rcpf(1.f + __expf(-1.702f * g)) * (fminf(fmaxf(u, -limit), limit) + 1.f);
}

// r = bf16(h + res) (h without res) for 8 elements at k
__device__ __forceinline__ bf16x8 load_r(const bf16* __restrict__ h, const bf16* __restrict__ res, int64_t off, int k) {
  bf16x8 hv = *reinterpret_cast<const bf16x8*>(h + off + k);
  if (res != nullptr) {
    const bf16x8 rv = *reinterpret_cast<const bf16x8*>(res + off + k);
#pragma unroll
    for (int j = 0; j < 8; ++j) hv[j] = (bf16)((float)hv[j] + (float)rv[j]);  // round like the unfused add
  }
  return hv;
}

// the GEMV operand chunk: bf16(r * gamma) with sum(r^2) accumulated into ss (NORM), else h itself
template <bool NORM>
__device__ __forceinline__ bf16x8 load_x(const bf16* __restrict__ h, const bf16* __restrict__ res,
                                         const bf16* __restrict__ gamma, int64_t off, int k, float& ss) {
  if constexpr (!NORM) {
    return *reinterpret_cast<const bf16x8*>(h + off + k);
  } else {
    const bf16x8 r = load_r(h, res, off, k);
    const bf16x8 g = *reinterpret_cast<const bf16x8*>(gamma + k);
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float v = (float)r[j];
      ss += v * v;
      o[j] = (bf16)(v * (float)g[j]);
    }
    return o;
  }
}

template <int MAXM, int R, bool NORM, bool GLU>
__global__ __launch_bounds__(256) void gemv_fused_kernel(const bf16* __restrict__ h, const bf16* __restrict__ res,
                                                         const bf16* __restrict__ gamma, float eps,
                                                         const bf16* __restrict__ w, bf16* __restrict__ y,
                                                         bf16* __restrict__ r_out, bf16* __restrict__ x_out, int act,
                                                         float limit, int M, int N, int K, int64_t ldh, int64_t ldy) {
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const int n0 = (blockIdx.x * 4 + wid) * R;  // output columns [n0, n0 + R)
  const bool writes_rows = NORM && blockIdx.x == 0 && (r_out != nullptr || x_out != nullptr);
  if (n0 >= N && !writes_rows) return;  // (workgroup 0's waves all run: they share the row writes below)
  constexpr int RR = GLU ? 2 * R : R;   // weight rows streamed per wave: the gate rows, then the up rows
  float acc[RR][MAXM], ss[MAXM];
#pragma unroll
  for (int m = 0; m < MAXM; ++m) {
    ss[m] = 0.f;
#pragma unroll
    for (int r = 0; r < RR; ++r) acc[r][m] = 0.f;
  }
  const bf16* wr[RR];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int n = min(n0 + r, N - 1);  // tail columns re-read column N-1 (unused)
    wr[r] = w + (int64_t)n * K;
    if constexpr (GLU) wr[R + r] = w + (int64_t)(N + n) * K;
  }
  int k0 = 8 * lane;
  for (; k0 + 512 < K; k0 += 1024) {
    bf16x8 wa[RR], wb[RR];
#pragma unroll
    for (int r = 0; r < RR; ++r) {
      wa[r] = load_nt(reinterpret_cast<const bf16x8*>(wr[r] + k0));
      wb[r] = load_nt(reinterpret_cast<const bf16x8*>(wr[r] + k0 + 512));
    }
#pragma unroll
    for (int m = 0; m < MAXM; ++m) {
      if (m < M) {
        const bf16x8 xa = load_x<NORM>(h, res, gamma, m * ldh, k0, ss[m]);
        const bf16x8 xb = load_x<NORM>(h, res, gamma, m * ldh, k0 + 512, ss[m]);
#pragma unroll
        for (int r = 0; r < RR; ++r) acc[r][m] = dot8(xb, wb[r], dot8(xa, wa[r], acc[r][m]));
      }
    }
  }
  if (k0 < K) {
    bf16x8 wa[RR];
#pragma unroll
    for (int r = 0; r < RR; ++r) wa[r] = load_nt(reinterpret_cast<const bf16x8*>(wr[r] + k0));
#pragma unroll
    for (int m = 0; m < MAXM; ++m) {
      if (m < M) {
        const bf16x8 xa = load_x<NORM>(h, res, gamma, m * ldh, k0, ss[m]);
#pragma unroll
        for (int r = 0; r < RR; ++r) acc[r][m] = dot8(xa, wa[r], acc[r][m]);
      }
    }
  }
  float rstd[MAXM];
#pragma unroll
  for (int m = 0; m < MAXM; ++m) rstd[m] = NORM ? rsqrtf(wave_sum(ss[m]) / (float)K + eps) : 1.f;
  if (writes_rows) {  // the 4 waves of workgroup 0 split the rows' chunks
    for (int c = (wid * 64 + lane) * 8; c < K; c += 2048) {
#pragma unroll
      for (int m = 0; m < MAXM; ++m) {
        if (m < M) {
          const bf16x8 r = load_r(h, res, m * ldh, c);
          if (r_out != nullptr && res != nullptr) *reinterpret_cast<bf16x8*>(r_out + m * ldh + c) = r;
          if (x_out != nullptr) {
            const bf16x8 g = *reinterpret_cast<const bf16x8*>(gamma + c);
            bf16x8 o;
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = (bf16)((float)r[j] * rstd[m] * (float)g[j]);
            *reinterpret_cast<bf16x8*>(x_out + m * ldh + c) = o;
          }
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int m = 0; m < MAXM; ++m) {
      if (m < M && n0 + r < N) {
        const float v = rstd[m] * wave_sum(acc[r][m]);
        if constexpr (GLU) {
          const float u = rstd[m] * wave_sum(acc[R + r][m]);
          if (lane == 0) y[m * ldy + n0 + r] = (bf16)gated_f((float)(bf16)v, (float)(bf16)u, act, limit);
        } else {
          if (lane == 0) y[m * ldy + n0 + r] = (bf16)v;
        }
      }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// One row. A wave of the kernels above walks whole weight rows, two pieces at a time: at N = 2048 that is 2 KB on the way a wave
// and a chain of K / 1024 round trips. Here a workgroup of four waves owns two columns (with GLU their gate and up rows) and
// the waves take turns at pieces of 512 U along K, so that a wave has all rows' pieces on the way and a chain a quarter as
// long; the sums meet in LDS once. The pre-norm works as above: its scale is one factor of the finished sums, the squares are
// summed beside them. Measured before -> now: [2 x 5632, 2048] with norm and GLU 13.1 -> 10.7 us, [3072, 2048] with norm 6.4
// -> 5.4, [2048, 5632] 6.6 -> 6.0, [2 x 14336, 4096] 45.7 -> 38.6 (6.1 TB/s), [4096, 4096] 8.5 -> 7.4, LM heads [32000, 2048]
// 27.3 -> 22.4 and [32000, 4096] 47.8 -> 40.6. Four or eight columns a workgroup are level or slower (11.6 and 12.9 us at the
// first), eight waves too.
struct OneRow {
  const bf16* h;      // [K]
  const bf16* res;    // [K] or null
  const bf16* gamma;  // [K]: NORM
  float eps;
  const bf16* w;
  const bf16* bias;   // [N] or null
  bf16* y;            // [N]
  bf16* r_out;        // [K] or null: h + res
  bf16* x_out;        // [K] or null: the normed row
  int N, K, act;
  float limit;
};

template <int U, bool NORM, bool GLU, bool GATHER>
__global__ __launch_bounds__(256) void gemv_row_kernel(OneRow p, Gather gather) {
  constexpr int R = 2, RR = GLU ? 2 * R : R, S = 4 * 512;
  __shared__ float red[4][RR + 1];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, n0 = blockIdx.x * R;
  const bf16* wr[RR];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int n = min(n0 + r, p.N - 1);  // a tail column re-reads column N - 1 (not stored)
    wr[r] = p.w + (int64_t)n * p.K;
    if constexpr (GLU) wr[R + r] = p.w + ((int64_t)p.N + n) * p.K;
  }
  float acc[RR], ss = 0.f;
#pragma unroll
  for (int r = 0; r < RR; ++r) acc[r] = 0.f;
  for (int k0 = 512 * wid + 8 * lane; k0 < p.K; k0 += S * U) {
    bf16x8 a[U][RR], x[U], g[U], q[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * S < p.K ? k0 + u * S : k0;
#pragma unroll
      for (int r = 0; r < RR; ++r) a[u][r] = load_nt(reinterpret_cast<const bf16x8*>(wr[r] + k));
      x[u] = *reinterpret_cast<const bf16x8*>(p.h + k);
      if constexpr (NORM) {
        g[u] = *reinterpret_cast<const bf16x8*>(p.gamma + k);
        if (p.res != nullptr) q[u] = *reinterpret_cast<const bf16x8*>(p.res + k);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u > 0 && k0 + u * S >= p.K) break;
      bf16x8 o = x[u];
      if constexpr (NORM) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          float v = (float)x[u][j];
          if (p.res != nullptr) v = (float)(bf16)(v + (float)q[u][j]);  // round like the unfused add
          ss += v * v;
          o[j] = (bf16)(v * (float)g[u][j]);
        }
      }
#pragma unroll
      for (int r = 0; r < RR; ++r) acc[r] = dot8(o, a[u][r], acc[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < RR; ++r) {
    acc[r] = wave_sum(acc[r]);
    if (lane == 0) red[wid][r] = acc[r];
  }
  if constexpr (NORM) {
    ss = wave_sum(ss);
    if (lane == 0) red[wid][RR] = ss;
  }
  __syncthreads();
  auto total = [&](int r) { return red[0][r] + red[1][r] + red[2][r] + red[3][r]; };
  const float rstd = NORM ? rsqrtf(total(RR) / (float)p.K + p.eps) : 1.f;
  if ((int)threadIdx.x < R && n0 + (int)threadIdx.x < p.N) {
    const int n = n0 + threadIdx.x;
    float v = rstd * total(threadIdx.x);
    if constexpr (GLU) {
      const float u = rstd * total(R + threadIdx.x);
      p.y[n] = (bf16)gated_f((float)(bf16)v, (float)(bf16)u, p.act, p.limit);
    } else {
      if (p.bias != nullptr) v += (float)p.bias[n];
      if constexpr (GATHER) v = gather(v, 0, n);
      p.y[n] = (bf16)v;
    }
  }
  if (NORM && blockIdx.x == 0 && (p.r_out != nullptr || p.x_out != nullptr)) {
    for (int c = threadIdx.x * 8; c < p.K; c += 2048) {
      const bf16x8 r = load_r(p.h, p.res, 0, c);
      if (p.r_out != nullptr && p.res != nullptr) *reinterpret_cast<bf16x8*>(p.r_out + c) = r;
      if (p.x_out != nullptr) {
        const bf16x8 g = *reinterpret_cast<const bf16x8*>(p.gamma + c);
        bf16x8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = (bf16)((float)r[j] * rstd * (float)g[j]);
        *reinterpret_cast<bf16x8*>(p.x_out + c) = o;
      }
    }
  }
}

// One row: where the kernels above, a column (or a few) of a wave, are still the faster ones. A turn of gemv_row_kernel is 2048 of
// K, and with a norm each pair of columns reads h and gamma again. us, this kernel / those:
// K up to 1024 (half of its waves have nothing to read): [1024, 512] 2.31 / 2.07, [3072, 1024] 3.36 / 3.16, [16384, 256] 6.86 / 4.32;
// with a norm [16384, 1024] 12.1 / 9.3. K = 768 is a piece and a half of those, which they make up for from 6144 columns on: [512,
// 768] 2.31 / 2.38, [6144, 768] 4.19 / 3.90;
// plain, K to 2048 and few columns: [2048, 2048] 3.61 / 3.44, [3072, 2048] 4.51 / 4.35, [4096, 2048] 5.16 / 5.46;
// a norm before many columns: [27648, 5120] 57.9 / 53.7, [28672, 14336] 163 / 152, [16384, 2560] 19.7 / 18.5; of K = 2048, 4096, 6144 and
// 8192, whole turns, this one: [16384, 2048] 14.8 / 17.9, [28672, 4096] 45.7 / 47.3, [12288, 6144] 31.4 / 34.0;
// gated without a norm, K of no whole turns: [2 x 2048, 2560] 6.6 / 6.4, [2 x 2048, 5120] 10.2 / 9.8, [2 x 4096, 2560] 9.9 / 10.2.
template <bool NORM, bool GLU>
bool row_by_columns(int N, int K) {
  if (K <= 1024) return (GLU && !NORM) || K % 512 == 0 || K < 512 || N >= 6144;
  if (NORM) return !GLU && N >= 12288 && (K % 2048 != 0 || K > 8192);
  if (GLU) return K % 2048 != 0 && K <= 5120 && N <= 2048;
  return K <= 2048 && K % 512 == 0 && N >= 768 && N <= 3072;
}

// Two pieces a wave on the way instead of one from the second turn on: plain [6144, 2560] 7.6 for 8.2 us (fewer columns stay with one:
// in a chain of launches [2048, 5632] takes 0.3 us more with two, where repeated by itself it is level), [28672, 4096] 39.7 / 39.5,
// [12288, 14336] 60.9 / 62.6, gated [2 x 14336, 3072] 31.3 / 32.0. With a norm, whose work a piece past the end repeats, only gated and
// where K has whole pairs: [2 x 8192, 4096] 26.8 for 27.7, [2 x 14336, 6144] 70.0 for 62.5; not gated [27648, 5120] 64.5 for 57.9.
template <bool NORM, bool GLU, bool GATHER>
int launch_row(const OneRow& p, const Gather& gather, hipStream_t st) {
  const dim3 grid((p.N + 1) / 2);
  if (NORM ? GLU && p.K % 4096 == 0 : p.K > 2048 && p.N >= 4096)
    hipLaunchKernelGGL((gemv_row_kernel<2, NORM, GLU, GATHER>), grid, dim3(256), 0, st, p, gather);
  else
    hipLaunchKernelGGL((gemv_row_kernel<1, NORM, GLU, GATHER>), grid, dim3(256), 0, st, p, gather);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------------
// Skinny GEMM for 2..16 token rows on the matrix cores: y[M, N] = x[M, K] . W[N, K]^T (+ bias).
// The VALU GEMV above spends 4 dot2 instructions per 16-B weight chunk PER ROW, so from a few rows on it is VALU-bound
// (o projection at M = 8: 1.7 TB/s) and hipBLASLt's small-M tiles stream at 3.5-3.7 TB/s. Here one
// mfma_f32_16x16x32_bf16 contracts a 16-row x 32-k weight tile with all (up to 16) token rows at once, so the
// kernel is a pure weight stream: A = W rows (lane l: row l & 15, k = 8 (l >> 4) .. +8), B = x^T
// (lane l: token l & 15, same k), C: token = l & 15, weight row 4 (l >> 4) + reg. A workgroup owns 16
// weight rows; its waves share K, and the partial tiles are summed through LDS.
// GLU: W is [gate; up] of 2 N rows, a tile is 8 gate rows and the 8 up rows that belong to them, so that there are as many
// workgroups as without (a tile of 16 + 16 rows left half of the chip's slots empty and lost against the separate
// kernel), and y = bf16(act(bf16(gate)) * bf16(up)).
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct SkinnyOut {
  const bf16* bias;
  bf16* y;
  int M, N;
  int64_t ldy;
  int act;  // GLU
  RowScale scale;  // SCALE
  RowNorm norm;    // NORM: y, r and res [M, N]
};

// W's row r (of 16) of the workgroup's tile; rows past the end re-read the last one (not stored)
template <bool GLU>
__device__ __forceinline__ int64_t skinny_row(int r, int N) {
  if constexpr (GLU) {
    const int n = min((int)blockIdx.x * 8 + (r & 7), N - 1);
    return r < 8 ? n : (int64_t)N + n;
  }
  return min((int)blockIdx.x * 16 + r, N - 1);
}

template <bool GATHER, bool GLU>
__device__ __forceinline__ void skinny_store(const SkinnyOut& o, const Gather& gather, f32x4 acc, int lane) {
  const int tok = lane & 15, g = lane >> 4;
  if constexpr (GLU) {  // lanes of the upper half hold the up rows of those 32 below
    const int n0 = blockIdx.x * 8 + 4 * (g & 1);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = n0 + r;
      float v = acc[r];
      if (o.bias != nullptr && n < o.N) v += (float)o.bias[lane < 32 ? n : o.N + n];
      const float up = __shfl_down(v, 32, 64);
      if (lane < 32 && tok < o.M && n < o.N)
        o.y[(int64_t)tok * o.ldy + n] = (bf16)(gate_f((float)(bf16)v, o.act) * (float)(bf16)up);
    }
  } else if (tok < o.M) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = blockIdx.x * 16 + 4 * g + r;
      if (n < o.N) {
        float v = acc[r];
        if (o.bias != nullptr) v += (float)o.bias[n];
        if constexpr (GATHER) v = gather(v, tok, n);
        o.y[(int64_t)tok * o.ldy + n] = (bf16)v;
      }
    }
  }
}

// The tokens are as many bytes of loads as the weights, served by the L2, and what bounds such a kernel is how many cache
// lines a CU can have on the way; with 16-B pieces of 16 weight rows, straight into the operand's registers, a load asks
// for half a line of each. Here a load takes whole lines (8 rows of 64 columns), which pass through the wave's own piece
// of LDS into the operand's layout (16-B pieces, placed by row ^ piece so that the reads spread over the banks); a wave has
// 128 columns in flight and there are up to 32 waves a CU to overlap them. Pieces (a quarter of K a wave) -> this, 2 / 4 / 8
// / 16 rows: [28672, 4096] 40.1 / 42.0 / 48.1 / 60.6 -> 39.6 / 40.0 / 41.3 / 48.8 us (4.8 TB/s at 16), [4096, 14336] 26.8 / 25.8 /
// 26.9 / 29.9 -> 22.8 / 22.1 / 22.4 / 25.5, [6144, 4096] 13.5 / 13.5 / 14.7 / 17.6 -> 12.8 / 12.2 / 12.7 / 13.8, [2048, 5632]
// 13.0 / 13.0 / 13.6 / 15.1 -> 8.7 / 7.7 / 8.5 / 10.2, [32000, 2048] 25.2 / 25.7 / 29.7 / 36.4 -> 24.9 / 25.4 / 26.2 / 29.9. Two
// tiles a workgroup halve the tokens' loads but were slower (54 to 59 us), the DMA into LDS is level.
// Weight rows of a multiple of 4 KB lie alike in the memory's channels, and workgroups that walk them side by side meet in
// the same ones. There each begins somewhere else, by the fractions of the golden ratio (any distance apart is far apart):
// 8 rows, [4096, 16384] 35.8 -> 24.0 us, [4096, 32768] 60 -> 46, [4096, 4096] 8.5 -> 7.7, [32000, 2048] level. With other rows
// it gains or loses up to 4 % ([5120, 13824]), with gate and up rows, which are a matrix apart, nothing.
// SCALE: rows of a residual stream that is still to be scaled; NORM: what becomes of the sums is such a stream (row_norm.h)
template <int NW, bool GATHER, bool GLU, bool SCALE = false, bool NORM = false>
__global__ __launch_bounds__(64 * NW) void skinny_lines_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                               int K, int64_t ldx, SkinnyOut o, Gather gather) {
  __shared__ __attribute__((aligned(16))) char buf[NW][4096];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int wr = lane >> 3, wz = lane & 7, rr = lane & 15, rp = lane >> 4;
  const bf16* w0 = w + skinny_row<GLU>(wr, o.N) * K + 8 * wz;
  const bf16* w1 = w + skinny_row<GLU>(8 + wr, o.N) * K + 8 * wz;
  const bf16* xp = x + (int64_t)min(rr, o.M - 1) * ldx + 8 * rp;  // (columns past M are not stored)
  char* mine = buf[wid];
  char* put = mine + wr * 128 + (wz ^ wr) * 16;
  const char* get0 = mine + rr * 128 + (rp ^ (rr & 7)) * 16;
  const char* get1 = mine + rr * 128 + ((rp + 4) ^ (rr & 7)) * 16;
  __shared__ __attribute__((aligned(16))) float red[SCALE ? NW * 16 : 4];
  RowSums<64 * NW> sums;
  if constexpr (SCALE) sums.load(o.scale);
  bf16x4 res{}, gamma{};
  const int64_t at = (int64_t)rr * o.N + blockIdx.x * 16 + 4 * rp;
  if constexpr (NORM) {
    if (wid == 0) {
      if (rr < o.M) res = *reinterpret_cast<const bf16x4*>(o.norm.res + at);
      gamma = *reinterpret_cast<const bf16x4*>(o.norm.gamma + blockIdx.x * 16 + 4 * rp);
    }
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const int parts = K >> 7, turn = GLU || K % 2048 ? 0 : (int)__umulhi(blockIdx.x * 2654435769u, (unsigned)parts);
  for (int c = wid; c < parts; c += NW) {  // K % 128 == 0
    int k = c + turn;
    k = (k < parts ? k : k - parts) << 7;
    bf16x8_t a[2][2], b[4];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      a[u][0] = load_nt(reinterpret_cast<const bf16x8_t*>(w0 + k + 64 * u));
      a[u][1] = load_nt(reinterpret_cast<const bf16x8_t*>(w1 + k + 64 * u));
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) b[u] = *reinterpret_cast<const bf16x8_t*>(xp + k + 32 * u);
    __builtin_amdgcn_sched_barrier(0);  // (the last of them waited for by itself: 54 us instead of 48 at [28672, 4096])
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      *reinterpret_cast<bf16x8_t*>(put + u * 2048) = a[u][0];
      *reinterpret_cast<bf16x8_t*>(put + u * 2048 + 1024) = a[u][1];
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const bf16x8_t p0 = *reinterpret_cast<const bf16x8_t*>(get0 + u * 2048);
      const bf16x8_t p1 = *reinterpret_cast<const bf16x8_t*>(get1 + u * 2048);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p0, b[2 * u], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p1, b[2 * u + 1], acc, 0, 0, 0);
    }
  }
  reinterpret_cast<f32x4*>(mine)[lane] = acc;
  if constexpr (SCALE) sums.add(o.scale, red);
  __syncthreads();
  if (wid > 0) return;
#pragma unroll
  for (int v = 1; v < NW; ++v) acc += reinterpret_cast<const f32x4*>(buf[v])[lane];
  if constexpr (SCALE) acc *= RowSums<64 * NW>::rstd(o.scale, red, rr);
  if constexpr (NORM) store_normed(o.norm, o.y, at, acc, res, gamma, blockIdx.x, lane, rr < o.M);
  else skinny_store<GATHER, GLU>(o, gather, acc, lane);
}

// Waves a workgroup: four where there are at least two workgroups a CU of whole K walks ([6144, 4096] 13.7 us against 14.7
// with eight, [28672, 4096] 48.6 / 50.4), eight where those are few ([4096, 14336] 26.6 against 27.9, [2048, 8192] 13.0 / 14.0)
// or short ([16384, 2048] 17.9 / 19.0), and at up to 8 rows, whose tokens take fewer loads ([28672, 4096], 7 rows: 40.1 / 41.7).
template <bool GATHER, bool GLU, bool SCALE = false, bool NORM = false>
int launch_skinny(const void* x, const void* w, int K, int64_t ldx, const SkinnyOut& o, const Gather& gather,
                  hipStream_t st) {
  const int per = GLU ? 8 : 16, tiles = (o.N + per - 1) / per;
#define HDS_SK(T, ...) \
  hipLaunchKernelGGL((__VA_ARGS__), dim3(tiles), dim3(T), 0, st, (const bf16*)x, (const bf16*)w, K, ldx, o, gather)
  if (o.M > 8 && tiles > 256 && K >= 4096)
    HDS_SK(256, skinny_lines_kernel<4, GATHER, GLU, SCALE, NORM>);
  else
    HDS_SK(512, skinny_lines_kernel<8, GATHER, GLU, SCALE, NORM>);
#undef HDS_SK
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------------
// One decode step of the gated recurrence (gated_scan.hip) with its projection: a wave owns one channel j and streams
// the three weight rows j, N + j, 2N + j (update gate, candidate, output gate) against up to MAXM token rows, each of
// another sequence; lane 0 then advances the channel's 32-bit state of every row and writes S * silu(c). The projected
// values are rounded to bf16 first, as the separate projection stores them.
__device__ __forceinline__ void sigmoid2_f(float x, float& s, float& c) {
  const float e = __expf(-fabsf(x)), r = 1.f / (1.f + e);
  s = x >= 0.f ? r : e * r;
  c = x >= 0.f ? e * r : r;
}

template <int MAXM>
__global__ __launch_bounds__(256) void gemv_recur_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                         const float* __restrict__ ba, const float* __restrict__ bb,
                                                         bf16* __restrict__ y, float* __restrict__ state,
                                                         int64_t slot_stride, const int* __restrict__ slots,
                                                         const int* __restrict__ seq_meta, int M, int N, int K,
                                                         int64_t ldx, int64_t ldy) {
  const int lane = threadIdx.x & 63;
  const int j = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (j >= N) return;
  float acc[3][MAXM];
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int m = 0; m < MAXM; ++m) acc[r][m] = 0.f;
  const bf16* wr[3];
#pragma unroll
  for (int r = 0; r < 3; ++r) wr[r] = w + ((int64_t)r * N + j) * K;
  int k0 = 8 * lane;
  for (; k0 + 512 < K; k0 += 1024) {
    bf16x8 wa[3], wb[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      wa[r] = load_nt(reinterpret_cast<const bf16x8*>(wr[r] + k0));
      wb[r] = load_nt(reinterpret_cast<const bf16x8*>(wr[r] + k0 + 512));
    }
#pragma unroll
    for (int m = 0; m < MAXM; ++m) {
      if (m < M) {
        const bf16x8 xa = *reinterpret_cast<const bf16x8*>(x + m * ldx + k0);
        const bf16x8 xb = *reinterpret_cast<const bf16x8*>(x + m * ldx + k0 + 512);
#pragma unroll
        for (int r = 0; r < 3; ++r) acc[r][m] = dot8(xb, wb[r], dot8(xa, wa[r], acc[r][m]));
      }
    }
  }
  if (k0 < K) {
    bf16x8 wa[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) wa[r] = load_nt(reinterpret_cast<const bf16x8*>(wr[r] + k0));
#pragma unroll
    for (int m = 0; m < MAXM; ++m) {
      if (m < M) {
        const bf16x8 xa = *reinterpret_cast<const bf16x8*>(x + m * ldx + k0);
#pragma unroll
        for (int r = 0; r < 3; ++r) acc[r][m] = dot8(xa, wa[r], acc[r][m]);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < MAXM; ++m) {
    if (m < M) {
      const float a = (float)(bf16)wave_sum(acc[0][m]) + ba[j], b = (float)(bf16)wave_sum(acc[1][m]) + bb[j];
      const float g = (float)(bf16)wave_sum(acc[2][m]);
      if (lane == 0) {
        float* st = state + (int64_t)slots[m] * slot_stride + j;
        const float s0 = seq_meta[3 * m + 2] > 0 ? *st : 0.f;
        float z, keep, us, uc, gs, gc;
        sigmoid2_f(a, z, keep);
        sigmoid2_f(b, us, uc);
        sigmoid2_f(g, gs, gc);
        const float s = keep * s0 + z * (b >= 0.f ? b + 0.5f : us);
        *st = s;
        y[m * ldy + j] = (bf16)(s * g * gs);
      }
    }
  }
}

}  // namespace

// A decode step of the recurrence for M <= 8 sequences (row m of x is the one new token of sequence m): w is [3N, K]
// (update gate, candidate, output gate rows), y [M, N] with row stride ldy. K % 8 == 0, 16-B aligned x and w.
HDS_EXPORT int hds_gemv_recur_bf16(const void* x, const void* w, const float* ba, const float* bb, void* y,
                                   float* state, int64_t slot_stride, const int* slots, const int* seq_meta, int M,
                                   int N, int K, int64_t ldx, int64_t ldy, hipStream_t st) {
  if (M < 1 || M > 8 || N < 1 || K < 8 || K % 8 || ldx % 8 || ldx < K || ldy < N || !state || !slots || !seq_meta)
    return hipErrorInvalidValue;
#define HDS_RC(MM)                                                                                                   \
  hipLaunchKernelGGL(gemv_recur_kernel<MM>, dim3((N + 3) / 4), dim3(256), 0, st, (const bf16*)x, (const bf16*)w, ba, \
                     bb, (bf16*)y, state, slot_stride, slots, seq_meta, M, N, K, ldx, ldy)
  if (M == 1) HDS_RC(1); else if (M <= 2) HDS_RC(2); else if (M <= 4) HDS_RC(4); else HDS_RC(8);
#undef HDS_RC
  return hipGetLastError();
}

// Skinny matrix-core GEMM: 1 <= M <= 16, K % 128 == 0, 16-B aligned rows. glu: 0, or 1 + activation code (0 silu, 1
// gelu_tanh, 2 relu) for w = [gate; up] of 2 N rows
HDS_EXPORT int hds_skinny_gemm_bf16(const void* x, const void* w, const void* bias, void* y, int M, int N, int K,
                                    int64_t ldx, int64_t ldy, int glu, hipStream_t st) {
  if (M < 1 || M > 16 || N < 1 || K < 128 || K % 128 || ldx % 8 || glu < 0 || glu > 3) return hipErrorInvalidValue;
  const SkinnyOut o{(const bf16*)bias, (bf16*)y, M, N, ldy, glu - 1, {}, {}};
  return glu ? launch_skinny<false, true>(x, w, K, ldx, o, Gather{}, st)
             : launch_skinny<false, false>(x, w, K, ldx, o, Gather{}, st);
}

// The same with a norm on either side (row_norm.h), M of 1 to 16 rows. ssq [parts][16] or null: x is a stream still to be scaled,
// of K = 16 parts columns. res [M, N] or null: y = x . W^T is added to it, r and bf16(r gamma) in y's place are stored, and
// the tiles' sums in ssq_out [N / 16][16]; N % 16 == 0, no gated unit.
HDS_EXPORT int hds_skinny_norm_bf16(const void* x, const void* w, void* y, const float* ssq, float eps, const void* res,
                                    const void* gamma, void* r, float* ssq_out, int M, int N, int K, int glu, hipStream_t st) {
  if (M < 1 || M > 16 || N < 1 || K < 128 || K % 128 || glu < 0 || glu > 3 || (ssq == nullptr && res == nullptr) ||
      (ssq != nullptr && res != nullptr) || (res != nullptr && (glu || N % 16 || !gamma || !r || !ssq_out)))
    return hipErrorInvalidValue;
  const SkinnyOut o{nullptr, (bf16*)y, M, N, N, glu - 1, {ssq, K / 16, eps}, {(const bf16*)res, (const bf16*)gamma, (bf16*)r, ssq_out}};
  if (res != nullptr) return launch_skinny<false, false, false, true>(x, w, K, K, o, Gather{}, st);
  return glu ? launch_skinny<false, true, true, false>(x, w, K, K, o, Gather{}, st)
             : launch_skinny<false, false, true, false>(x, w, K, K, o, Gather{}, st);
}

// Fused decode GEMV (see gemv_fused_kernel): y[M, N] = norm(h (+ res)) . W^T, or with glu = 1 + activation code
// (0 silu, 1 gelu_tanh, 2 relu, 5 the clamped gate with its limit), y[M, N] = act(x . Wg^T) * (x . Wu^T) for W = [Wg; Wu] of 2N rows (x normed when gamma is given, else h itself). r_out /
// x_out (workgroup 0, with gamma): the new residual rows and the normed rows. ldh: row stride of h / res / r_out /
// x_out (elements); ldy: row stride of y. Shapes: M <= 8, K % 8 == 0, 16-B aligned operands (checked by the caller).
HDS_EXPORT int hds_gemv_fused_bf16(const void* h, const void* res, const void* gamma, float eps, const void* w,
                                   void* y, void* r_out, void* x_out, int glu, float limit, int M, int N, int K,
                                   int64_t ldh, int64_t ldy, hipStream_t st) {
  if (M < 1 || M > 8 || N < 1 || K < 8 || K % 8 || ldh % 8 || glu < 0 || glu > 6 || glu == 4 || glu == 5) return hipErrorInvalidValue;
  const int act = glu - 1;
  if (gamma == nullptr && (r_out != nullptr || x_out != nullptr || res != nullptr)) return hipErrorInvalidValue;
  if (M == 1 && !(gamma != nullptr ? (glu ? row_by_columns<true, true>(N, K) : row_by_columns<true, false>(N, K))
                                   : row_by_columns<false, true>(N, K))) {
    const OneRow p{(const bf16*)h, (const bf16*)res, (const bf16*)gamma, eps, (const bf16*)w, nullptr, (bf16*)y,
                   (bf16*)r_out, (bf16*)x_out, N, K, act, limit};
    if (gamma != nullptr) return glu ? launch_row<true, true, false>(p, Gather{}, st) : launch_row<true, false, false>(p, Gather{}, st);
    return glu ? launch_row<false, true, false>(p, Gather{}, st) : hipErrorInvalidValue;  // plain GEMV: hds_gemv_bf16
  }
  const int R = N >= 8192 ? (glu ? 2 : 4) : (N >= 4096 ? 2 : 1);
#define HDS_GF(MM, RR, NN, GG)                                                                                   \
  hipLaunchKernelGGL((gemv_fused_kernel<MM, RR, NN, GG>), dim3((N + 4 * RR - 1) / (4 * RR)), dim3(256), 0, st,  \
                     (const bf16*)h, (const bf16*)res, (const bf16*)gamma, eps, (const bf16*)w, (bf16*)y,      \
                     (bf16*)r_out, (bf16*)x_out, act, limit, M, N, K, ldh, ldy)
#define HDS_GFM(RR, NN, GG)                                                                                    \
  if (M == 1) HDS_GF(1, RR, NN, GG); else if (M <= 2) HDS_GF(2, RR, NN, GG);                                   \
  else if (M <= 4) HDS_GF(4, RR, NN, GG); else HDS_GF(8, RR, NN, GG);
#define HDS_GFR(NN, GG)                                                                                        \
  if (R == 4) { HDS_GFM(4, NN, GG) } else if (R == 2) { HDS_GFM(2, NN, GG) } else { HDS_GFM(1, NN, GG) }
  if (gamma != nullptr) {
    if (glu) { HDS_GFR(true, true) } else { HDS_GFR(true, false) }
  } else {
    if (glu) { HDS_GFR(false, true) } else { return hipErrorInvalidValue; }  // plain GEMV: hds_gemv_bf16
  }
#undef HDS_GFR
#undef HDS_GFM
#undef HDS_GF
  return hipGetLastError();
}

// Shapes the kernel takes: M <= 8 rows, K a multiple of 8 (16-B rows), 16-B aligned operands (checked by the caller).
HDS_EXPORT int hds_gemv_bf16_supported(int M, int N, int K) { return M >= 1 && M <= 8 && N >= 1 && K >= 8 && K % 8 == 0; }

HDS_EXPORT int hds_gemv_bf16(const void* x, const void* w, const void* bias, void* y, int M, int N, int K, int64_t ldx,
                             int64_t ldy, hipStream_t st) {
  if (!hds_gemv_bf16_supported(M, N, K) || ldx % 8) return hipErrorInvalidValue;
  if (M == 1 && !row_by_columns<false, false>(N, K))
    return launch_row<false, false, false>(OneRow{(const bf16*)x, nullptr, nullptr, 0.f, (const bf16*)w, (const bf16*)bias,
                                                  (bf16*)y, nullptr, nullptr, N, K, 0, 0.f}, Gather{}, st);
  // R = 4 rows per wave while that still leaves >= 2 waves per SIMD on 256 CUs, else 2 / 1 (parallelism)
#define HDS_GV(MM, RR)                                                                                        \
  hipLaunchKernelGGL((gemv_bf16_kernel<MM, RR>), dim3((N + 4 * RR - 1) / (4 * RR)), dim3(256), 0, st, (const bf16*)x, \
                     (const bf16*)w, (const bf16*)bias, (bf16*)y, M, N, K, ldx, ldy)
#define HDS_GVM(RR)                                                                                           \
  if (M == 1) HDS_GV(1, RR); else if (M <= 2) HDS_GV(2, RR); else if (M <= 4) HDS_GV(4, RR); else HDS_GV(8, RR);
  if (N >= 8192) {
    HDS_GVM(4)
  } else if (N >= 4096) {
    HDS_GVM(2)
  } else {
    HDS_GVM(1)
  }
#undef HDS_GVM
#undef HDS_GV
  return hipGetLastError();
}

// y[M, N] = act(x . W^T) * table[ids[m], :N] (act: 0 silu, 1 gelu_tanh, 2 relu) for up to 16 rows: one row takes the GEMV
// (K % 8 == 0), more the skinny GEMM (K % 128 == 0). 16-B aligned x and w.
HDS_EXPORT int hds_gather_gemv_bf16(const void* x, const void* w, const void* table, int64_t ldt, const int64_t* ids,
                                    int vocab, int act, void* y, int M, int N, int K, int64_t ldx, int64_t ldy,
                                    hipStream_t st) {
  if (M < 1 || M > 16 || N < 1 || K < 8 || K % (M == 1 ? 8 : 128) || ldx % 8 || ldx < K || ldt < N || ldy < N ||
      vocab < 1 || act < 0 || act > 2 || table == nullptr || ids == nullptr)
    return hipErrorInvalidValue;
  const Gather gather{(const bf16*)table, ldt, ids, vocab, act};
  if (M == 1)
    return launch_row<false, false, true>(OneRow{(const bf16*)x, nullptr, nullptr, 0.f, (const bf16*)w, nullptr, (bf16*)y,
                                                 nullptr, nullptr, N, K, 0, 0.f}, gather, st);
  else
    return launch_skinny<true, false>(x, w, K, ldx, SkinnyOut{nullptr, (bf16*)y, M, N, ldy, 0, {}, {}}, gather, st);
  return hipGetLastError();
}
