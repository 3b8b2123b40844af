// RMSNorm / LayerNorm forward + backward with fused residual add, gfx950.
//
// Capability parity: the reference's inference-only norms
// (deepspeed/inference/v2/kernels/core_ops/cuda_rms_norm/rms_norm_cuda.cu `rms_norm`/`pre_rms_norm`,
//  cuda_layer_norm/layer_norm_cuda.cu `fused_ln`/`fused_residual_ln`)
// and the training LayerNorm of csrc/transformer/normalize_kernels.cu (K4). Here both
// forward AND backward exist for both norms, because the training engine uses them.
//
// Design (MI355X-first):
//   * one wave64 per row (two or four for few rows); the row lives in registers (NV = H/512 16-byte vectors per lane,
//     shared by the row's waves), so x is read from HBM exactly once in forward;
//   * residual add + norm + store of the new residual happen in one pass
//     (pre-norm transformer: h = x + r; y = norm(h)) -- one read of x and r,
//     one write of h and y, instead of three kernels;
//   * backward keeps dgamma/dbeta partials in registers across the rows a wave
//     owns, reduces across the block's waves in LDS and writes one fp32 partial
//     row per block; a second tiny kernel reduces the partials (deterministic,
//     no float atomics).
#include "hds_common.h"

using namespace hds;

namespace {

constexpr int kRowsPerBlock = 4;  // 4 waves per block, one row each per iteration
constexpr int kFewRows = 64;

// ---------------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------------
// PICK 1: with pick, output row i is made from rows pick[i] of x and res, of which there are n_in; negative ones count from
// the end, and a row outside them gives NaN. (Without PICK nothing asks at run time, which cost norms of one wave a row 0.1 us, 3 to
// 5 % of 256 rows of 512 to 2,048.) A serving step normalises only the rows whose logits are wanted: gathering
// them first took four launches (two index conversions, two gathers; 18 us of a 490 us decode step of 16 sequences).
// PICK 2: pick holds 64-bit ids and x is an embedding: its rows are copied to res_out beside their norm, an id outside it gives
// NaN in both. A step's lookup and first norm in one launch: a chain of kernels waits 2 to 4 us for each, and a long prompt's rows are
// read once less (in a graph, lookup and norm apart -> here: 4 rows of 2,048 3.6 -> 2.2 us, 16 of 4,096 3.8 -> 2.4, 2,048 of 4,096
// 16.0 -> 9.4, 16,000 of 2,048 40.8 -> 30.0).
struct PickedRow {
  int row;
  bool ok;
};
template <int PICK>
__device__ __forceinline__ PickedRow picked_row(const int* pick, int row, int n_in) {
  if constexpr (PICK == 2) {
    const int64_t id = reinterpret_cast<const int64_t*>(pick)[row];
    const bool ok = id >= 0 && id < n_in;
    return {ok ? (int)id : 0, ok};
  }
  if (!PICK || pick == nullptr) return {row, true};
  int r = pick[row];
  if (r < 0) r += n_in;
  const bool ok = r >= 0 && r < n_in;
  return {ok ? r : 0, ok};
}

// sum over a row's WPR waves; every wave of the workgroup comes here the same number of times
template <int WPR>
__device__ __forceinline__ float row_sum(float v, float* red) {
  v = wave_sum(v);
  if constexpr (WPR == 1) return v;
  const int wid = threadIdx.x >> 6;
  red[wid] = v;  // (all lanes the same)
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < WPR; ++k) s += red[wid / WPR * WPR + k];
  return s;
}

// WPR waves take a row. The few rows of a decode step would leave the latencies of a whole row's loads and stores to one wave
// each: with a residual, 16 rows of 2048 / 4096 / 8192 2.6 / 3.4 / 5.1 us, with four waves a row 2.1 / 2.4 / 2.7.
template <typename T, typename WT, int NV, bool LN, int WPR, int PICK>
__global__ __launch_bounds__(256) void norm_fwd_kernel(const T* __restrict__ x, const T* __restrict__ res,
                                                       T* __restrict__ res_out, const WT* __restrict__ w,
                                                       const WT* __restrict__ b, T* __restrict__ y,
                                                       float* __restrict__ stat_mean, float* __restrict__ stat_rstd,
                                                       int rows, int cols, float eps, const int* __restrict__ pick,
                                                       int n_in) {
  static_assert(NV % WPR == 0, "whole vectors a wave");
  constexpr int V = NV / WPR;
  __shared__ float red[2][4];
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const int row_at = blockIdx.x * (kRowsPerBlock / WPR) + wid / WPR;
  if (WPR == 1 && row_at >= rows) return;
  const bool live = row_at < rows;  // (the waves of a workgroup stay together for the sums)
  const int row = live ? row_at : rows - 1;
  const int c0 = (wid % WPR * V * 64 + lane) * 8;
  const PickedRow in = picked_row<PICK>(pick, row, n_in);
  const T* xr = x + (int64_t)in.row * cols;
  float v[V][8], wv[V][8];
#pragma unroll
  for (int i = 0; i < V; ++i) Vec8<T>::load(xr + c0 + i * 512, v[i]);
  if (res != nullptr) {
    const T* rr = res + (int64_t)in.row * cols;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      float r[8];
      Vec8<T>::load(rr + c0 + i * 512, r);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[i][j] = to_f(from_f<T>(v[i][j] + r[j]));  // round like the unfused add
    }
  }
  if constexpr (PICK == 2) {
    if (!in.ok)
#pragma unroll
      for (int i = 0; i < V; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] = NAN;
  }
  if ((PICK == 2 || res != nullptr) && res_out != nullptr && live) {
    T* ro = res_out + (int64_t)row * cols;
#pragma unroll
    for (int i = 0; i < V; ++i) Vec8<T>::store(ro + c0 + i * 512, v[i]);
  }
  if constexpr (WPR > 1) {  // in front of the barriers; with whole rows a wave the registers are worth more
#pragma unroll
    for (int i = 0; i < V; ++i) Vec8<WT>::load(w + c0 + i * 512, wv[i]);
  }
  float mean = 0.f;
  if constexpr (LN) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < V; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) s += v[i][j];
    mean = row_sum<WPR>(s, red[0]) / (float)cols;
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float d = v[i][j] - mean;
      ss += d * d;
    }
  const float sum = row_sum<WPR>(ss, red[1]);
  const float rstd = in.ok ? rsqrtf(sum / (float)cols + eps) : NAN;
  if (WPR > 1 && !live) return;
  T* yr = y + (int64_t)row * cols;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = c0 + i * 512;
    float o[8];
    if constexpr (WPR == 1) Vec8<WT>::load(w + c, wv[i]);
    if constexpr (LN) {
      float bv[8];
      if (b != nullptr) Vec8<WT>::load(b + c, bv);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (v[i][j] - mean) * rstd * wv[i][j] + (b != nullptr ? bv[j] : 0.f);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = v[i][j] * rstd * wv[i][j];
    }
    Vec8<T>::store(yr + c, o);
  }
  if (PICK != 2 && lane == 0 && wid % WPR == 0) {
    stat_rstd[row] = rstd;
    if constexpr (LN) stat_mean[row] = mean;
  }
}

// Generic-width forward (cols % 8 == 0, any cols): two passes over the row (second hits L1/L2).
template <typename T, typename WT, bool LN, int PICK>
__global__ __launch_bounds__(256) void norm_fwd_generic(const T* __restrict__ x, const T* __restrict__ res,
                                                        T* __restrict__ res_out, const WT* __restrict__ w,
                                                        const WT* __restrict__ b, T* __restrict__ y,
                                                        float* __restrict__ stat_mean, float* __restrict__ stat_rstd,
                                                        int rows, int cols, float eps, const int* __restrict__ pick,
                                                        int n_in) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const PickedRow in = picked_row<PICK>(pick, row, n_in);
  const T* xr = x + (int64_t)in.row * cols;
  const T* rr = res ? res + (int64_t)in.row * cols : nullptr;
  T* ro = res_out ? res_out + (int64_t)row * cols : nullptr;
  float s = 0.f, ss = 0.f;
  for (int c = lane * 8; c < cols; c += 512) {
    float v[8];
    Vec8<T>::load(xr + c, v);
    if (rr) {
      float r[8];
      Vec8<T>::load(rr + c, r);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = to_f(from_f<T>(v[j] + r[j]));
    }
    if constexpr (PICK == 2) {
      if (!in.ok)
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = NAN;
    }
    if (ro && (PICK == 2 || rr)) Vec8<T>::store(ro + c, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      s += v[j];
      ss += v[j] * v[j];
    }
  }
  s = wave_sum(s);
  ss = wave_sum(ss);
  const float mean = LN ? s / cols : 0.f;
  const float var = LN ? fmaxf(ss / cols - mean * mean, 0.f) : ss / cols;
  const float rstd = in.ok ? rsqrtf(var + eps) : NAN;
  T* yr = y + (int64_t)row * cols;
  for (int c = lane * 8; c < cols; c += 512) {
    float v[8], wv[8], o[8];
    Vec8<T>::load(xr + c, v);
    if (rr) {
      float r[8];
      Vec8<T>::load(rr + c, r);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = to_f(from_f<T>(v[j] + r[j]));
    }
    Vec8<WT>::load(w + c, wv);
    float bv[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (LN && b) Vec8<WT>::load(b + c, bv);
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (v[j] - mean) * rstd * wv[j] + bv[j];
    Vec8<T>::store(yr + c, o);
  }
  if (PICK != 2 && lane == 0) {
    stat_rstd[row] = rstd;
    if (LN) stat_mean[row] = mean;
  }
}

// ---------------------------------------------------------------------------------
// backward:  h = norm input (after the fused residual add), dy = dL/dy,
//            dres = gradient arriving at h through the residual stream (optional).
// dx = rstd * (w*dy - xhat * mean(w*dy*xhat) [- mean(w*dy) for LN]) + dres
// dw_part[block] = sum_rows dy * xhat ; db_part[block] = sum_rows dy
// ---------------------------------------------------------------------------------
template <typename T, typename WT, int NV, bool LN>
__global__ __launch_bounds__(256) void norm_bwd_kernel(const T* __restrict__ dy, const T* __restrict__ h,
                                                       const T* __restrict__ dres, const WT* __restrict__ w,
                                                       const float* __restrict__ stat_mean,
                                                       const float* __restrict__ stat_rstd, T* __restrict__ dx,
                                                       float* __restrict__ dw_part, float* __restrict__ db_part,
                                                       int rows, int cols) {
  typedef T vec8 __attribute__((ext_vector_type(8)));
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  float accw[NV][8], accb[LN ? NV : 1][8];
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) accw[i][j] = 0.f;
#pragma unroll
  for (int i = 0; i < (LN ? NV : 1); ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) accb[i][j] = 0.f;

  for (int row = blockIdx.x * kRowsPerBlock + wid; row < rows; row += gridDim.x * kRowsPerBlock) {
    const int64_t base = (int64_t)row * cols;
    const float rstd = stat_rstd[row];
    const float mean = LN ? stat_mean[row] : 0.f;
    vec8 hv[NV], dv[NV], rv[NV];  // packed in the activation dtype: 4 VGPRs per vector for bf16
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = (i * 64 + lane) * 8;
      hv[i] = *reinterpret_cast<const vec8*>(h + base + c);
      dv[i] = *reinterpret_cast<const vec8*>(dy + base + c);
    }
    // the residual gradient is issued with the row's other loads, so its latency hides behind the reduction
    if (dres != nullptr) {
#pragma unroll
      for (int i = 0; i < NV; ++i) rv[i] = *reinterpret_cast<const vec8*>(dres + base + (i * 64 + lane) * 8);
    }
    float sum_gx = 0.f, sum_g = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      float wv[8];
      Vec8<WT>::load(w + (i * 64 + lane) * 8, wv);  // L1/L2 resident across rows
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float xh = (to_f(hv[i][j]) - mean) * rstd;
        const float d = to_f(dv[i][j]);
        const float g = d * wv[j];
        sum_gx += g * xh;
        sum_g += g;
        accw[i][j] += d * xh;
        if constexpr (LN) accb[i][j] += d;
      }
    }
    sum_gx = wave_sum(sum_gx) / (float)cols;
    if (LN) sum_g = wave_sum(sum_g) / (float)cols;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = (i * 64 + lane) * 8;
      float wv[8], o[8];
      Vec8<WT>::load(w + c, wv);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float xh = (to_f(hv[i][j]) - mean) * rstd;
        const float g = to_f(dv[i][j]) * wv[j];
        const float d = rstd * (g - xh * sum_gx - (LN ? sum_g : 0.f));
        o[j] = d + (dres != nullptr ? to_f(rv[i][j]) : 0.f);
      }
      Vec8<T>::store(dx + base + c, o);
    }
  }
  // block reduction of the weight-gradient partials through LDS (one fp32 row per block)
  __shared__ float red[kRowsPerBlock][512];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
#pragma unroll
    for (int j = 0; j < 8; ++j) red[wid][lane * 8 + j] = accw[i][j];
    __syncthreads();
    for (int e = threadIdx.x; e < 512; e += 256) {
      const int col = i * 512 + (e / 8) * 8 + (e % 8);  // = i*512 + e
      dw_part[(int64_t)blockIdx.x * cols + col] = red[0][e] + red[1][e] + red[2][e] + red[3][e];
    }
    __syncthreads();
    if constexpr (LN) {
#pragma unroll
      for (int j = 0; j < 8; ++j) red[wid][lane * 8 + j] = accb[i][j];
      __syncthreads();
      for (int e = threadIdx.x; e < 512; e += 256)
        db_part[(int64_t)blockIdx.x * cols + i * 512 + e] = red[0][e] + red[1][e] + red[2][e] + red[3][e];
      __syncthreads();
    }
  }
}

// generic-width backward: per-row two passes, partial weight grads via atomics into
// the block's own partial row (no cross-block contention; order fixed per block).
template <typename T, typename WT, bool LN>
__global__ __launch_bounds__(256) void norm_bwd_generic(const T* __restrict__ dy, const T* __restrict__ h,
                                                        const T* __restrict__ dres, const WT* __restrict__ w,
                                                        const float* __restrict__ stat_mean,
                                                        const float* __restrict__ stat_rstd, T* __restrict__ dx,
                                                        float* __restrict__ dw_part, float* __restrict__ db_part,
                                                        int rows, int cols) {
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  // zero this block's partial rows
  for (int c = threadIdx.x; c < cols; c += 256) {
    dw_part[(int64_t)blockIdx.x * cols + c] = 0.f;
    if (LN) db_part[(int64_t)blockIdx.x * cols + c] = 0.f;
  }
  __syncthreads();
  for (int row = blockIdx.x * kRowsPerBlock + wid; row < rows; row += gridDim.x * kRowsPerBlock) {
    const int64_t base = (int64_t)row * cols;
    const float rstd = stat_rstd[row];
    const float mean = LN ? stat_mean[row] : 0.f;
    float sgx = 0.f, sg = 0.f;
    for (int c = lane * 8; c < cols; c += 512) {
      float hv[8], dv[8], wv[8];
      Vec8<T>::load(h + base + c, hv);
      Vec8<T>::load(dy + base + c, dv);
      Vec8<WT>::load(w + c, wv);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float xh = (hv[j] - mean) * rstd;
        const float g = dv[j] * wv[j];
        sgx += g * xh;
        sg += g;
        atomicAdd(&dw_part[(int64_t)blockIdx.x * cols + c + j], dv[j] * xh);
        if (LN) atomicAdd(&db_part[(int64_t)blockIdx.x * cols + c + j], dv[j]);
      }
    }
    sgx = wave_sum(sgx) / cols;
    sg = LN ? wave_sum(sg) / cols : 0.f;
    for (int c = lane * 8; c < cols; c += 512) {
      float hv[8], dv[8], wv[8], o[8], dr[8];
      Vec8<T>::load(h + base + c, hv);
      Vec8<T>::load(dy + base + c, dv);
      Vec8<WT>::load(w + c, wv);
      if (dres) Vec8<T>::load(dres + base + c, dr);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float xh = (hv[j] - mean) * rstd;
        o[j] = rstd * (dv[j] * wv[j] - xh * sgx - sg) + (dres ? dr[j] : 0.f);
      }
      Vec8<T>::store(dx + base + c, o);
    }
  }
}

// partial [nparts, cols] fp32 -> out[cols] (dtype WT), optionally accumulated into out.
// Bound by its round trips to memory: 32 columns x 32 part groups a workgroup (a wave reads two rows of 128 B), a thread's up
// to 16 parts all on their way. 512 parts of 4096: 33 -> 4.7 us, 255 of 2048: 20.5 -> below 5 (64 columns x 4 groups, 64 or 32
// workgroups whose threads walked 128 parts).
template <typename WT>
__global__ __launch_bounds__(1024) void reduce_parts_kernel(const float* __restrict__ part, WT* __restrict__ out,
                                                            int nparts, int cols, int accumulate) {
  __shared__ float red[16][32];
  constexpr int U = 16, G = 32;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int c = blockIdx.x * 32 + (lane & 31), pg = 2 * wid + (lane >> 5);
  float s = 0.f;
  if (c < cols)
    for (int p = pg; p < nparts; p += U * G) {
      float v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = p + u * G < nparts ? part[(int64_t)(p + u * G) * cols + c] : 0.f;
#pragma unroll
      for (int u = 0; u < U; ++u) s += v[u];
    }
  s += __shfl_xor(s, 32, 64);
  if (lane < 32) red[wid][lane] = s;
  __syncthreads();
  if (threadIdx.x >= 32 || c >= cols) return;
  float t = 0.f;
#pragma unroll
  for (int k = 0; k < 16; ++k) t += red[k][lane];
  if (accumulate) t += to_f(out[c]);
  out[c] = from_f<WT>(t);
}

template <typename T, typename WT, bool LN, int PICK>
hipError_t launch_fwd_rows(const void* x, const void* res, void* res_out, const void* w, const void* b, void* y,
                           float* mean, float* rstd, int rows, int cols, float eps, const int* pick, int n_in,
                           hipStream_t st) {
  auto args = [&](auto kern, int wpr) {
    hipLaunchKernelGGL(kern, dim3((rows * wpr + kRowsPerBlock - 1) / kRowsPerBlock), dim3(256), 0, st, (const T*)x,
                       (const T*)res, (T*)res_out, (const WT*)w, (const WT*)b, (T*)y, mean, rstd, rows, cols, eps, pick, n_in);
  };
  // Several waves a row up to 64 rows (1,024 rows 4.0 / 6.4 / 11.2 -> 3.6 / 5.5 / 10.9 us, 8,192 19.9 / 42 / 103 -> 20.5 / 39 /
  // 93): longer steps, the training ones among them, keep the sums of one wave in their order.
#define HDS_NF(COLS, NV, WPR)                                              \
  case COLS:                                                               \
    if (rows <= kFewRows) args(norm_fwd_kernel<T, WT, NV, LN, WPR, PICK == 2 ? 2 : 1>, WPR); \
    else args(norm_fwd_kernel<T, WT, NV, LN, 1, PICK>, 1);                 \
    break
  switch (cols) {
    case 512: args(norm_fwd_kernel<T, WT, 1, LN, 1, PICK>, 1); break;
    HDS_NF(1024, 2, 2);
    HDS_NF(2048, 4, 4);
    HDS_NF(3072, 6, 2);
    HDS_NF(4096, 8, 4);
    HDS_NF(5120, 10, 2);
    HDS_NF(6144, 12, 4);
    HDS_NF(8192, 16, 4);
    default: args(norm_fwd_generic<T, WT, LN, PICK>, 1); break;
  }
#undef HDS_NF
  return hipGetLastError();
}

template <typename T, typename WT, bool LN>
hipError_t launch_fwd(const void* x, const void* res, void* res_out, const void* w, const void* b, void* y,
                      float* mean, float* rstd, int rows, int cols, float eps, const int* pick, int n_in,
                      hipStream_t st) {
  if (pick != nullptr)
    return launch_fwd_rows<T, WT, LN, 1>(x, res, res_out, w, b, y, mean, rstd, rows, cols, eps, pick, n_in, st);
  return launch_fwd_rows<T, WT, LN, 0>(x, res, res_out, w, b, y, mean, rstd, rows, cols, eps, pick, n_in, st);
}

template <typename T, typename WT, bool LN>
hipError_t launch_bwd(const void* dy, const void* h, const void* dres, const void* w, const float* mean,
                      const float* rstd, void* dx, float* dw_part, float* db_part, int nparts, void* dw, void* db,
                      int accumulate, int rows, int cols, hipStream_t st) {
  dim3 grid(nparts), block(256);
  auto args = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, block, 0, st, (const T*)dy, (const T*)h, (const T*)dres, (const WT*)w, mean,
                       rstd, (T*)dx, dw_part, db_part, rows, cols);
  };
  switch (cols) {
    case 512: args(norm_bwd_kernel<T, WT, 1, LN>); break;
    case 1024: args(norm_bwd_kernel<T, WT, 2, LN>); break;
    case 2048: args(norm_bwd_kernel<T, WT, 4, LN>); break;
    case 3072: args(norm_bwd_kernel<T, WT, 6, LN>); break;
    case 4096: args(norm_bwd_kernel<T, WT, 8, LN>); break;
    case 5120: args(norm_bwd_kernel<T, WT, 10, LN>); break;
    case 6144: args(norm_bwd_kernel<T, WT, 12, LN>); break;
    case 8192: args(norm_bwd_kernel<T, WT, 16, LN>); break;
    default: args(norm_bwd_generic<T, WT, LN>); break;
  }
  dim3 rg((cols + 31) / 32), rb(1024);
  if (dw) hipLaunchKernelGGL(reduce_parts_kernel<WT>, rg, rb, 0, st, dw_part, (WT*)dw, nparts, cols, accumulate);
  if (LN && db) hipLaunchKernelGGL(reduce_parts_kernel<WT>, rg, rb, 0, st, db_part, (WT*)db, nparts, cols, accumulate);
  return hipGetLastError();
}

}  // namespace

// dtype: activation dtype code; wdtype: weight dtype code (DType enum)
#define HDS_DISPATCH2(dtype, wdtype, LN, FN, ...)                                              \
  do {                                                                                         \
    if (dtype == kBF16 && wdtype == kBF16) return FN<bf16, bf16, LN>(__VA_ARGS__);             \
    if (dtype == kBF16 && wdtype == kF32) return FN<bf16, float, LN>(__VA_ARGS__);             \
    if (dtype == kF32 && wdtype == kF32) return FN<float, float, LN>(__VA_ARGS__);             \
    if (dtype == kF16 && wdtype == kF16) return FN<_Float16, _Float16, LN>(__VA_ARGS__);       \
    if (dtype == kF16 && wdtype == kF32) return FN<_Float16, float, LN>(__VA_ARGS__);          \
    return hipErrorInvalidValue;                                                               \
  } while (0)

HDS_EXPORT int hds_norm_fwd(int is_ln, int dtype, int wdtype, const void* x, const void* res, void* res_out,
                            const void* w, const void* b, void* y, float* mean, float* rstd, int rows, int cols,
                            float eps, const int* pick, int n_in, hipStream_t st) {
  if (cols % 8 || (pick != nullptr && n_in < 1)) return hipErrorInvalidValue;
  if (is_ln)
    HDS_DISPATCH2(dtype, wdtype, true, launch_fwd, x, res, res_out, w, b, y, mean, rstd, rows, cols, eps, pick, n_in, st);
  HDS_DISPATCH2(dtype, wdtype, false, launch_fwd, x, res, res_out, w, b, y, mean, rstd, rows, cols, eps, pick, n_in, st);
}

// y[i] = RMSNorm(table[ids[i]]) * w and h[i] = table[ids[i]]; table [n_rows, cols]
HDS_EXPORT int hds_embed_norm(int dtype, const void* table, const int64_t* ids, const void* w, void* h, void* y, int n,
                              int cols, int n_rows, float eps, hipStream_t st) {
  if (n < 0 || cols < 8 || cols % 8 || n_rows < 1) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  auto go = [&](auto t) {
    using T = decltype(t);
    return launch_fwd_rows<T, T, false, 2>(table, nullptr, h, w, nullptr, y, nullptr, nullptr, n, cols, eps, (const int*)ids,
                                           n_rows, st);
  };
  if (dtype == kBF16) return go(bf16{});
  if (dtype == kF32) return go(0.f);
  if (dtype == kF16) return go((_Float16)0.f);
  return hipErrorInvalidValue;
}

static int g_norm_bwd_max_parts = 512;

// cap on the backward's workgroups = fp32 weight-gradient partial rows (A/B knob; 512 = 8 waves per CU)
HDS_EXPORT int hds_norm_bwd_set_max_parts(int n) {
  if (n < 1 || n > 8192) return hipErrorInvalidValue;
  g_norm_bwd_max_parts = n;
  return 0;
}

HDS_EXPORT int hds_norm_bwd_nparts(int rows) {
  int n = (rows + kRowsPerBlock - 1) / kRowsPerBlock;
  return n < g_norm_bwd_max_parts ? (n < 1 ? 1 : n) : g_norm_bwd_max_parts;
}

HDS_EXPORT int hds_norm_bwd(int is_ln, int dtype, int wdtype, const void* dy, const void* h, const void* dres,
                            const void* w, const float* mean, const float* rstd, void* dx, float* dw_part,
                            float* db_part, int nparts, void* dw, void* db, int accumulate, int rows, int cols,
                            hipStream_t st) {
  if (cols % 8) return hipErrorInvalidValue;
  if (is_ln)
    HDS_DISPATCH2(dtype, wdtype, true, launch_bwd, dy, h, dres, w, mean, rstd, dx, dw_part, db_part, nparts, dw, db,
                  accumulate, rows, cols, st);
  HDS_DISPATCH2(dtype, wdtype, false, launch_bwd, dy, h, dres, w, mean, rstd, dx, dw_part, db_part, nparts, dw, db,
                accumulate, rows, cols, st);
}
