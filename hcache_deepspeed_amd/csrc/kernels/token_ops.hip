// Token-routing kernels for random layerwise token dropping (random-LTD) and channels-last bias fusions for
// diffusion UNet / VAE blocks.
//
// Capability parity:
//   * csrc/random_ltd/{gather_scatter.cu,token_sort.cu,slice_attn_masks.cu}:
//     token_sort_ (sort the sampled indices of every (layer, batch) row), token_gather / token_scatter
//     ([B, S, H] <-> [B, R, H] rows), slice_gpt_mask / slice_bert_mask.
//   * csrc/spatial/csrc/opt_bias_add.cu (N19): nhwc_bias_add, nhwc_bias_add_add, nhwc_bias_add_bias_add.
// Design: every row moves with 16-byte vectors (8 x bf16 per lane); the sort is one LDS bitonic network per row
// (a workgroup per row, up to 16384 keys = 64 KB of the 160 KB LDS); mask slicing gathers rows and columns in one
// pass. All are bandwidth kernels, so the grids have one workgroup per row (B * R >> 256 for real shapes).
#include "hds_common.h"

using namespace hds;

namespace {

// out[b, r, :] = x[b, idx[b, r], :]   (x: [B, S, H], idx: [B, R] int32)
template <typename T>
__global__ __launch_bounds__(256) void token_gather_kernel(const T* __restrict__ x, const int* __restrict__ idx,
                                                           T* __restrict__ out, int S, int R, int H) {
  const int row = blockIdx.x;  // b * R + r
  const int b = row / R;
  const int s = idx[row];
  if (s < 0 || s >= S) return;
  const T* src = x + ((int64_t)b * S + s) * H;
  T* dst = out + (int64_t)row * H;
  for (int c = threadIdx.x * 8; c < H; c += 256 * 8) {
    float v[8];
    Vec8<T>::load(src + c, v);
    Vec8<T>::store(dst + c, v);
  }
}

// Rows of a table by 64-bit ids, as bytes (an embedding lookup): one 16-byte access a thread, a row's accesses spread over
// blockIdx.y. An id outside the table gives a row of set bits, which are NaNs. Latency bound: 16 rows of 8 KB
// 13.2 us with torch's small-index kernel, 4.4 us here.
__global__ __launch_bounds__(256) void gather_rows_kernel(const u32x4* __restrict__ table,
                                                          const int64_t* __restrict__ ids, u32x4* __restrict__ out,
                                                          int64_t n_rows, int64_t chunks) {
  const int64_t c = (int64_t)blockIdx.y * 256 + threadIdx.x;
  if (c >= chunks) return;
  const int64_t id = ids[blockIdx.x];
  const u32x4 none = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu};
  out[blockIdx.x * chunks + c] = id >= 0 && id < n_rows ? table[id * chunks + c] : none;
}

// out[b, idx[b, r], :] = part[b, r, :]   (out already holds the full [B, S, H] input)
template <typename T>
__global__ __launch_bounds__(256) void token_scatter_kernel(const T* __restrict__ part, const int* __restrict__ idx,
                                                            T* __restrict__ out, int S, int R, int H) {
  const int row = blockIdx.x;
  const int b = row / R;
  const int s = idx[row];
  if (s < 0 || s >= S) return;
  const T* src = part + (int64_t)row * H;
  T* dst = out + ((int64_t)b * S + s) * H;
  for (int c = threadIdx.x * 8; c < H; c += 256 * 8) {
    float v[8];
    Vec8<T>::load(src + c, v);
    Vec8<T>::store(dst + c, v);
  }
}

// Ascending in-place sort of each row of `keys` [rows, n] (n <= 16384) with an LDS bitonic network.
__global__ __launch_bounds__(1024) void token_sort_kernel(int* __restrict__ keys, int n, int npow2) {
  extern __shared__ int sk[];
  int* row = keys + (int64_t)blockIdx.x * n;
  for (int i = threadIdx.x; i < npow2; i += blockDim.x) sk[i] = i < n ? row[i] : 0x7fffffff;
  __syncthreads();
  for (int k = 2; k <= npow2; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < npow2; i += blockDim.x) {
        const int p = i ^ j;
        if (p > i) {
          const int a = sk[i], c = sk[p];
          const bool up = (i & k) == 0;
          if ((a > c) == up) {
            sk[i] = c;
            sk[p] = a;
          }
        }
      }
      __syncthreads();
    }
  }
  for (int i = threadIdx.x; i < n; i += blockDim.x) row[i] = sk[i];
}

// out[l, b, i, j] = mask[b', idx[l, b, i], idx[l, b, j]]  (mask [Bm, S, S], Bm in {1, B}; out [L, B, R, R])
template <typename T>
__global__ __launch_bounds__(256) void slice_mask_kernel(const T* __restrict__ mask, const int* __restrict__ idx,
                                                         T* __restrict__ out, int B, int Bm, int S, int R) {
  const int row = blockIdx.x;  // (l * B + b) * R + i
  const int lb = row / R, i = row - lb * R;
  const int b = lb % B;
  const int* ix = idx + (int64_t)lb * R;
  const T* src = mask + ((int64_t)(Bm == 1 ? 0 : b) * S + ix[i]) * S;
  T* dst = out + (int64_t)row * R;
  for (int j = threadIdx.x; j < R; j += 256) dst[j] = src[ix[j]];
}

// Channels-last bias fusions over [N*H*W, C] rows (C % 8 == 0):
//   mode 0: out = a + bias;  mode 1: out = a + bias + other;  mode 2: out = a + bias + other + other_bias
template <typename T>
__global__ __launch_bounds__(256) void nhwc_bias_add_kernel(const T* __restrict__ a, const T* __restrict__ bias,
                                                            const T* __restrict__ other,
                                                            const T* __restrict__ other_bias, T* __restrict__ out,
                                                            int64_t n_vec, int C, int mode) {
  const int cv = C / 8;
  for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < n_vec; v += (int64_t)gridDim.x * 256) {
    const int c = (int)(v % cv) * 8;
    float x[8], bb[8];
    Vec8<T>::load(a + v * 8, x);
    Vec8<T>::load(bias + c, bb);
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] += bb[i];
    if (mode >= 1) {
      float o[8];
      Vec8<T>::load(other + v * 8, o);
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] += o[i];
    }
    if (mode == 2) {
      float ob[8];
      Vec8<T>::load(other_bias + c, ob);
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] += ob[i];
    }
    Vec8<T>::store(out + v * 8, x);
  }
}

// Embedding weight gradient, accumulated in place: grad[id, :] += sum of dy[t, :] over tokens t with ids[t] == id.
// ``sorted``/``perm`` come from a stable sort of the ids, so every id's tokens are one contiguous run and the
// first position of each run owns the row: one read-modify-write per touched row, fp32 sums in a fixed
// (token) order -- deterministic, no atomics, and no dense [V, D] temporary (the sort-based framework path
// materialises and then adds one). One workgroup per sorted position; non-leading positions exit at once.
template <typename T>
__global__ __launch_bounds__(256) void embed_bwd_kernel(const T* __restrict__ dy, const int64_t* __restrict__ sorted,
                                                        const int64_t* __restrict__ perm, T* __restrict__ grad,
                                                        int64_t n, int D, int64_t V, int64_t pad_idx) {
  const int64_t i = blockIdx.x;
  const int64_t id = sorted[i];
  if ((i > 0 && sorted[i - 1] == id) || id == pad_idx || id < 0 || id >= V) return;
  int64_t end = i + 1;
  while (end < n && sorted[end] == id) ++end;
  T* g = grad + id * (int64_t)D;
  for (int c = threadIdx.x * 8; c < D; c += 256 * 8) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int64_t j = i; j < end; ++j) {
      float v[8];
      Vec8<T>::load(dy + perm[j] * (int64_t)D + c, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += v[e];
    }
    float old[8];
    Vec8<T>::load(g + c, old);
#pragma unroll
    for (int e = 0; e < 8; ++e) old[e] += acc[e];
    Vec8<T>::store(g + c, old);
  }
}

// The same without sorting, for few ids: the workgroup of every position compares its id with all of them, 64 a wave, and goes on
// where no earlier one is the same. What bounds short steps' sorts is their launches and a workgroup's passes over the digits.
// Sort and kernel above -> this, rows of 2,048, launch by launch: 64 / 1,018 / 2,046 / 3,000 / 4,096 ids 30.0 / 35.1 / 41.1 /
// 53.6 / 56.2 -> 8.6 / 9.6 / 9.2 / 13.6 / 21.0 us; beyond, the comparisons grow with the square. Rows of one id are added in their order,
// kAtOnce of them on their way: 4,096 ids, half of them one 867 -> 279 (row by row 606), 1,018, three in ten 105 -> 30 (52).
constexpr int kFewIds = 4096;  // (a lane for each 64)
constexpr int kAtOnce = 8;     // rows on their way: an id of padding may be half of all

template <typename T>
__global__ __launch_bounds__(256) void embed_bwd_few_kernel(const T* __restrict__ dy, const int64_t* __restrict__ ids,
                                                            T* __restrict__ grad, int n, int D, int64_t V, int64_t pad_idx) {
  __shared__ uint64_t same[kFewIds / 64];
  __shared__ uint16_t list[kFewIds];
  const int i = blockIdx.x, words = (n + 63) / 64, w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t id = ids[i];
  if (id == pad_idx || id < 0 || id >= V) return;
#pragma unroll 4
  for (int k = w; k < words; k += 4) {
    const int j = 64 * k + lane;
    const uint64_t m = __ballot(j < n && ids[min(j, n - 1)] == id);
    if (lane == 0) same[k] = m;
  }
  __syncthreads();
  // every wave for itself, a lane a word: is an earlier position's id the same, how many are
  uint64_t m = lane < words ? same[lane] : 0;
  const uint64_t earlier = lane < i / 64 ? m : lane == i / 64 ? m & ((1ull << (i % 64)) - 1) : 0;
  if (__any(earlier != 0)) return;
  int upto = __popcll(m);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(upto, o, 64);
    if (lane >= o) upto += v;
  }
  const int count = __shfl(upto, 63, 64);
  if (count > 1) {
    if (w == 0)
      for (int p = upto - __popcll(m); m != 0; m &= m - 1) list[p++] = (uint16_t)(64 * lane + __builtin_ctzll(m));
    __syncthreads();
  }
  T* g = grad + id * (int64_t)D;
  for (int c = threadIdx.x * 8; c < D; c += 256 * 8) {
    float acc[8], old[8];
    Vec8<T>::load(g + c, old);
    Vec8<T>::load(dy + i * (int64_t)D + c, acc);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += 0.f;
    for (int p = 1; p < count; p += kAtOnce) {
      float v[kAtOnce][8];
#pragma unroll
      for (int u = 0; u < kAtOnce; ++u) Vec8<T>::load(dy + list[min(p + u, count - 1)] * (int64_t)D + c, v[u]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < kAtOnce; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = p + u < count ? acc[e] + v[u][e] : acc[e];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) old[e] += acc[e];
    Vec8<T>::store(g + c, old);
  }
}

#define HDS_TOK_DISPATCH(dtype, ...)                  \
  switch (dtype) {                                    \
    case kF32: { typedef float T; __VA_ARGS__; break; }    \
    case kBF16: { typedef bf16 T; __VA_ARGS__; break; }    \
    case kF16: { typedef _Float16 T; __VA_ARGS__; break; } \
    default: return (int)hipErrorInvalidValue;       \
  }

}  // namespace

HDS_EXPORT int hds_token_gather(int dtype, const void* x, const int* idx, void* out, int B, int S, int R, int H,
                                hipStream_t st) {
  if (H % 8 || B <= 0 || R <= 0) return (int)hipErrorInvalidValue;
  HDS_TOK_DISPATCH(dtype, hipLaunchKernelGGL(token_gather_kernel<T>, dim3(B * R), dim3(256), 0, st,
                                             (const T*)x, idx, (T*)out, S, R, H));
  return (int)hipGetLastError();
}

// table [n_rows, row_bytes] and out [n, row_bytes] with 16-byte rows
HDS_EXPORT int hds_gather_rows(const void* table, const int64_t* ids, void* out, int n, int64_t row_bytes,
                               int64_t n_rows, hipStream_t st) {
  if (n <= 0) return 0;
  const int64_t chunks = row_bytes / 16, cols = (chunks + 255) / 256;
  if (row_bytes < 16 || row_bytes % 16 || cols > 65535) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(gather_rows_kernel, dim3(n, (int)cols), dim3(256), 0, st, (const u32x4*)table, ids, (u32x4*)out,
                     n_rows, chunks);
  return (int)hipGetLastError();
}

HDS_EXPORT int hds_token_scatter(int dtype, const void* part, const int* idx, void* out, int B, int S, int R, int H,
                                 hipStream_t st) {
  if (H % 8 || B <= 0 || R <= 0) return (int)hipErrorInvalidValue;
  HDS_TOK_DISPATCH(dtype, hipLaunchKernelGGL(token_scatter_kernel<T>, dim3(B * R), dim3(256), 0, st,
                                             (const T*)part, idx, (T*)out, S, R, H));
  return (int)hipGetLastError();
}

HDS_EXPORT int hds_token_sort(int* keys, int rows, int n, hipStream_t st) {
  if (n <= 0 || n > 16384 || rows <= 0) return (int)hipErrorInvalidValue;
  int p = 1;
  while (p < n) p <<= 1;
  const int nt = p < 1024 ? (p < 64 ? 64 : p) : 1024;
  hipLaunchKernelGGL(token_sort_kernel, dim3(rows), dim3(nt), p * sizeof(int), st, keys, n, p);
  return (int)hipGetLastError();
}

HDS_EXPORT int hds_slice_mask(int dtype, const void* mask, const int* idx, void* out, int L, int B, int Bm, int S,
                              int R, hipStream_t st) {
  if (L <= 0 || B <= 0 || R <= 0 || (Bm != 1 && Bm != B)) return (int)hipErrorInvalidValue;
  HDS_TOK_DISPATCH(dtype, hipLaunchKernelGGL(slice_mask_kernel<T>, dim3(L * B * R), dim3(256), 0, st,
                                             (const T*)mask, idx, (T*)out, B, Bm, S, R));
  return (int)hipGetLastError();
}

HDS_EXPORT int hds_nhwc_bias_add(int dtype, const void* a, const void* bias, const void* other, const void* other_bias,
                                 void* out, int64_t rows, int C, int mode, hipStream_t st) {
  if (C % 8 || rows <= 0 || mode < 0 || mode > 2) return (int)hipErrorInvalidValue;
  const int64_t n_vec = rows * (C / 8);
  const int64_t want = (n_vec + 255) / 256;
  const int grid = (int)(want < 256 * 32 ? want : 256 * 32);
  HDS_TOK_DISPATCH(dtype, hipLaunchKernelGGL(nhwc_bias_add_kernel<T>, dim3(grid), dim3(256), 0, st, (const T*)a,
                                             (const T*)bias, (const T*)other, (const T*)other_bias, (T*)out, n_vec,
                                             C, mode));
  return (int)hipGetLastError();
}

HDS_EXPORT int hds_embed_bwd(int dtype, const void* dy, const int64_t* sorted, const int64_t* perm, void* grad,
                             int64_t n, int D, int64_t V, int64_t pad_idx, hipStream_t st) {
  if (n <= 0) return 0;
  if (D % 8 || n > 0x7fffffff) return (int)hipErrorInvalidValue;
  HDS_TOK_DISPATCH(dtype, hipLaunchKernelGGL(embed_bwd_kernel<T>, dim3((unsigned)n), dim3(256), 0, st, (const T*)dy,
                                             sorted, perm, (T*)grad, n, D, V, pad_idx));
  return (int)hipGetLastError();
}

// ids [n] as they come, of at most hds_embed_bwd_few_max()
HDS_EXPORT int hds_embed_bwd_few(int dtype, const void* dy, const int64_t* ids, void* grad, int n, int D, int64_t V,
                                 int64_t pad_idx, hipStream_t st) {
  if (n <= 0) return 0;
  if (D % 8 || n > kFewIds) return (int)hipErrorInvalidValue;
  HDS_TOK_DISPATCH(dtype, hipLaunchKernelGGL(embed_bwd_few_kernel<T>, dim3(n), dim3(256), 0, st, (const T*)dy, ids, (T*)grad,
                                             n, D, V, pad_idx));
  return (int)hipGetLastError();
}

HDS_EXPORT int hds_embed_bwd_few_max() { return kFewIds; }
