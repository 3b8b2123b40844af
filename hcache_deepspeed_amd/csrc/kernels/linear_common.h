// What the products of many rows share (linear.hip, linear_packed.hip): the matrix instruction, LDS-DMA through a buffer
// descriptor, the gated unit and the sum of slices.
#pragma once
#include "attn_common.h"

namespace {

using namespace hds;
using namespace hds::attn;

// gated unit, by the codes of act.hip: 0 silu, 1 gelu_tanh, 2 relu; the projections rounded as a kernel of its own reads them
__device__ __forceinline__ bf16 gated(float g, float u, int act) {
  const float v = (float)(bf16)g;
  float a;
  if (act == 2) a = fmaxf(v, 0.f);
  else if (act == 1) a = 0.5f * v * (1.f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
  else a = v * __builtin_amdgcn_rcpf(1.f + __expf(-v));
  return (bf16)(a * (float)(bf16)u);
}

__device__ __forceinline__ f32x4 mfma16(const bf16x8& a, const bf16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// 16 or 4 bytes a lane from `base` + voff + soff into LDS, lane after lane; zeros from `bytes` on. NT: past the caches
template <bool NT>
__device__ __forceinline__ void load_lds(const void* base, uint32_t bytes, char* lds, uint32_t voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, bytes, 0x00020000),
                                           (lds_void*)lds, 16, voff, soff, 0, NT ? 2 : 0);
}
__device__ __forceinline__ void load_lds_4(const void* base, uint32_t bytes, char* lds, uint32_t voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, bytes, 0x00020000),
                                           (lds_void*)lds, 4, voff, 0, 0, 0);
}

struct SumArgs {
  const float* part;  // [S, M, N] (gated: [S, M, 2N])
  const bf16* bias;  // or null
  bf16* y;  // [M, ldy]
  int64_t ldy;
  int M, N, S, act;
};

// y = sum over the S parts, in their order; N % 4 == 0
template <bool GLU>
__global__ __launch_bounds__(256) void linear_sum_kernel(SumArgs p) {
  const int i = blockIdx.x * 256 + threadIdx.x, quads = p.N / 4;
  if (i >= p.M * quads) return;
  const int m = i / quads, c = 4 * (i - m * quads), width = GLU ? 2 * p.N : p.N;
  const float* src = p.part + (int64_t)m * width + c;
  f32x4 v[GLU ? 2 : 1];
#pragma unroll
  for (int h = 0; h < (GLU ? 2 : 1); ++h) {
    v[h] = *reinterpret_cast<const f32x4*>(src + h * p.N);
    for (int s = 1; s < p.S; ++s) v[h] += *reinterpret_cast<const f32x4*>(src + h * p.N + (int64_t)s * p.M * width);
    if (p.bias != nullptr)
      for (int e = 0; e < 4; ++e) v[h][e] += (float)p.bias[h * p.N + c + e];
  }
  bf16x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = GLU ? gated(v[0][e], v[GLU ? 1 : 0][e], p.act) : (bf16)v[0][e];
  *reinterpret_cast<bf16x4*>(p.y + m * p.ldy + c) = o;
}

}  // namespace
