// Weight-only codes as matrix operands (wmix_gemm.hip, linear_packed.hip): a lane's 32 consecutive k of a packed weight row.
#pragma once
#include "hds_common.h"

namespace {

using namespace hds;

enum WFmt : int { kInt8 = 0, kInt4 = 1, kFp6 = 2 };

template <int FMT> struct WRaw;
template <> struct WRaw<kInt8> { uint4 a, b; };
template <> struct WRaw<kInt4> { uint4 a; };
template <> struct WRaw<kFp6> { uint2 a, b, c; };

// The codes as bf16, which holds them exactly (int4: kUnit times the result). fp6 codes become bf16 in one instruction for 32 of
// them, int8 and int4 in one and a half and two a code.
typedef uint32_t u32x6 __attribute__((ext_vector_type(6)));
typedef __bf16 bf16x32 __attribute__((ext_vector_type(32)));

template <int FMT>
constexpr float kUnit = FMT == kInt4 ? 0.0625f : 1.f;

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
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) f[i >> 1][4 * (i & 1) + t] = (bf16)(float)(int8_t)(dw[i] >> (8 * t));
  } else {
    const uint32_t dw[4] = {r.a.x, r.a.y, r.a.z, r.a.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // in the upper halves of bytes, with their sign: 16 times the code (kUnit)
      const uint32_t lo = (dw[i] << 4) & 0xf0f0f0f0u, hi = dw[i] & 0xf0f0f0f0u;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        f[i][2 * t] = (bf16)(float)(int8_t)(lo >> (8 * t));
        f[i][2 * t + 1] = (bf16)(float)(int8_t)(hi >> (8 * t));
      }
    }
  }
}

}  // namespace
