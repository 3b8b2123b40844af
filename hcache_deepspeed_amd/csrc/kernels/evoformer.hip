// Evoformer attention with MSA-mask and pair biases (DS4Sci_EvoformerAttention), forward and backward, gfx950.
//
// Reference parity: csrc/deepspeed4science/evoformer_attn (CUTLASS memory-efficient attention with bias). Not a
// translation.
//
// q, k, v [B, N, L, H, D]; bias1 [B, N, 1, 1, L] (mask), bias2 [B, 1, H, L, L] (pair bias, shared by the N rows), both in
// bf16 or both in fp32 and added in fp32. The sequences are short (16 to 400 positions), the heads small (32, 64), the
// rows many: the products are a few GFLOP and the inputs a few tens of MB, so the kernels are bound by the vector
// instructions between the products (exponential, differences, conversion) and by how the operands get there.
//   * forward and dQ: a wave holds 32 queries of one (b, n, h), the workgroup stages its keys and values in LDS once
//     (LDS-DMA, 32 KB a chunk, so that several workgroups share a CU). S^T = K Q^T puts the query on the lane: softmax
//     statistics are lane-local and the S^T accumulator is the B operand of the next product (acc_to_b); V^T and K^T
//     come out of the row-major tiles by transposing LDS reads. dQ also makes rowsum(dO * O), which the others read.
//   * dK / dV: the same with 32 keys on the lanes and queries and output gradients in LDS.
//   * dQ, dK and dV of rows of up to 256 positions, heads of 32 and bf16 biases: in one kernel, see evo_bwd_kernel.
//   * pair-bias gradient: the sum of dS over the N rows stays in registers. A wave owns 32 queries x 64 keys of one
//     (b, h) and walks over a chunk of the rows, recomputing the two products that dS needs; chunks are added by a second
//     kernel that also rounds. No atomics, the same result every time.
// Measured (B = 1, N = 128, L = 256, H = 8, D = 32, both biases bf16): a forward and backward 137 us (with a forward workgroup a
// row and the pair bias through the matrix cores in every row 147; with dQ and dK / dV apart and the pair gradient's rows
// loaded by wave 199); in a kernel trace, where launches do not overlap, forward 38 us (a workgroup a row 42 to 45), dQ + dK +
// dV 68 (apart 52 + 51), pair gradient 34 + 4 (bias through the matrix cores 43 + 4, rows by wave 56 + 4)
// (before: one wave a workgroup with operands from global memory and 2-byte reads of V 169 us; the FlashAttention
// backward kernels with 32-bit atomics into the pair gradient 271 + 1,585 us).
#include <algorithm>
#include <cmath>

#include "attn_common.h"

using namespace hds;
using namespace hds::attn;

namespace {

constexpr float kLog2e = 1.4426950408889634f;

// ---------------------------------------------------------------------------------------------------------------
// LDS tiles: rows of 2 D bytes whose 16-byte chunks are XOR-swizzled by the row, so that 16 lanes reading 16 rows at one
// chunk (ds_read_b128), and 16 lanes reading 32 bytes of 4 rows (ds_read_b64_tr_b16), meet every bank once
// ---------------------------------------------------------------------------------------------------------------
// most waves of a workgroup: the 128-wide accumulators want more than the 256 registers that eight leave each
template <int D>
constexpr int kWaves = D == 128 ? 4 : 8;

template <int D>
struct Tile {
  static constexpr int RB = 2 * D, CH = D / 8;       // bytes, chunks of a row
  static constexpr int ROWS = 8192 / D;              // rows of a chunk: 16 KB a matrix
  static constexpr int KS = D / 16, DT = D / 32;     // steps of a contraction over D, 32-column blocks
  static __device__ __forceinline__ int mix(int row) {
    if constexpr (D == 32) return (row >> 2) & 3;
    if constexpr (D == 64) return ((row & 2)) | ((row & 4)) | ((row >> 3) & 1);
    return swz(row);
  }
  static __device__ __forceinline__ int off(int row, int ch) { return row * RB + 16 * (ch ^ mix(row)); }

  // rows row0 .. row0 + 32 nt - 1 of a matrix [L, ld] to LDS (rows past the end: the last one)
  static __device__ __forceinline__ void stage(char* lds, const bf16* m, int64_t ld, int row0, int nt, int L, int nw) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    constexpr int PER = 1024 / RB;  // rows of one wave instruction
    for (int i = w; i < nt * 32 / PER; i += nw) {
      const int row = i * PER + lane / CH;
      const int ch = (lane % CH) ^ mix(row);
      const bf16* src = m + (int64_t)min(row0 + row, L - 1) * ld + 8 * ch;
      __builtin_amdgcn_global_load_lds((gbl_void*)src, (lds_void*)(lds + i * 1024), 16, 0, 0);
    }
  }
  // rows row0 + (lane & 31), elements 16 ks + 8 (lane >> 5) .. + 7
  static __device__ __forceinline__ bf16x8 rows(const char* lds, int row0, int ks) {
    const int lane = threadIdx.x & 63;
    return *reinterpret_cast<const bf16x8*>(lds + off(row0 + (lane & 31), 2 * ks + (lane >> 5)));
  }
  // the transposed tile: column 32 dt + (lane & 31), rows row0 + 16 s + .. in the order of acc_to_b
  static __device__ __forceinline__ bf16x8 cols(const char* lds, int row0, int s, int dt) {
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, i = lane & 15, q = i >> 2, p = i & 3;
    const int row = row0 + 16 * s + 4 * (g >> 1) + q;
    const int ch = 4 * dt + 2 * (g & 1) + (p >> 1);
    const char* a0 = lds + off(row, ch) + 8 * (p & 1);
    const char* a1 = lds + off(row + 8, ch) + 8 * (p & 1);
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(a0));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(a1));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
  // the same for both steps of a tile of 32 columns at `lds`, here when it returns
  static __device__ __forceinline__ void cols_now(const char* lds, bf16x8 (&f)[2]) {
    static_assert(D == 32, "rows of 64 bytes: 16 further ones have the same swizzle");
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, i = lane & 15, q = i >> 2, p = i & 3;
    const int row = 4 * (g >> 1) + q, ch = 2 * (g & 1) + (p >> 1);
    const uint32_t a0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)(lds + off(row, ch) + 8 * (p & 1));
    const uint32_t a1 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)(lds + off(row + 8, ch) + 8 * (p & 1));
    u32x2 r[4];
    asm volatile(
        "ds_read_b64_tr_b16 %0, %4\n\tds_read_b64_tr_b16 %1, %5\n\tds_read_b64_tr_b16 %2, %4 offset:1024\n\t"
        "ds_read_b64_tr_b16 %3, %5 offset:1024\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
        : "v"(a0), "v"(a1)
        : "memory");
#pragma unroll
    for (int st = 0; st < 2; ++st)
      f[st] = __builtin_bit_cast(bf16x8, u32x4{r[2 * st][0], r[2 * st][1], r[2 * st + 1][0], r[2 * st + 1][1]});
  }
};

// Tile::stage for a kernel that walks over rows n: nt tiles from position row0 on, at distances from the start of a row n that
// are made once. Positions past the end are read as zeros.
template <int D>
struct Stager {
  using T = Tile<D>;
  static constexpr int PER = 1024 / T::RB;
  uint32_t first, even, odd;  // of a lane: of the wave's first instruction; without its number, by that number's parity: a tile's swizzle looks as far
  int w, count, step;
  uint32_t bytes, stride;
  __device__ __forceinline__ Stager(int row0, int nt, int nw, int64_t ld, int L) {
    const int lane = threadIdx.x & 63, row = lane / T::CH;
    w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    count = nt * 32 / PER;
    step = nw;
    stride = PER * 2 * (uint32_t)ld;
    bytes = (uint32_t)(L - 1) * 2 * (uint32_t)ld + 2 * D;
    even = 2 * (uint32_t)ld * (row0 + row) + 16 * ((lane % T::CH) ^ T::mix(row));
    odd = 2 * (uint32_t)ld * (row0 + row) + 16 * ((lane % T::CH) ^ T::mix(PER + row));
    first = (w & 1 ? odd : even) + w * stride;
  }
  // The whole distance goes into the vector offset: only that is held against the range, so that positions past the end are.
  // (one: of whole workgroups that move 1 KB a wave)
  __device__ __forceinline__ void stage(char* lds, const bf16* m, bool one) const {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)m, (short)0, bytes, 0x00020000);
    const uint32_t at[2] = {even, odd};
    if (one) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)(lds + w * 1024), 16, first, 0, 0, 0);
      return;
    }
    for (int i = w; i < count; i += step) {
      uint32_t voff = at[0];
      if (i & 1) voff = at[1];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)(lds + i * 1024), 16, voff + i * stride, 0, 0, 0);
    }
  }
};

// ---------------------------------------------------------------------------------------------------------------
// biases
// ---------------------------------------------------------------------------------------------------------------
// They are added to the raw scores. The scale is rest * 2^e with rest in [0.5, 1), and a score is rest * log2(e) * (2^e q . k
// + bias / rest): the power of two goes into the operand that a wave keeps in registers and rounds nothing, and a finite
// bias of up to 1.7e38 stays finite (divided by the whole scale it would not from 3e37 on: a query whose keys are all
// masked by -1e38 has its softmax over them). bf16 biases go
// through the matrix cores, which have room: a pair bias tile times the matrix (1 / rest) I, a mask as an outer product
// with 1 / rest. 1 / rest is cut into bf16 pieces (one for D = 64, three otherwise, which make up all 24 bits), so
// that the products are exact. That takes two 16-byte loads a lane and no vector instruction a score, where unpacking
// and adding took four, and two-byte loads where keys are on the lanes (forward 53 -> 42 us, dQ 58 -> 51, dK / dV
// 124 -> 51, pair gradient 78 -> 59). Zeros of I meet other keys of the same query only: minus
// infinity is made the lowest finite value first, which 1 / rest > 1 takes back to minus infinity. fp32 biases are
// added by vector instructions.
struct __attribute__((packed, aligned(2))) Eight {  // L may be odd: rows are aligned to their element only
  u32x4 v;
};
struct __attribute__((packed, aligned(4))) Four {
  f32x4 v;
};

template <int D>
struct Inverse {  // 1 / rest in bf16 pieces, rounded towards zero: all of one sign
  static constexpr int N = D == 64 ? 1 : 3;
  bf16 v[N];
  __device__ __forceinline__ explicit Inverse(float rest) {
    float r = 1.f / rest;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float t = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, r) & 0xffff0000u);
      v[i] = (bf16)t;
      r -= t;
    }
  }
};

// Fragments of (1 / rest) I, either operand: row or column lane & 31, elements 16 ks + 8 hf ..
template <int D>
struct Diagonal {
  bf16x8 f[Inverse<D>::N][2];
  __device__ __forceinline__ explicit Diagonal(const Inverse<D>& inv) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int at = (lane & 31) - 16 * ks - 8 * (lane >> 5);  // the element that is not zero, if it is one of 0 .. 7
#pragma unroll
      for (int i = 0; i < Inverse<D>::N; ++i) {
        const uint32_t v = (uint32_t)__builtin_bit_cast(uint16_t, inv.v[i]) << (16 * (at & 1));
        u32x4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = at >> 1 == e ? v : 0u;
        f[i][ks] = __builtin_bit_cast(bf16x8, r);
      }
    }
  }
};

constexpr uint32_t kLowest = 0xff7fff7fu;  // two bf16

__device__ __forceinline__ u32x4 finite(u32x4 v) {  // minus infinity (and negative NaN) to the lowest finite value
  typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
  const u16x8 low = __builtin_bit_cast(u16x8, u32x4{kLowest, kLowest, kLowest, kLowest});
  return __builtin_bit_cast(u32x4, __builtin_elementwise_min(__builtin_bit_cast(u16x8, v), low));
}

// elements k .. k + 7 of a row of L; TAIL: past the end the lowest value
template <bool TAIL>
__device__ __forceinline__ u32x4 load_eight(const bf16* row, int k, int L) {
  if constexpr (!TAIL) return reinterpret_cast<const Eight*>(row + k)->v;
  typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
  u16x8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e)
    r[e] = k + e < L ? __builtin_bit_cast(uint16_t, row[min(k + e, L - 1)]) : (uint16_t)kLowest;
  return __builtin_bit_cast(u32x4, r);
}

// a mask value per lane (row or column lane & 31) against 1 / rest on the other side
template <int D>
__device__ __forceinline__ bf16x8 spread(bf16 v) {
  bf16x8 f{};
  // minus infinity as in finite(): a piece of 1 / rest may be zero (NaN stays)
  if (__builtin_bit_cast(uint16_t, v) == 0xff80u) v = __builtin_bit_cast(bf16, (uint16_t)kLowest);
  if ((threadIdx.x & 63) < 32) {
#pragma unroll
    for (int i = 0; i < Inverse<D>::N; ++i) f[i] = v;
  }
  return f;
}
template <int D>
__device__ __forceinline__ bf16x8 pieces(const Inverse<D>& inv) {
  bf16x8 f{};
  if ((threadIdx.x & 63) < 32) {
#pragma unroll
    for (int i = 0; i < Inverse<D>::N; ++i) f[i] = inv.v[i];
  }
  return f;
}

// Biases of a wave's tiles with keys down the rows of S^T and a query on each lane
template <int D, typename TB>
struct QueryBias;

template <int D>
struct QueryBias<D, bf16> {
  const bf16 *b1, *b2;  // the row of (b, n), the row of (b, h, query)
  Diagonal<D> eye;
  bf16x8 inv;
  u32x4 seen;  // largest bit patterns met: above 0xff80 is a negative NaN, which finite() hides
  __device__ __forceinline__ QueryBias(const bf16* m, const bf16* pair, float rest)
      : b1(m), b2(pair), eye(Inverse<D>(rest)), inv(pieces<D>(Inverse<D>(rest))), seen{} {}
  template <bool TAIL>
  __device__ __forceinline__ void load_pair(int k0, int L, u32x4 (&f)[2]) const {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) f[ks] = load_eight<TAIL>(b2, k0 + 16 * ks + 8 * ((threadIdx.x & 63) >> 5), L);
  }
  __device__ __forceinline__ f32x16 add_pair(const u32x4 (&f)[2], f32x16 s) const {  // made finite
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < Inverse<D>::N; ++i) s = mfma(eye.f[i][ks], __builtin_bit_cast(bf16x8, f[ks]), s);
    return s;
  }
  // what the scores start from: the mask, so that beside a huge one all keys' scores round alike
  template <bool TAIL>
  __device__ __forceinline__ bf16 mask(int k0, int L) const {
    const int k = k0 + (threadIdx.x & 31);
    return b1 != nullptr ? b1[TAIL ? min(k, L - 1) : k] : (bf16)0.f;
  }
  template <bool TAIL>
  __device__ __forceinline__ f32x16 start(bf16 v, int k0, int L) const {
    f32x16 s{};
    if (TAIL || b1 != nullptr) {
      if (TAIL && k0 + (int)(threadIdx.x & 31) >= L) v = __builtin_bit_cast(bf16, (uint16_t)kLowest);
      s = mfma(spread<D>(v), inv, s);
    }
    return s;
  }
  template <bool TAIL>
  __device__ __forceinline__ f32x16 start(int k0, int L) const {
    return start<TAIL>(mask<TAIL>(k0, L), k0, L);
  }
  __device__ __forceinline__ void watch(const u32x4 (&f)[2]) {
    typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      seen = __builtin_bit_cast(u32x4, __builtin_elementwise_max(__builtin_bit_cast(u16x8, seen),
                                                                 __builtin_bit_cast(u16x8, f[ks])));
  }
  template <bool TAIL, bool WATCH = false>
  __device__ __forceinline__ f32x16 add(int k0, int hf, int L, f32x16 s) {
    if (b2 != nullptr) {
      u32x4 f[2];
      load_pair<TAIL>(k0, L, f);
      if constexpr (WATCH) watch(f);
      f[0] = finite(f[0]);
      f[1] = finite(f[1]);
      s = add_pair(f, s);
    }
    return s;
  }
  __device__ __forceinline__ bool nan() const {
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) bad |= (seen[i] & 0xffffu) > 0xff80u || (seen[i] >> 16) > 0xff80u;
    return bad;
  }
};

template <int D>
struct QueryBias<D, float> {
  const float *b1, *b2;
  float r;
  __device__ __forceinline__ QueryBias(const float* m, const float* pair, float rest) : b1(m), b2(pair), r(1.f / rest) {}
  template <bool TAIL>
  static __device__ __forceinline__ void row(const float* b, int k0, int hf, int L, float r, f32x16& s) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int k = k0 + 8 * g + 4 * hf;
      f32x4 f;
      if constexpr (TAIL) {
#pragma unroll
        for (int t = 0; t < 4; ++t) f[t] = b[min(k + t, L - 1)];
      } else {
        f = reinterpret_cast<const Four*>(b + k)->v;
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) s[4 * g + t] += f[t] * r;
    }
  }
  template <bool TAIL>
  __device__ __forceinline__ f32x16 mask_end(int k0, int hf, int L, f32x16 s) const {
    if constexpr (TAIL) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (k0 + acc_row(i, hf) >= L) s[i] = -INFINITY;
    }
    return s;
  }
  template <bool TAIL>
  __device__ __forceinline__ float mask(int, int) const {
    return 0.f;
  }
  template <bool TAIL>
  __device__ __forceinline__ f32x16 start(float, int, int) const {
    return f32x16{};
  }
  template <bool TAIL>
  __device__ __forceinline__ f32x16 start(int, int) const {
    return f32x16{};
  }
  template <bool TAIL, bool WATCH = false>
  __device__ __forceinline__ f32x16 add(int k0, int hf, int L, f32x16 s) {
    if (b1 != nullptr) row<TAIL>(b1, k0, hf, L, r, s);
    if (b2 != nullptr) row<TAIL>(b2, k0, hf, L, r, s);
    return mask_end<TAIL>(k0, hf, L, s);
  }
  __device__ __forceinline__ bool nan() const { return false; }
};

// Exponents of base 2 are s c - ref with one rounding, where ref, the row's maximum or normaliser times c, is not far from
// zero: its own rounding is a factor that the whole row shares. Far off (rows whose keys all have a mask of -1e9 or below)
// that factor could be anything, and the difference is taken first.
__device__ __forceinline__ bool far_off(float ref) { return fabsf(ref) > 256.f && fabsf(ref) < INFINITY; }
constexpr float kNone = -3e38f;  // the maximum of a row without a visible key so far, minus infinity but for its differences
// A large positive bias (or a NaN) beside a large negative one may give a score near zero, which then depends on the order of
// the sums, and overflow by itself over the whole scale: such ones, too, go the way of the rows far off
constexpr int16_t kLarge = 0x4380;  // 256 in bf16
__device__ __forceinline__ bool any_large(const u32x4& f) {
  typedef int16_t s16x8 __attribute__((ext_vector_type(8)));
  const s16x8 v = __builtin_bit_cast(s16x8, f);
  bool large = false;
#pragma unroll
  for (int i = 0; i < 8; ++i) large |= v[i] > kLarge;
  return large;
}
__device__ __forceinline__ bool is_large(bf16 v) { return __builtin_bit_cast(int16_t, v) > kLarge; }

struct EvoParams {
  const bf16 *q, *k, *v, *o, *dout;
  const void *b1, *b2;  // [B N, L], [B, H, L, L], or null
  bf16 *out, *dq, *dk, *dv;
  float *lse, *delta;   // [B N, H, L]: natural log of the softmax normaliser; rowsum(dO * O)
  float* db1;           // [B N, L] or null
  float* part;          // [chunks, B, H, L, L]
  int B, N, L, H;
  float scale, rest, power;  // scale = rest * power, see the biases
};

// Workgroups of one row n next to each other on one XCD: neighbouring heads share cache lines, q blocks share k and v
__device__ __forceinline__ int xcd_id() {
  const int n = gridDim.x, i = blockIdx.x, q = n / 8, r = n % 8, x = i % 8;
  return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + i / 8;
}

struct Place {
  int blk, h, bn, b;
  int64_t ld, base;  // between tokens; of (b, n, 0, h, 0)
};
template <int D>
__device__ __forceinline__ Place place(const EvoParams& p, int blocks) {
  Place a;
  int id = xcd_id();
  a.blk = id % blocks;
  id /= blocks;
  a.h = id % p.H;
  a.bn = id / p.H;
  a.b = a.bn / p.N;
  a.ld = (int64_t)p.H * D;
  a.base = (int64_t)a.bn * p.L * a.ld + (int64_t)a.h * D;
  return a;
}

// fragments of row `row` (each lane's own), 16 ks + 8 hf .. + 7
template <int D>
__device__ __forceinline__ void load_frags(const bf16* m, int64_t ld, int row, bf16x8 (&f)[D / 16]) {
  const bf16* r = m + (int64_t)row * ld + 8 * ((threadIdx.x & 63) >> 5);
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) f[ks] = *reinterpret_cast<const bf16x8*>(r + 16 * ks);
}
template <int D>
__device__ __forceinline__ void times(bf16x8& f, float power) {
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = (bf16)((float)f[e] * power);
}
template <int D>
__device__ __forceinline__ void times(bf16x8 (&f)[D / 16], float power) {
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks)
#pragma unroll
    for (int e = 0; e < 8; ++e) f[ks][e] = (bf16)((float)f[ks][e] * power);
}

// ---------------------------------------------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------------------------------------------
// one tile of 32 keys of a wave's 32 queries: m is the largest raw score, l this lane's sum of exponentials
template <int D, bool TAIL, typename Bias>
__device__ __forceinline__ void evo_tile(Bias& bias, const char* sk, const char* sv, int t0, int k0, int hf, int L, float c,
                                       const bf16x8 (&qf)[D / 16], f32x16 (&acc)[D / 32], float& m, float& l) {
  using T = Tile<D>;
  f32x16 s = bias.template start<TAIL>(k0, L);
#pragma unroll
  for (int ks = 0; ks < T::KS; ++ks) s = mfma(T::rows(sk, t0, ks), qf[ks], s);
  s = bias.template add<TAIL, true>(k0, hf, L, s);
  float top = s[0];
#pragma unroll
  for (int r = 1; r < 15; r += 2) top = fmaxf(fmaxf(top, s[r]), s[r + 1]);
  top = fmaxf(top, s[15]);
  top = fmaxf(top, __shfl_xor(top, 32, 64));
  const float mn = fmaxf(m, top);
  const float alpha = m == -INFINITY ? 0.f : fast_exp2((m - mn) * c);
  const float ref = mn == -INFINITY ? 0.f : mn;  // no visible key so far: probabilities of zero, not NaN
  m = mn;
  float sum = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    s[r] = fast_exp2((s[r] - ref) * c);  // (not s c - mn c: a row whose keys all have a mask of -1e9 or below)
    sum += s[r];
  }
  l = l * alpha + sum;  // of this lane's keys; both halves are added at the end
  const bf16x8 pb[2] = {acc_to_b<0>(s), acc_to_b<1>(s)};
#pragma unroll
  for (int dt = 0; dt < T::DT; ++dt) {
    acc[dt] *= alpha;
#pragma unroll
    for (int st = 0; st < 2; ++st) acc[dt] = mfma(T::cols(sv, t0, st, dt), pb[st], acc[dt]);
  }
}

template <int D, typename TB>
__global__ __launch_bounds__(64 * kWaves<D>) void evo_fwd_kernel(EvoParams p, int blocks) {
  using T = Tile<D>;
  __shared__ __attribute__((aligned(1024))) char smem[2 * 16384];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int hf = lane >> 5, j = lane & 31, L = p.L;
  const Place a = place<D>(p, blocks);
  const int q0 = 32 * (a.blk * nw + w), myq = q0 + j, qc = min(myq, L - 1);
  const bool live = q0 < L;
  const float c = p.rest * kLog2e;
  bf16x8 qf[T::KS];
  load_frags<D>(p.q + a.base, a.ld, qc, qf);
  times<D>(qf, p.power);
  f32x16 acc[T::DT];
#pragma unroll
  for (int dt = 0; dt < T::DT; ++dt) acc[dt] = f32x16{};
  float m = -INFINITY, l = 0.f;  // largest raw score, sum of the exponentials
  QueryBias<D, TB> bias(p.b1 != nullptr ? (const TB*)p.b1 + (int64_t)a.bn * L : nullptr,
                        p.b2 != nullptr ? (const TB*)p.b2 + ((int64_t)(a.b * p.H + a.h) * L + qc) * L : nullptr, p.rest);

  auto tile = [&](const char* sk, const char* sv, int t0, int k0, auto tail) {
    evo_tile<D, decltype(tail)::value>(bias, sk, sv, t0, k0, hf, L, c, qf, acc, m, l);
  };

  for (int c0 = 0; c0 < L; c0 += T::ROWS) {
    const int nt = (min(T::ROWS, L - c0) + 31) / 32;
    if (c0 > 0) __syncthreads();
    T::stage(smem, p.k + a.base, a.ld, c0, nt, L, nw);
    T::stage(smem + 16384, p.v + a.base, a.ld, c0, nt, L, nw);
    __syncthreads();
    if (!live) continue;
    for (int t = 0; t < nt; ++t) {
      const int k0 = c0 + 32 * t;
      if (k0 + 32 <= L) tile(smem, smem + 16384, 32 * t, k0, std::false_type{});
      else tile(smem, smem + 16384, 32 * t, k0, std::true_type{});
    }
  }
  if (!live) return;
  if (bias.nan()) l = __builtin_nanf("");
  l += __shfl_xor(l, 32, 64);
  if (myq < L) {
    const float inv = l == 0.f ? 0.f : 1.f / l;
    bf16* row = p.out + a.base + (int64_t)myq * a.ld;
#pragma unroll
    for (int dt = 0; dt < T::DT; ++dt) store_row_block<D>(row, acc[dt], dt, hf, inv);
    // (no visible key: infinity, so that the backward's probabilities are zero)
    if (hf == 0) p.lse[((int64_t)a.bn * p.H + a.h) * L + myq] = l == 0.f ? INFINITY : (m * c + log2f(l)) / kLog2e;
  }
}

// The same for heads of 32, rows of up to 256 positions and bf16 biases. In the kernel above all workgroups of a launch are on
// the chip at once and wait for their operands together, then compute together; here a workgroup walks over rows n of one head,
// and a row's operands are on their way while the one before is computed. The pair bias is the same for all of them: each wave
// keeps its 32 queries' as what the scores start from, in 32 bits (128 registers), instead of multiplying it in again. Scores
// are q . k + bias / scale, and exponents take one fused operation (see far_off). The maximum is raised with every tile, as above:
// raised only where a score exceeds it by 2^8, the largest weight, too, is rounded to bf16 (error against 64 bits 0.00225 instead of
// 0.00198; with every second tile 0.00200 and 2 us of 36 less). Rows that this does not hold for are computed again as above:
// where one of the maxima met is far off, where no key is visible or the sum is no number, and where a bias is large.
// A kernel for each count of tiles: in one for several, the way of a last single tile lay between those of the pairs (34 KB of
// code instead of 20, and 13 registers in scratch memory).
// Its time, by counters at 128 x 256 positions, 8 heads: 73,500 cycles a wave, of which a SIMD's two waves issue vector
// instructions (4,800 each, for the pair bias and four rows) for 60 % and products for 18 %; a wave waits for 38 %, for the
// pair bias and the first row and at the four rows' barriers.
template <int NT>
struct RowRing {
  static constexpr int M = 32 * NT * 64, kMask = 256 * ((NT + 1) / 2);  // bytes of K or V, of the mask (4 a key)
  static constexpr int kRow = 2 * M + kMask;
};

template <int NT>
__global__ __launch_bounds__(64 * NT, 2) void evo_fwd_rows_kernel(EvoParams p, int rows_per) {
  constexpr int D = 32;
  using T = Tile<D>;
  using W = RowRing<NT>;
  __shared__ __attribute__((aligned(1024))) char smem[2 * W::kRow];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nt = blockDim.x >> 6;
  const int hf = lane >> 5, j = lane & 31, L = p.L;
  int id = xcd_id();
  const int h = id % p.H;
  id /= p.H;
  const int chunks = (p.N + rows_per - 1) / rows_per, b = id / chunks;
  const int n0 = (id % chunks) * rows_per, n1 = min(p.N, n0 + rows_per);
  const int myq = 32 * w + j, qc = min(myq, L - 1);
  const uint32_t ld = p.H * D;
  const float c = p.rest * kLog2e, mul = p.scale * kLog2e;
  // (made anew where it is asked for: its 30 registers shall not stay through the loop)
  auto biases = [&](int n) {
    int q = qc;
    float rest = p.rest;
    asm volatile("" : "+v"(q), "+v"(rest));
    return QueryBias<D, bf16>(p.b1 != nullptr ? (const bf16*)p.b1 + ((int64_t)b * p.N + n) * L : nullptr,
                              p.b2 != nullptr ? (const bf16*)p.b2 + ((int64_t)(b * p.H + h) * L + q) * L : nullptr, rest);
  };

  Stager<D> of_k(0, NT, NT, ld, L);
  const uint32_t mask_at = 2 * threadIdx.x, q_at = 2 * (qc * ld + 8 * hf);
  bf16x8 qn[2];
  auto load = [&](int n) {
    const int64_t bn = (int64_t)b * p.N + n, base = bn * L * ld + (int64_t)h * D;
    char* s = smem + (n & 1) * W::kRow;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) qn[ks] = *reinterpret_cast<const bf16x8*>((const char*)(p.q + base) + (q_at + 32 * ks));
    of_k.stage(s, p.k + base, false);
    of_k.stage(s + W::M, p.v + base, false);
    if (p.b1 != nullptr && w < (NT + 1) / 2)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          __builtin_amdgcn_make_buffer_rsrc((void*)((const bf16*)p.b1 + bn * L), (short)0, 2 * L, 0x00020000),
          (lds_void*)(s + 2 * W::M + 256 * w), 2, mask_at, 0, 0, 0);
  };
  load(n0);

  f32x16 start[NT];
  bf16x8 inv = pieces<D>(Inverse<D>(p.rest));
  times<16>(inv, 1.f / p.power);
  QueryBias<D, bf16> bias = biases(n0);
  bool fine = true;
  u32x4 pair[NT][2] = {};  // (all on their way at once)
#pragma unroll
  for (int t = 0; t < NT; ++t)
    if (p.b2 != nullptr) {
      if (t + 1 < NT || 32 * NT == L) bias.template load_pair<false>(32 * t, L, pair[t]);
      else bias.template load_pair<true>(32 * t, L, pair[t]);
    }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    __builtin_amdgcn_sched_barrier(0);  // (tile by tile, here and below: the scheduler would spill)
    start[t] = f32x16{};
    if (p.b2 != nullptr) {
      bias.watch(pair[t]);
      fine &= !any_large(pair[t][0]) && !any_large(pair[t][1]);
      pair[t][0] = finite(pair[t][0]);
      pair[t][1] = finite(pair[t][1]);
      start[t] = bias.add_pair(pair[t], start[t]) * (1.f / p.power);
    }
    if (t + 1 == NT) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (32 * t + acc_row(r, hf) >= L) start[t][r] = -INFINITY;
    }
  }
  const bool nan = bias.nan();

  auto store = [&](int n, const f32x16& acc, float top, float l) {
    if (nan) l = __builtin_nanf("");
    l += __shfl_xor(l, 32, 64);  // both halves' keys
    const int64_t bn = (int64_t)b * p.N + n;
    if (myq < L) {
      store_row_block<D>(p.out + bn * L * ld + (int64_t)h * D + myq * ld, acc, 0, hf, l == 0.f ? 0.f : 1.f / l);
      if (hf == 0) p.lse[(bn * p.H + h) * L + myq] = l == 0.f ? INFINITY : (top + log2f(l)) / kLog2e;
    }
  };

  auto arrived = [&] { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" : "+v"(qn[0]), "+v"(qn[1])::"memory"); };
  arrived();
  uint64_t again = 0;  // rows to be computed again
#pragma unroll 1
  for (int n = n0; n < n1; ++n) {
    const char* sk = smem + (n & 1) * W::kRow;
    const char* sv = sk + W::M;
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");  // (the barrier alone orders no access of the compiler's)
    bf16x8 qf[2] = {qn[0], qn[1]};
    if (n + 1 < n1) load(n + 1);

    float ref = kNone, l = 0.f;
    bool good = fine;  // no bias is large, no maximum so far is far off: beside one, keys seen later would count as anything
    f32x16 acc[1] = {};
    // C tiles at a time: their products, and what follows of each, lie in the other's shadow
    auto tiles = [&](auto count, int t0) {
      constexpr int C = decltype(count)::value;
      f32x16 x[C];
      bf16x8 vt[C][2];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < C; ++i) {
        const bf16 v = p.b1 != nullptr ? *reinterpret_cast<const bf16*>(sv + W::M + 4 * (32 * (t0 + i) + j)) : (bf16)0.f;
        x[i] = mfma(spread<D>(v), inv, start[t0 + i]);
        good &= !is_large(v);
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < C; ++i) x[i] = mfma(T::rows(sk, 32 * (t0 + i), ks), qf[ks], x[i]);
      // V^T beside the products. (The compiler lets such a read of its own wait for the next row's operands too.)
#pragma unroll
      for (int i = 0; i < C; ++i) T::cols_now(sv + 32 * (t0 + i) * T::RB, vt[i]);
#pragma unroll
      for (int i = 0; i < C; ++i) {
        float top = x[i][0];
#pragma unroll
        for (int r = 1; r < 15; r += 2) top = fmaxf(fmaxf(top, x[i][r]), x[i][r + 1]);
        top = fmaxf(top, x[i][15]);
        const auto o = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, top), __builtin_bit_cast(uint32_t, top), false, false);
        top = fmaxf(__builtin_bit_cast(float, (uint32_t)o[0]), __builtin_bit_cast(float, (uint32_t)o[1]));
        const float next = fmaxf(ref, top * mul), alpha = fast_exp2(ref - next);
        ref = next;
        good &= ref >= -256.f || ref == kNone;
        float sum[2] = {};
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          x[i][r] = fast_exp2(__builtin_fmaf(x[i][r], mul, -ref));
          sum[r & 1] += x[i][r];
        }
        l = l * alpha + (sum[0] + sum[1]);
        acc[0] *= alpha;
        const bf16x8 pb[2] = {acc_to_b<0>(x[i]), acc_to_b<1>(x[i])};
#pragma unroll
        for (int st = 0; st < 2; ++st) acc[0] = mfma(vt[i][st], pb[st], acc[0]);
      }
    };
#pragma unroll
    for (int t = 0; t < NT; t += 2) {
      if (t >= nt) break;
      if constexpr (NT > 1)
        if (t + 1 < NT) tiles(std::integral_constant<int, 2>{}, t);
      if (t + 1 == NT) tiles(std::integral_constant<int, 1>{}, t);
    }
    if (!__all(good && fabsf(ref) <= 256.f && l < INFINITY)) again |= 1ull << (n - n0);
    arrived();  // the next row's; what is stored here is on its way while that one is computed
    store(n, acc[0], ref, l);
  }

  // rows that want the finite biases as they are
  __shared__ uint64_t s_again[NT];
  if (lane == 0) s_again[w] = again;
  __syncthreads();
  uint64_t all = 0;
  for (int i = 0; i < NT; ++i) all |= s_again[i];
  for (int n = n0; n < n1; ++n) {
    if (!(all >> (n - n0) & 1)) continue;  // (the same for all waves)
    __syncthreads();
    load(n);
    arrived();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (!(again >> (n - n0) & 1)) continue;
    const char* sk = smem + (n & 1) * W::kRow;
    bf16x8 qf[2] = {qn[0], qn[1]};
    times<D>(qf, p.power);
    float m = -INFINITY, l = 0.f;
    f32x16 acc[1] = {};
    QueryBias<D, bf16> rows = biases(n);
#pragma unroll 1
    for (int t = 0; t < NT; ++t) evo_tile<D, true>(rows, sk, sk + W::M, 32 * t, 32 * t, hf, L, c, qf, acc, m, l);
    store(n, acc[0], m * c, l);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// dQ, and rowsum(dO * O)
// ---------------------------------------------------------------------------------------------------------------
template <int D, typename TB>
__global__ __launch_bounds__(64 * kWaves<D>) void evo_dq_kernel(EvoParams p, int blocks) {
  using T = Tile<D>;
  __shared__ __attribute__((aligned(1024))) char smem[2 * 16384];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int hf = lane >> 5, j = lane & 31, L = p.L;
  const Place a = place<D>(p, blocks);
  const int q0 = 32 * (a.blk * nw + w), myq = q0 + j, qc = min(myq, L - 1);
  const bool live = q0 < L;
  const float c = p.rest * kLog2e;
  bf16x8 qf[T::KS], df[T::KS];
  load_frags<D>(p.q + a.base, a.ld, qc, qf);
  times<D>(qf, p.power);
  load_frags<D>(p.dout + a.base, a.ld, qc, df);
  const int64_t stat = ((int64_t)a.bn * p.H + a.h) * L;
  float delta = 0.f;
  {
    bf16x8 of[T::KS];
    load_frags<D>(p.o + a.base, a.ld, qc, of);
#pragma unroll
    for (int ks = 0; ks < T::KS; ++ks)
#pragma unroll
      for (int e = 0; e < 8; ++e) delta += (float)of[ks][e] * (float)df[ks][e];
    delta += __shfl_xor(delta, 32, 64);
    if (live && myq < L && hf == 0) p.delta[stat + myq] = delta;
  }
  const float lse_raw = p.lse[stat + qc] / p.rest;
  f32x16 acc[T::DT];
#pragma unroll
  for (int dt = 0; dt < T::DT; ++dt) acc[dt] = f32x16{};
  QueryBias<D, TB> bias(p.b1 != nullptr ? (const TB*)p.b1 + (int64_t)a.bn * L : nullptr,
                        p.b2 != nullptr ? (const TB*)p.b2 + ((int64_t)(a.b * p.H + a.h) * L + qc) * L : nullptr, p.rest);

  auto tile = [&](const char* sk, const char* sv, int t0, int k0, auto tail) {
    constexpr bool TAIL = decltype(tail)::value;
    f32x16 s = bias.template start<TAIL>(k0, L), d = f32x16{};
#pragma unroll
    for (int ks = 0; ks < T::KS; ++ks) s = mfma(T::rows(sk, t0, ks), qf[ks], s);
    s = bias.template add<TAIL>(k0, hf, L, s);
#pragma unroll
    for (int ks = 0; ks < T::KS; ++ks) d = mfma(T::rows(sv, t0, ks), df[ks], d);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2((s[r] - lse_raw) * c) * (d[r] - delta);
      if (TAIL && k0 + acc_row(r, hf) >= L) s[r] = 0.f;
    }
    const bf16x8 sb[2] = {acc_to_b<0>(s), acc_to_b<1>(s)};
#pragma unroll
    for (int dt = 0; dt < T::DT; ++dt)
#pragma unroll
      for (int st = 0; st < 2; ++st) acc[dt] = mfma(T::cols(sk, t0, st, dt), sb[st], acc[dt]);
  };

  for (int c0 = 0; c0 < L; c0 += T::ROWS) {
    const int nt = (min(T::ROWS, L - c0) + 31) / 32;
    if (c0 > 0) __syncthreads();
    T::stage(smem, p.k + a.base, a.ld, c0, nt, L, nw);
    T::stage(smem + 16384, p.v + a.base, a.ld, c0, nt, L, nw);
    __syncthreads();
    if (!live) continue;
    for (int t = 0; t < nt; ++t) {
      const int k0 = c0 + 32 * t;
      if (k0 + 32 <= L) tile(smem, smem + 16384, 32 * t, k0, std::false_type{});
      else tile(smem, smem + 16384, 32 * t, k0, std::true_type{});
    }
  }
  if (live && myq < L) {
    bf16* row = p.dq + a.base + (int64_t)myq * a.ld;
#pragma unroll
    for (int dt = 0; dt < T::DT; ++dt) store_row_block<D>(row, acc[dt], dt, hf, p.scale);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// dK, dV and the mask's gradient
// ---------------------------------------------------------------------------------------------------------------
template <int D, typename TB, bool MASK>
__global__ __launch_bounds__(64 * kWaves<D>) void evo_dkdv_kernel(EvoParams p, int blocks) {
  using T = Tile<D>;
  __shared__ __attribute__((aligned(1024))) char smem[2 * 16384];
  __shared__ __attribute__((aligned(16))) float s_lse[T::ROWS], s_delta[T::ROWS];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int hf = lane >> 5, j = lane & 31, L = p.L;
  const Place a = place<D>(p, blocks);
  const int k0 = 32 * (a.blk * nw + w), myk = k0 + j, kc = min(myk, L - 1);
  const bool live = k0 < L;
  const float c = p.rest * kLog2e;
  bf16x8 kf[T::KS], vf[T::KS];
  load_frags<D>(p.k + a.base, a.ld, kc, kf);
  times<D>(kf, p.power);
  load_frags<D>(p.v + a.base, a.ld, kc, vf);
  const int64_t stat = ((int64_t)a.bn * p.H + a.h) * L;
  const TB mask = p.b1 != nullptr ? ((const TB*)p.b1)[(int64_t)a.bn * L + kc] : (TB)0.f;
  const TB* b2 = p.b2 != nullptr ? (const TB*)p.b2 + (int64_t)(a.b * p.H + a.h) * L * L : nullptr;
  const Inverse<D> inv(p.rest);
  const Diagonal<D> eye(inv);
  const bf16x8 one = pieces<D>(inv), maskf = spread<D>((bf16)to_f(mask));
  const bool full = k0 + 32 <= L;
  f32x16 dk[T::DT], dv[T::DT];
#pragma unroll
  for (int dt = 0; dt < T::DT; ++dt) dk[dt] = dv[dt] = f32x16{};
  float db1 = 0.f;

  for (int c0 = 0; c0 < L; c0 += T::ROWS) {
    const int nt = (min(T::ROWS, L - c0) + 31) / 32;
    if (c0 > 0) __syncthreads();
    T::stage(smem, p.q + a.base, a.ld, c0, nt, L, nw);
    T::stage(smem + 16384, p.dout + a.base, a.ld, c0, nt, L, nw);
    for (int i = threadIdx.x; i < 32 * nt; i += blockDim.x) {
      const bool ok = c0 + i < L;  // queries past the end: a probability of zero
      s_lse[i] = ok ? p.lse[stat + c0 + i] / p.rest : INFINITY;
      s_delta[i] = ok ? p.delta[stat + c0 + i] : 0.f;
    }
    __syncthreads();
    if (!live) continue;
    for (int t = 0; t < nt; ++t) {
      f32x16 s = f32x16{}, d = f32x16{};
      if (sizeof(TB) == 2 && p.b1 != nullptr) s = mfma(one, maskf, s);
#pragma unroll
      for (int ks = 0; ks < T::KS; ++ks) s = mfma(T::rows(smem, 32 * t, ks), kf[ks], s);
      if constexpr (sizeof(TB) == 2) {  // queries down the rows: the pair bias is the left operand, its keys contract
        if (b2 != nullptr) {
          const bf16* row = (const bf16*)b2 + (int64_t)min(c0 + 32 * t + j, L - 1) * L;
          u32x4 f[2];
#pragma unroll
          for (int ks = 0; ks < 2; ++ks)
            f[ks] = full ? load_eight<false>(row, k0 + 16 * ks + 8 * hf, L) : load_eight<true>(row, k0 + 16 * ks + 8 * hf, L);
#pragma unroll
          for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < Inverse<D>::N; ++i) s = mfma(__builtin_bit_cast(bf16x8, finite(f[ks])), eye.f[i][ks], s);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int qr = min(c0 + 32 * t + acc_row(r, hf), L - 1);
          s[r] += (b2 != nullptr ? to_f(b2[(int64_t)qr * L + kc]) + to_f(mask) : to_f(mask)) / p.rest;
        }
      }
#pragma unroll
      for (int ks = 0; ks < T::KS; ++ks) d = mfma(T::rows(smem + 16384, 32 * t, ks), vf[ks], d);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 ls = *reinterpret_cast<const f32x4*>(&s_lse[32 * t + 8 * g + 4 * hf]);
        const f32x4 de = *reinterpret_cast<const f32x4*>(&s_delta[32 * t + 8 * g + 4 * hf]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 4 * g + i;
          const float pr = fast_exp2((s[r] - ls[i]) * c);
          s[r] = pr;
          d[r] = pr * (d[r] - de[i]);
          if (MASK) db1 += d[r];
        }
      }
      const bf16x8 pb[2] = {acc_to_b<0>(s), acc_to_b<1>(s)}, sb[2] = {acc_to_b<0>(d), acc_to_b<1>(d)};
#pragma unroll
      for (int dt = 0; dt < T::DT; ++dt)
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          dv[dt] = mfma(T::cols(smem + 16384, 32 * t, st, dt), pb[st], dv[dt]);
          dk[dt] = mfma(T::cols(smem, 32 * t, st, dt), sb[st], dk[dt]);
        }
    }
  }
  if (!live) return;
  db1 += __shfl_xor(db1, 32, 64);
  if (myk < L) {
    const int64_t row = a.base + (int64_t)myk * a.ld;
#pragma unroll
    for (int dt = 0; dt < T::DT; ++dt) {
      store_row_block<D>(p.dk + row, dk[dt], dt, hf, p.scale);
      store_row_block<D>(p.dv + row, dv[dt], dt, hf, 1.f);
    }
    if (MASK && hf == 0) unsafeAtomicAdd(p.db1 + (int64_t)a.bn * L + myk, db1);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// dQ, dK, dV and the mask's gradient of short rows: all of a (b, n, h) in one workgroup
// ---------------------------------------------------------------------------------------------------------------
template <int D>
struct Whole {  // a workgroup of one wave per 32 positions, a matrix of nt tiles in LDS
  using T = Tile<D>;
  static constexpr int CH = T::CH, PER = CH / 2;  // 16-byte chunks of a row; chunks of a matrix that a thread moves
  static constexpr int SB = 128;                  // bytes of a row of dS^T: one key, 64 queries
  static constexpr __host__ __device__ int bytes(int nt) { return 32 * nt * (3 * T::RB + SB + 8); }
  // the thread's number, made anew where it is asked for: addresses that are needed once a row of the loop shall not
  // stay in registers through it
  static __device__ __forceinline__ int tid() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
  }
  static __device__ __forceinline__ int row(int i, int t) { return (i * (int)blockDim.x + t) / CH; }
  // (32-bit offsets from a base that all lanes share: a register each where addresses would take two per matrix)
  static __device__ __forceinline__ void load(const bf16* m, uint32_t ld, int L, int t, u32x4 (&r)[PER]) {
#pragma unroll
    for (int i = 0; i < PER; ++i)
      r[i] = *reinterpret_cast<const u32x4*>((const char*)m + 2 * ((uint32_t)min(row(i, t), L - 1) * ld + 8 * (t % CH)));
  }
  static __device__ __forceinline__ void put(char* lds, int t, const u32x4 (&r)[PER]) {
#pragma unroll
    for (int i = 0; i < PER; ++i) *reinterpret_cast<u32x4*>(lds + T::off(row(i, t), t % CH)) = r[i];
  }
  // a transposed 4 x 16 piece and the one `step` bytes further
  static __device__ __forceinline__ bf16x8 tr_pair(const char* a, int step) {
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(a));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(a + step));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
  // dS^T: 16 lanes that write 8 bytes of 16 keys, and 32 lanes that read 32 bytes of 8 keys, meet every bank once
  static __device__ __forceinline__ int ds_off(int key, int ch) {
    return key * SB + 16 * (ch ^ ((key & 2) | ((key >> 1) & 4) | ((key >> 2) & 1)));
  }
};

// Wave w holds keys 32 w .. on its lanes, as the dK / dV kernel does, and walks over the queries. Every 64 queries the
// waves leave their dS in LDS and each makes 16 x 16 pieces of dQ from all keys. The workgroup walks over rows n of one
// head: the pair bias stays in registers, and the operands of the next row are on the way while this one is computed.
// Against a dQ and a dK / dV kernel: scores, exponentials and differences once, the inputs read once (66 us against 103,
// see the head of the file). Two waves a SIMD is what 230 to 256 registers leave, so that latencies bound it: products and
// vector instructions take 87,000 of its 135,000 cycles. Pair tiles loaded when they are needed (205 registers, but every
// wait for them waits for the next row's operands too) 86 us. Wider heads do not fit: dK and dV alone take twice as many.
template <int D, int NT, bool MASK>
__global__ __launch_bounds__(64 * NT, 2) void evo_bwd_kernel(EvoParams p, int rows_per) {
  using T = Tile<D>;
  using W = Whole<D>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nt = blockDim.x >> 6;
  constexpr int Lp = 32 * NT;  // (places in LDS are offsets of the instructions)
  const int hf = lane >> 5, j = lane & 31, L = p.L;
  char *sq = smem, *sd = sq + Lp * T::RB, *sk = sd + Lp * T::RB, *ss = sk + Lp * T::RB;
  float *s_lse = (float*)(ss + Lp * W::SB), *s_delta = s_lse + Lp;
  int id = xcd_id();
  const int h = id % p.H;
  id /= p.H;
  const int chunks = (p.N + rows_per - 1) / rows_per, b = id / chunks;
  const int n0 = (id % chunks) * rows_per, n1 = min(p.N, n0 + rows_per);
  const int k0 = 32 * w, myk = k0 + j, kc = min(myk, L - 1);
  const bool full = k0 + 32 <= L;
  const float c = p.rest * kLog2e;
  const uint32_t ld = p.H * D;
  const Inverse<D> inv(p.rest);
  const Diagonal<D> eye(inv);
  const bf16x8 one = pieces<D>(inv);
  u32x4 pair[NT][2] = {};
  if (p.b2 != nullptr) {
    const bf16* b2 = (const bf16*)p.b2 + (int64_t)(b * p.H + h) * L * L;
#pragma unroll
    for (int t = 0; t < NT; ++t)
      if (t < nt) {
        const bf16* row = b2 + (int64_t)min(32 * t + j, L - 1) * L;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const int k = k0 + 16 * ks + 8 * hf;
          pair[t][ks] = full ? load_eight<false>(row, k, L) : load_eight<true>(row, k, L);
        }
      }
#pragma unroll
    for (int t = 0; t < NT; ++t)  // (behind all loads)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) pair[t][ks] = finite(pair[t][ks]);
  }

  u32x4 rq[W::PER], rd[W::PER], ro[W::PER], rk[W::PER];
  bf16x8 rv[T::KS];
  float rl = INFINITY;  // queries past the end: a probability of zero
  bf16 rm = (bf16)0.f;
  auto load = [&](int n) {
    const int64_t bn = (int64_t)b * p.N + n, base = bn * L * ld + (int64_t)h * D;
    const int tid = W::tid(), kc = min(k0 + (tid & 31), L - 1);
    W::load(p.q + base, ld, L, tid, rq);
    W::load(p.dout + base, ld, L, tid, rd);
    W::load(p.o + base, ld, L, tid, ro);
    W::load(p.k + base, ld, L, tid, rk);
#pragma unroll
    for (int ks = 0; ks < T::KS; ++ks)
      rv[ks] = *reinterpret_cast<const bf16x8*>((const char*)(p.v + base) + 2 * (kc * ld + 16 * ks + 8 * ((tid & 63) >> 5)));
    if (tid < L) rl = (p.lse + (bn * p.H + h) * L)[(uint32_t)tid];
    if (p.b1 != nullptr) rm = ((const bf16*)p.b1 + bn * L)[(uint32_t)kc];
  };
  load(n0);

#pragma unroll 1
  for (int n = n0; n < n1; ++n) {
    const int64_t bn = (int64_t)b * p.N + n, base = bn * L * ld + (int64_t)h * D, stat = (bn * p.H + h) * L;
    if (n > n0) __syncthreads();
    const int tid = W::tid();
    W::put(sq, tid, rq);
    W::put(sd, tid, rd);
    W::put(sk, tid, rk);
#pragma unroll
    for (int i = 0; i < W::PER; ++i) {  // rowsum(dO * O)
      const bf16x8 a = __builtin_bit_cast(bf16x8, rd[i]), o = __builtin_bit_cast(bf16x8, ro[i]);
      float delta = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) delta += (float)a[e] * (float)o[e];
#pragma unroll
      for (int x = 1; x < W::CH; x *= 2) delta += __shfl_xor(delta, x, 64);
      if (tid % W::CH == 0) {
        const int q = W::row(i, tid);
        s_delta[q] = -delta;
        if (q < L) (p.delta + stat)[(uint32_t)q] = delta;
      }
    }
    if (tid < Lp) s_lse[tid] = rl / p.rest;
    bf16x8 vf[T::KS], kf[T::KS];
#pragma unroll
    for (int ks = 0; ks < T::KS; ++ks) vf[ks] = rv[ks];
    const bf16x8 maskf = spread<D>(rm);
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < T::KS; ++ks) kf[ks] = T::rows(sk, k0, ks);
    times<D>(kf, p.power);
    if (n + 1 < n1) load(n + 1);
    f32x16 dk[T::DT], dv[T::DT];
#pragma unroll
    for (int dt = 0; dt < T::DT; ++dt) dk[dt] = dv[dt] = f32x16{};
    float db1 = 0.f;

#pragma unroll
    for (int u = 0; u < (NT + 1) / 2; ++u) {
      if (2 * u >= nt) break;
      if (u > 0) __syncthreads();  // the waves have read dS of the queries before
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        const int t = 2 * u + tt;
        if (t >= NT || t >= nt) break;
        __builtin_amdgcn_sched_barrier(0);  // (tile by tile: the scheduler would spill)
        f32x16 s = mfma(one, maskf, f32x16{}), d;
#pragma unroll
        for (int ks = 0; ks < T::KS; ++ks) s = mfma(T::rows(sq, 32 * t, ks), kf[ks], s);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int i = 0; i < Inverse<D>::N; ++i)
            s = mfma(__builtin_bit_cast(bf16x8, pair[t < NT ? t : 0][ks]), eye.f[i][ks], s);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 de = *reinterpret_cast<const f32x4*>(&s_delta[32 * t + 8 * g + 4 * hf]);
#pragma unroll
          for (int i = 0; i < 4; ++i) d[4 * g + i] = de[i];
        }
#pragma unroll
        for (int ks = 0; ks < T::KS; ++ks) d = mfma(T::rows(sd, 32 * t, ks), vf[ks], d);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 ls = *reinterpret_cast<const f32x4*>(&s_lse[32 * t + 8 * g + 4 * hf]);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int r = 4 * g + i;
            const float pr = fast_exp2((s[r] - ls[i]) * c);
            s[r] = pr;
            d[r] *= pr;
            if (MASK) db1 += d[r];
          }
        }
        const bf16x8 pb[2] = {acc_to_b<0>(s), acc_to_b<1>(s)};
        const bf16x8 sb[2] = {acc_to_b<0>(d), acc_to_b<1>(d)};
#pragma unroll
        for (int dt = 0; dt < T::DT; ++dt)
#pragma unroll
          for (int st = 0; st < 2; ++st) {
            dv[dt] = mfma(T::cols(sd, 32 * t, st, dt), pb[st], dv[dt]);
            dk[dt] = mfma(T::cols(sq, 32 * t, st, dt), sb[st], dk[dt]);
          }
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          u32x4 x = __builtin_bit_cast(u32x4, sb[st]);
          if (!full && myk >= L) x = u32x4{0, 0, 0, 0};
          *reinterpret_cast<u32x2*>(ss + W::ds_off(myk, 4 * tt + 2 * st) + 8 * hf) = u32x2{x[0], x[1]};
          *reinterpret_cast<u32x2*>(ss + W::ds_off(myk, 4 * tt + 2 * st + 1) + 8 * hf) = u32x2{x[2], x[3]};
        }
      }
      __syncthreads();
      // lane group g reads keys 4 perm(g) .. + 3 of 16, so that two groups read at once from all banks
      const int ln = W::tid() & 63, g = ln >> 4, i16 = ln & 15, kq = 4 * (((g & 1) << 1) | (g >> 1)) + (i16 >> 2), pp = i16 & 3;
      const int pieces16 = min(2, nt - 2 * u) * 2 * (D / 16);
      for (int x = w; x < pieces16; x += nt) {
        const int d16 = x % (D / 16), q16 = x / (D / 16);
        const char* ka = sk + T::off(kq, 2 * d16 + (pp >> 1)) + 8 * (pp & 1);
        const char* ea = ss + W::ds_off(kq, 2 * q16 + (pp >> 1)) + 8 * (pp & 1);
        f32x4 acc[2] = {};
#pragma unroll
        for (int kb = 0; kb < NT; ++kb) {
          if (kb >= nt) break;
          acc[kb & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W::tr_pair(ka + 32 * kb * T::RB, 16 * T::RB),
                                                                W::tr_pair(ea + 32 * kb * W::SB, 16 * W::SB), acc[kb & 1], 0, 0, 0);
        }
        const int q = 64 * u + 16 * q16 + i16;
        if (q < L) {
          bf16x4 v;
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = (bf16)((acc[0][i] + acc[1][i]) * p.scale);
          *reinterpret_cast<bf16x4*>((char*)(p.dq + base) + 2 * (q * ld + 16 * d16 + 4 * g)) = v;
        }
      }
    }
    if (MASK) db1 += __shfl_xor(db1, 32, 64);
    const int ek = k0 + (W::tid() & 31);
    if (ek < L) {
      const uint32_t row = 2 * ek * ld;
#pragma unroll
      for (int dt = 0; dt < T::DT; ++dt) {
        store_row_block<D>((bf16*)((char*)(p.dk + base) + row), dk[dt], dt, hf, p.scale);
        store_row_block<D>((bf16*)((char*)(p.dv + base) + row), dv[dt], dt, hf, 1.f);
      }
      if (MASK && hf == 0) unsafeAtomicAdd(p.db1 + bn * L + myk, db1);
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// gradient of the pair bias: sum of dS over the rows
// ---------------------------------------------------------------------------------------------------------------
constexpr int kPairTiles = 2;  // of 32 keys: a wave's 32 sums and 32 biases a lane leave room for four waves a SIMD

template <typename Sums>
__device__ __forceinline__ void store_pair_sums(float* out, const Sums& sum, int k0, int hf, int L) {
#pragma unroll
  for (int t = 0; t < kPairTiles; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int k = k0 + 32 * t + 8 * g + 4 * hf;
      if (L % 4 == 0 && k < L) {
        *reinterpret_cast<f32x4*>(out + k) = f32x4{sum[t][4 * g], sum[t][4 * g + 1], sum[t][4 * g + 2], sum[t][4 * g + 3]};
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (k + i < L) out[k + i] = sum[t][4 * g + i];
      }
    }
}

template <int D, typename TB>
__global__ __launch_bounds__(256, 2) void evo_dpair_kernel(EvoParams p, int qblocks, int kblocks, int rows_per) {
  using T = Tile<D>;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int hf = lane >> 5, j = lane & 31, L = p.L;
  int id = xcd_id();
  const int qb = id % qblocks;
  id /= qblocks;
  const int kb = id % kblocks;
  id /= kblocks;
  const int h = id % p.H;
  id /= p.H;
  const int b = id % p.B, chunk = id / p.B;
  const int q0 = 32 * (qb * nw + w), myq = q0 + j, qc = min(myq, L - 1);
  if (q0 >= L) return;
  const int n0 = chunk * rows_per, n1 = min(p.N, n0 + rows_per);
  const float c = p.rest * kLog2e;
  const int64_t ld = (int64_t)p.H * D;
  QueryBias<D, TB> bias(nullptr, (const TB*)p.b2 + ((int64_t)(b * p.H + h) * L + qc) * L, p.rest);
  const int kk0 = 32 * kb * kPairTiles;
  f32x16 sum[kPairTiles];
#pragma unroll
  for (int t = 0; t < kPairTiles; ++t) sum[t] = f32x16{};

  auto walk = [&](auto tail) {
    constexpr bool TAIL = decltype(tail)::value;
    u32x4 pair[kPairTiles][2];
    if constexpr (sizeof(TB) == 2) {
#pragma unroll
      for (int t = 0; t < kPairTiles; ++t) {
        bias.template load_pair<TAIL>(kk0 + 32 * t, L, pair[t]);
        pair[t][0] = finite(pair[t][0]);
        pair[t][1] = finite(pair[t][1]);
      }
    }
#pragma unroll 1
    for (int n = n0; n < n1; ++n) {
      const int64_t bn = (int64_t)b * p.N + n, base = bn * L * ld + (int64_t)h * D, stat = (bn * p.H + h) * L;
      bf16x8 qf[T::KS], df[T::KS];
      load_frags<D>(p.q + base, ld, qc, qf);
      load_frags<D>(p.dout + base, ld, qc, df);
      times<D>(qf, p.power);
      const float lse_raw = p.lse[stat + qc] / p.rest, delta = p.delta[stat + qc];
      if (p.b1 != nullptr) bias.b1 = (const TB*)p.b1 + bn * L;
#pragma unroll
      for (int t = 0; t < kPairTiles; ++t) {
        const int k0 = kk0 + 32 * t, kr = TAIL ? min(k0 + j, L - 1) : k0 + j;
        bf16x8 kf[T::KS], vf[T::KS];
        load_frags<D>(p.k + base, ld, kr, kf);
        load_frags<D>(p.v + base, ld, kr, vf);
        f32x16 s = bias.template start<TAIL>(k0, L), d = f32x16{};
#pragma unroll
        for (int ks = 0; ks < T::KS; ++ks) s = mfma(kf[ks], qf[ks], s);
        if constexpr (sizeof(TB) == 2) s = bias.add_pair(pair[t], s);
        else s = bias.template add<TAIL>(k0, hf, L, s);
#pragma unroll
        for (int ks = 0; ks < T::KS; ++ks) d = mfma(vf[ks], df[ks], d);
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[t][r] += fast_exp2((s[r] - lse_raw) * c) * (d[r] - delta);
      }
    }
  };
  if (kk0 + 32 * kPairTiles <= L) walk(std::false_type{}); else walk(std::true_type{});
  if (myq >= L) return;
  store_pair_sums(p.part + (((int64_t)chunk * p.B + b) * p.H + h) * L * L + (int64_t)myq * L, sum, kk0, hf, L);
}

// The same for narrower heads, whose operands of two rows fit in LDS (32 or 64 KB a row; D = 128 would want 128), where
// hds_evoformer_pair_staged says so: a workgroup of up to 4 x 2 waves stages the queries and the keys that its waves share, a
// row ahead (three rows ahead is level). In the kernel above each wave loads its own, between them almost three times the bytes, in pieces of 16
// bytes a row, and waits for them: 128 rows of 256, 8 heads, D = 32 58 -> 42 us; a training pass with D = 64 296 -> 251 us.
// The pair bias is what the scores start from (of near rows, see far_off) instead of six products a tile, the exponent's argument
// takes one operation, and the distances of a row's loads are made once: 42 -> 34 us. By counters, of 64,600 cycles a wave a SIMD's
// two waves issue vector instructions for 45 % and products for 17 %; a wave waits for 36 %, at the start and for each row.
template <int D>
struct PairRows {
  static constexpr int M = 128 * Tile<D>::RB;    // bytes of a matrix: 128 rows
  static constexpr int kAux = 768;               // of a wave: its queries' lse and delta, its keys' mask, 4 bytes a lane
  static constexpr int kRow = 4 * M + 8 * kAux;  // Q, dO, K, V of a row n, and the waves' own
};

template <int D, typename TB>
__global__ __launch_bounds__(512, 2) void evo_dpair_rows_kernel(EvoParams p, int qblocks, int kblocks, int rows_per,
                                                                int nwq) {
  using T = Tile<D>;
  using W = PairRows<D>;
  constexpr int M = W::M;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6, nwk = nw / nwq;
  const int hf = lane >> 5, j = lane & 31, L = p.L, wq = w % nwq, wk = w / nwq;
  int id = xcd_id();
  const int qb = id % qblocks;
  id /= qblocks;
  const int kb = id % kblocks;
  id /= kblocks;
  const int h = id % p.H;
  id /= p.H;
  const int b = id % p.B, chunk = id / p.B;
  const int qs = 32 * qb * nwq, ks0 = 32 * kPairTiles * kb * nwk;  // of the workgroup
  const int myq = qs + 32 * wq + j, qc = min(myq, L - 1), kk0 = ks0 + 32 * kPairTiles * wk;
  const bool live = qs + 32 * wq < L && kk0 < L;
  const int n0 = chunk * rows_per, n1 = min(p.N, n0 + rows_per);
  const float c = p.rest * kLog2e;
  const int64_t ld = (int64_t)p.H * D;
  QueryBias<D, TB> bias(nullptr, (const TB*)p.b2 + ((int64_t)(b * p.H + h) * L + qc) * L, p.rest);
  float sum[kPairTiles][16];  // (single values: as vectors they are copied where the paths below meet)
#pragma unroll
  for (int t = 0; t < kPairTiles; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) sum[t][r] = 0.f;

  // the pair bias, the rows' normalisers and masks, on their way together
  u32x4 pair[kPairTiles][2] = {};
  if constexpr (sizeof(TB) == 2) {
#pragma unroll
    for (int t = 0; t < kPairTiles; ++t) {
      if (kk0 + 32 * t + 32 <= L) bias.template load_pair<false>(kk0 + 32 * t, L, pair[t]);
      else bias.template load_pair<true>(kk0 + 32 * t, L, pair[t]);
    }
  }
  bool far = false;
  const bool masked = sizeof(TB) == 2 && p.b1 != nullptr;
  const int mk = min(kk0 + lane, L - 1);
  for (int n = n0; n < n1; n += 16) {
    float v[16];
    bf16 m[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int64_t bn = (int64_t)b * p.N + min(n + i, n1 - 1);
      v[i] = (p.lse + (bn * p.H + h) * L)[(uint32_t)qc];
      m[i] = *(masked ? (const bf16*)p.b1 + bn * L + mk : p.q);  // (a branch would have every row wait for the one before)
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) far = far | far_off(v[i] * kLog2e) | (masked & is_large(m[i]));
  }
  if constexpr (sizeof(TB) == 2) {
#pragma unroll
    for (int t = 0; t < kPairTiles; ++t) {
      far |= any_large(pair[t][0]) || any_large(pair[t][1]);
      pair[t][0] = finite(pair[t][0]);
      pair[t][1] = finite(pair[t][1]);
    }
  }
  far = __any(far);
  auto walk = [&](auto is_far) {
    // (32-bit biases: whole workgroups only. The others' tail is a choice a tile)
    constexpr bool TAIL = sizeof(TB) == 2, FAR = decltype(is_far)::value;
    // Near rows: scores are q . k + bias / scale, and a bias that overflows is one whose weight is zero. Far ones as elsewhere
    constexpr bool kPlain = sizeof(TB) == 2 && !FAR;
    const float mul = kPlain ? p.scale * kLog2e : c;
    // (in the forward's order: beside 1e9 each sum rounds by more than what an exponent can take).
    f32x16 start[kPairTiles];  // the pair bias, which the scores of near rows start from
    if constexpr (sizeof(TB) == 2) {
      if constexpr (!FAR) {
#pragma unroll
        for (int t = 0; t < kPairTiles; ++t) start[t] = bias.add_pair(pair[t], f32x16{}) * (1.f / p.power);
        times<16>(bias.inv, 1.f / p.power);
      }
    }
    // What a lane takes from a row n lies at the same distance from the row's start for every n: the distances are made once
    Stager<D> of_q(qs, nwq, nw, ld, L), of_k(ks0, kPairTiles * nwk, nw, ld, L);
    const uint32_t stat_at = 4 * qc, mask_at = 2 * min(kk0 + lane, L - 1);
    auto rsrc = [&](const void* m, int size) { return __builtin_amdgcn_make_buffer_rsrc((void*)m, (short)0, size * L, 0x00020000); };
    const bool one = D == 32 && nw == 8 && nwq == 4;
    auto load = [&](int n) {
      const int64_t bn = (int64_t)b * p.N + n, base = bn * L * ld + (int64_t)h * D;
      char* s = smem + (n - n0) % 2 * W::kRow;
      char* mine = s + 4 * M + w * W::kAux;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc(p.lse + (bn * p.H + h) * L, 4), (lds_void*)mine, 4, stat_at, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc(p.delta + (bn * p.H + h) * L, 4), (lds_void*)(mine + 256), 4, stat_at, 0, 0, 0);
      if (sizeof(TB) == 2 && p.b1 != nullptr)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc((const bf16*)p.b1 + bn * L, 2), (lds_void*)(mine + 512), 2, mask_at, 0, 0, 0);
      of_q.stage(s, p.q + base, one);
      of_q.stage(s + M, p.dout + base, one);
      of_k.stage(s + 2 * M, p.k + base, one);
      of_k.stage(s + 3 * M, p.v + base, one);
    };
    load(n0);
#pragma unroll 1
    for (int n = n0; n < n1; ++n) {
      const char* s = smem + (n - n0) % 2 * W::kRow;
      // this row has arrived, and every wave is done with the one whose place the next one takes
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (n + 1 < n1) load(n + 1);
      if (!live) continue;
      const char* mine = s + 4 * M + w * W::kAux;
      const float lse = *reinterpret_cast<const float*>(mine + 4 * j), delta = *reinterpret_cast<const float*>(mine + 256 + 4 * j);
      TB mask[kPairTiles];
#pragma unroll
      for (int t = 0; t < kPairTiles; ++t) {
        if constexpr (sizeof(TB) == 2)
          mask[t] = p.b1 != nullptr ? *reinterpret_cast<const bf16*>(mine + 512 + 128 * t + 4 * j) : (bf16)0.f;
        else mask[t] = 0.f;
      }
      if (p.b1 != nullptr) bias.b1 = (const TB*)p.b1 + ((int64_t)b * p.N + n) * L;
      bf16x8 qf[T::KS], df[T::KS];
#pragma unroll
      for (int ks = 0; ks < T::KS; ++ks) {
        qf[ks] = T::rows(s, 32 * wq, ks);
        df[ks] = T::rows(s + M, 32 * wq, ks);
      }
      if constexpr (!kPlain) times<D>(qf, p.power);
      const float ref = lse * kLog2e, lse_raw = FAR ? lse / p.rest : 0.f;
      f32x16 less;
#pragma unroll
      for (int r = 0; r < 16; ++r) less[r] = -delta;
      f32x16 x[kPairTiles], d[kPairTiles];
      auto products = [&](int t) {
        const int k0 = kk0 + 32 * t, kr = 32 * (kPairTiles * wk + t);
        d[t] = less;
        if constexpr (sizeof(TB) == 2) {
          TB v = mask[t];
          if (TAIL && k0 + j >= L) v = __builtin_bit_cast(bf16, (uint16_t)kLowest);
          if constexpr (FAR) x[t] = mfma(spread<D>(v), bias.inv, f32x16{});
          else x[t] = mfma(spread<D>(v), bias.inv, start[t]);
        } else {
          x[t] = f32x16{};
        }
#pragma unroll
        for (int ks = 0; ks < T::KS; ++ks) {
          x[t] = mfma(T::rows(s + 2 * M, kr, ks), qf[ks], x[t]);
          d[t] = mfma(T::rows(s + 3 * M, kr, ks), df[ks], d[t]);
        }
        if constexpr (sizeof(TB) == 4) x[t] = bias.template add<TAIL>(k0, hf, L, x[t]);
        else if constexpr (FAR) x[t] = bias.add_pair(pair[t], x[t]);
      };
      products(0);
#pragma unroll
      for (int t = 0; t < kPairTiles; ++t) {
        __builtin_amdgcn_sched_barrier(0);
        if (t + 1 < kPairTiles) products(t + 1);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float v = FAR ? (x[t][r] - lse_raw) * c : __builtin_fmaf(x[t][r], mul, -ref);
          sum[t][r] += fast_exp2(v) * d[t][r];
        }
        if (t + 1 < kPairTiles) {  // the products of one tile beside the exponents of the other
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
            __builtin_amdgcn_sched_group_barrier(0x400, 2, 0);
          }
        }
      }
    }
  };
  if (!far) walk(std::false_type{}); else walk(std::true_type{});  // (waves of either kind meet at the barriers, as many in both)
  if (!live || myq >= L) return;
  store_pair_sums(p.part + (((int64_t)chunk * p.B + b) * p.H + h) * L * L + (int64_t)myq * L, sum, kk0, hf, L);
}

template <typename TB>
__global__ __launch_bounds__(256) void evo_pair_sum_kernel(const float* __restrict__ part, TB* __restrict__ out,
                                                           int64_t n, int chunks) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  if (n % 4 == 0) {
    f32x4 s = *reinterpret_cast<const f32x4*>(part + i);
#pragma unroll 4
    for (int c = 1; c < chunks; ++c) s += *reinterpret_cast<const f32x4*>(part + c * n + i);
#pragma unroll
    for (int t = 0; t < 4; ++t) out[i + t] = from_f<TB>(s[t]);
    return;
  }
  for (int t = 0; t < 4 && i + t < n; ++t) {
    float s = 0.f;
    for (int c = 0; c < chunks; ++c) s += part[c * n + i + t];
    out[i + t] = from_f<TB>(s);
  }
}

bool bad_shape(int bias_dtype, int B, int N, int L, int H, int D) {
  const int64_t blocks = (int64_t)B * N * H * ((L + 31) / 32);
  return (D != 32 && D != 64 && D != 128) || (bias_dtype != kBF16 && bias_dtype != kF32) || blocks > 0x7fffffff;
}

// rest in [0.49, 0.99]: the lowest bf16 value over it is minus infinity. False for a scale that the kernels cannot take: one
// that is not positive and normal, or with bf16 biases of D = 64 one whose 1 / rest is more than one bf16 piece.
bool set_scale(EvoParams& p, float scale, int bias_dtype, int D) {
  if (!std::isnormal(scale) || scale < 0.f) return false;
  int e;
  p.scale = scale;
  p.rest = std::frexp(scale, &e);
  if (p.rest > 0.99f) {
    p.rest *= 0.5f;
    ++e;
  }
  p.power = std::ldexp(1.f, e);
  const float inv = 1.f / p.rest;
  const bool one_piece = (__builtin_bit_cast(uint32_t, inv) & 0xffffu) == 0;
  return D != 64 || bias_dtype != kBF16 || one_piece || (p.b1 == nullptr && p.b2 == nullptr);
}

// Waves of a workgroup: 32 positions each, at most 256 of them (a row's operands are then staged once), evenly spread
int waves_of(int L, int most) {
  const int tiles = (L + 31) / 32, blocks = (tiles + most - 1) / most;
  return (tiles + blocks - 1) / blocks;
}

}  // namespace

#define HDS_EVO_ALL(CALL)                                                                                           \
  if (bias_dtype == kBF16) {                                                                                        \
    if (D == 32) CALL(32, bf16); else if (D == 64) CALL(64, bf16); else CALL(128, bf16);                            \
  } else {                                                                                                          \
    if (D == 32) CALL(32, float); else if (D == 64) CALL(64, float); else CALL(128, float);                         \
  }

// Rows that a forward workgroup of heads of 32 with bf16 biases walks over (evo_fwd_rows_kernel), 0: a workgroup a row. Where
// there are more than two rows for each workgroup that the chip holds at once (slots) and an estimate is for it. A walk is one
// batch b, so that few rows n make many short ones. In units of a row that is walked over: a workgroup costs its rows and 1 to 1.25 for
// the pair bias, in whole rounds where one fills a CU; a workgroup a row costs 1.45 (1.35 with five tiles) a row and slot. Up to
// 64 positions walking is the faster one throughout. us, a workgroup a row / walking, 8 heads, B x N: 256 positions 1 x 65 27.7 /
// 26.6, 1 x 128 38.6 / 34.0, 1 x 256 70 / 56, 192 x 1 78.8 / 100.9, 96 x 2 58.2 / 65.4, 64 x 3 56.4 / 55.6, 48 x 4 55.3 / 63.0, 32 x 6 55.7 / 45.5,
// 24 x 8 54.1 / 62.5; 128 positions 1 x 131 16.1 / 17.2, 1 x 192 19.8 / 18.8, 1 x 512 43.5 / 34.7, 384 x 1 38.1 / 47.1, 192 x 2 35.6 /
// 37.1, 96 x 4 34.7 / 31.6; 154 positions 1 x 128 27.8 / 22.8; 64 positions 1 x 261 14.5 / 12.4, 768 x 1 35.1 / 28.1; 32, 1536 x 1 41.5 / 22.2.
// (A row's bit in one word: no more than 64.)
HDS_EXPORT int hds_evoformer_walk(int B, int N, int L, int H) {
  const int64_t nt = (L + 31) / 32, heads = (int64_t)B * H, rows = heads * N;
  if (B <= 0 || N <= 0 || L <= 0 || H <= 0 || nt > 8 || (L + 31) * (int64_t)H * 32 >= (int64_t)1 << 31)  // (Stager: 32 bits, whole tiles)
    return 0;
  const int64_t slots = 256 * (8 / nt), even = std::min<int64_t>(N, (rows + slots - 1) / slots);
  if (rows <= 2 * slots || even > 64) return 0;
  if (nt <= 2) return (int)even;
  auto cost = [&](int64_t per) {
    const float rounds = (float)(heads * ((N + per - 1) / per)) / (float)slots;
    return std::max(1.f, nt > 4 ? std::ceil(rounds) : rounds) * ((float)per + (nt > 4 ? 1.25f : 1.f));
  };
  const int64_t chunks = std::max<int64_t>(1, std::min<int64_t>(N, slots / heads)), once = (N + chunks - 1) / chunks;
  const int64_t per = once <= 64 && cost(once) < cost(even) ? once : even;
  const float each = (float)rows / (float)slots;
  return cost(per) < (nt == 5 ? 1.35f : 1.45f) * (nt > 4 ? std::ceil(each) : each) ? (int)per : 0;
}

// q/k/v/o [B, N, L, H, D] bf16, 16-byte aligned; b1 [B, N, 1, 1, L] or null; b2 [B, 1, H, L, L] or null (bias dtype: 1 =
// bf16, 0 = fp32); lse [B, N, H, L] fp32 (natural log of the softmax normaliser of the scaled + biased scores). A query whose keys
// are all masked by minus infinity gives zeros (and no gradients); its lse is plus infinity. scale > 0; with D = 64 and
// bf16 biases one over a power of two times at most eight bits (1 / 8 there: 64^-0.5), see set_scale.
HDS_EXPORT int hds_evoformer_fwd(const void* q, const void* k, const void* v, const void* b1, const void* b2,
                                 int bias_dtype, void* o, float* lse, int B, int N, int L, int H, int D, float scale,
                                 hipStream_t st) {
  if (B <= 0 || N <= 0 || L <= 0 || H <= 0) return 0;
  if (bad_shape(bias_dtype, B, N, L, H, D)) return hipErrorInvalidValue;
  EvoParams p{};
  p.q = (const bf16*)q; p.k = (const bf16*)k; p.v = (const bf16*)v; p.b1 = b1; p.b2 = b2; p.out = (bf16*)o; p.lse = lse;
  p.B = B; p.N = N; p.L = L; p.H = H;
  if (!set_scale(p, scale, bias_dtype, D)) return hipErrorInvalidValue;
  if (const int per = bias_dtype == kBF16 && D == 32 ? hds_evoformer_walk(B, N, L, H) : 0; per > 0) {
    const int nt = (L + 31) / 32;
    const dim3 grid(B * H * ((N + per - 1) / per)), threads(64 * nt);
    switch (nt) {
#define HDS_EVO_ROWS(NT) \
  case NT: hipLaunchKernelGGL(evo_fwd_rows_kernel<NT>, grid, threads, 0, st, p, per); break
      HDS_EVO_ROWS(1);
      HDS_EVO_ROWS(2);
      HDS_EVO_ROWS(3);
      HDS_EVO_ROWS(4);
      HDS_EVO_ROWS(5);
      HDS_EVO_ROWS(6);
      HDS_EVO_ROWS(7);
      HDS_EVO_ROWS(8);
#undef HDS_EVO_ROWS
    }
    return hipGetLastError();
  }
  const int nw = waves_of(L, D == 128 ? kWaves<128> : kWaves<32>), blocks = (L + 32 * nw - 1) / (32 * nw);
#define HDS_EVO(DD, TT)                                                                                             \
  hipLaunchKernelGGL((evo_fwd_kernel<DD, TT>), dim3(blocks * H * B * N), dim3(64 * nw), 0, st, p, blocks)
  HDS_EVO_ALL(HDS_EVO)
#undef HDS_EVO
  return hipGetLastError();
}

// Chunks of rows that the pair bias' gradient is summed in, and so the floats of scratch it wants: chunks * B * H * L * L.
// A workgroup walks over its chunk alone, so there are as many as fill the chip twice over, of at least four rows.
HDS_EXPORT int hds_evoformer_pair_chunks(int B, int N, int L, int H) {
  if (B <= 0 || N <= 0 || L <= 0 || H <= 0) return 0;
  const int64_t waves = (int64_t)B * H * ((L + 31) / 32) * ((L + 32 * kPairTiles - 1) / (32 * kPairTiles));
  int64_t chunks = (2 * 4 * 256 + waves - 1) / waves;
  const int64_t most = (N + 3) / 4;
  if (chunks > most) chunks = most;
  const int per = (int)((N + chunks - 1) / chunks);
  return (N + per - 1) / per;
}

// Are the rows of the pair bias' gradient staged by workgroups (evo_dpair_rows_kernel), rather than loaded by each wave for
// itself? Where waves share something (more than one tile of keys) and there are enough of them that the rate counts and not
// the way of a row through LDS. D = 32 wants most of its workgroups' tiles to be real, and 32-bit biases, whose tail is
// vector instructions of every wave in the workgroup, none of them beyond the end. us, waves / staged: D = 32, 512 x 32
// positions, 8 heads 25.9 / 30.1, 64 x 128, 4 heads 14.5 / 16.4, 128 x 96, 8 heads 21.5 / 20.4, 512 x 160 132 / 170, 512 x 192
// 158 / 133, 4 x 512 19.1 / 20.8, 20 x 512, 4 heads 25.5 / 20.3; D = 64, 512 x 32 30.2 / 60.8, 512 x 64 44.5 / 55.8, 64 x 96, 4
// heads 16.6 / 20.0, 64 x 128 19.4 / 18.3, 512 x 80, 8 heads 102 / 71, 512 x 160 232 / 213; 32-bit biases, D = 32, 512 x 192 264 /
// 349, 512 x 256 333 / 294, D = 64, 418 / 440 and 524 / 330.
HDS_EXPORT int hds_evoformer_pair_staged(int B, int N, int L, int H, int D, int bias_dtype) {
  if (D == 128 || L <= 32 * kPairTiles || ((int64_t)L + 127) * H * D >= (int64_t)1 << 31) return 0;  // (Stager: 32 bits, 128 rows)
  const int64_t q32 = (L + 31) / 32, k64 = (L + 32 * kPairTiles - 1) / (32 * kPairTiles);
  const int64_t waves = (int64_t)hds_evoformer_pair_chunks(B, N, L, H) * B * H * q32 * k64;
  if (bias_dtype != kBF16) return waves > 1024 && L % (64 * kPairTiles) == 0;
  if (D == 64) return waves >= 512;
  const int64_t w4 = waves_of(L, 4), q = (q32 + w4 - 1) / w4 * w4 * 32, k = (k64 + 1) / 2 * 64 * kPairTiles;
  return waves > 1024 && 4 * (int64_t)L * L >= 3 * q * k;
}

// Gradients of the forward above from its result and lse. delta [B, N, H, L] fp32 scratch. db1 [B, N, L] fp32, zeroed, or
// null; db2 [B, H, L, L] of the biases' dtype, or null; part: see hds_evoformer_pair_chunks (with db2).
HDS_EXPORT int hds_evoformer_bwd(const void* q, const void* k, const void* v, const void* o, const float* lse,
                                 const void* dout, void* dq, void* dk, void* dv, float* delta, const void* b1,
                                 const void* b2, int bias_dtype, float* db1, void* db2, float* part, int B, int N, int L,
                                 int H, int D, float scale, hipStream_t st) {
  if (B <= 0 || N <= 0 || L <= 0 || H <= 0) return 0;
  if (bad_shape(bias_dtype, B, N, L, H, D) || (db2 != nullptr && (b2 == nullptr || part == nullptr)))
    return hipErrorInvalidValue;
  EvoParams p{};
  p.q = (const bf16*)q; p.k = (const bf16*)k; p.v = (const bf16*)v; p.o = (const bf16*)o; p.dout = (const bf16*)dout;
  p.b1 = b1; p.b2 = b2; p.dq = (bf16*)dq; p.dk = (bf16*)dk; p.dv = (bf16*)dv; p.lse = (float*)lse; p.delta = delta;
  p.db1 = db1; p.part = part; p.B = B; p.N = N; p.L = L; p.H = H;
  if (!set_scale(p, scale, bias_dtype, D)) return hipErrorInvalidValue;
  const int nt = (L + 31) / 32;
  if (bias_dtype == kBF16 && D == 32 && nt <= 8 && (int64_t)L * H * D < (1 << 30)) {  // (offsets in 32 bits)
    // as many workgroups as the chip holds at once, two waves a SIMD, if there are rows for them. Each size has its LDS: with
    // the 21 KB of two tiles for one, seven workgroups fit where eight are counted on (512 rows of 16 / 32, 8 heads: 17.7 /
    // 20.4 us, with its own 10 KB 12.0 / 18.0; 256 of 32 11.6 and 9.1)
    const int64_t rows = (int64_t)B * N * H, slots = 256 * (8 / nt);
    const int per = (int)((rows + slots - 1) / slots);
    const dim3 grid(B * H * ((N + per - 1) / per)), threads(64 * nt);
    auto launch = [&](auto tiles, auto mask) {
      constexpr int NT = decltype(tiles)::value, least = NT <= 2 ? NT : NT / 2 + 1;
      static_assert(Whole<32>::bytes(NT) * (8 / least) <= 160 * 1024, "fewer workgroups on a CU than are counted on");
      auto* kernel = evo_bwd_kernel<32, NT, decltype(mask)::value>;
      const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                               Whole<32>::bytes(NT));  // (of the current device)
      if (e == hipSuccess) hipLaunchKernelGGL(kernel, grid, threads, Whole<32>::bytes(NT), st, p, per);
      return e;
    };
    auto choose = [&](auto mask) {
      if (nt == 1) return launch(std::integral_constant<int, 1>{}, mask);
      if (nt == 2) return launch(std::integral_constant<int, 2>{}, mask);
      if (nt <= 4) return launch(std::integral_constant<int, 4>{}, mask);
      return launch(std::integral_constant<int, 8>{}, mask);
    };
    const hipError_t e = db1 != nullptr ? choose(std::true_type{}) : choose(std::false_type{});
    if (e != hipSuccess) return e;
  } else {
    const int nw = waves_of(L, D == 128 ? kWaves<128> : kWaves<32>), blocks = (L + 32 * nw - 1) / (32 * nw);
    const dim3 grid(blocks * H * B * N), threads(64 * nw);
#define HDS_EVO(DD, TT)                                                                                             \
  do {                                                                                                              \
    hipLaunchKernelGGL((evo_dq_kernel<DD, TT>), grid, threads, 0, st, p, blocks);                                   \
    if (db1 != nullptr)                                                                                             \
      hipLaunchKernelGGL((evo_dkdv_kernel<DD, TT, true>), grid, threads, 0, st, p, blocks);                         \
    else                                                                                                            \
      hipLaunchKernelGGL((evo_dkdv_kernel<DD, TT, false>), grid, threads, 0, st, p, blocks);                        \
  } while (0)
    HDS_EVO_ALL(HDS_EVO)
#undef HDS_EVO
  }
  if (db2 != nullptr) {
    const int chunks = hds_evoformer_pair_chunks(B, N, L, H), per = (N + chunks - 1) / chunks;
    const int64_t n = (int64_t)B * H * L * L;
    const bool staged = hds_evoformer_pair_staged(B, N, L, H, D, bias_dtype);
    const int w4 = waves_of(L, 4), qblocks = (L + 32 * w4 - 1) / (32 * w4);
    const int kt = (L + 32 * kPairTiles - 1) / (32 * kPairTiles);
    const int kblocks = staged ? (kt + 1) / 2 : kt, wk = (kt + kblocks - 1) / kblocks;
    const int64_t grid2 = (int64_t)chunks * B * H * kblocks * qblocks;
    if (grid2 > 0x7fffffff || (n + 1023) / 1024 > 0x7fffffff) return hipErrorInvalidValue;
    auto pair = [&](auto dim, auto type) -> hipError_t {
      constexpr int DD = decltype(dim)::value;
      using TB = decltype(type);
      if constexpr (DD < 128) {
        if (staged) {
          auto* kernel = evo_dpair_rows_kernel<DD, TB>;
          constexpr int lds = 2 * PairRows<DD>::kRow;
          const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
          if (e == hipSuccess)
            hipLaunchKernelGGL(kernel, dim3(grid2), dim3(64 * w4 * wk), lds, st, p, qblocks, kblocks, per, w4);
          return e;
        }
      }
      hipLaunchKernelGGL((evo_dpair_kernel<DD, TB>), dim3(grid2), dim3(64 * w4), 0, st, p, qblocks, kblocks, per);
      return hipSuccess;
    };
    auto of_type = [&](auto dim) { return bias_dtype == kBF16 ? pair(dim, bf16{}) : pair(dim, 0.f); };
    const hipError_t e = D == 32 ? of_type(std::integral_constant<int, 32>{})
                         : D == 64 ? of_type(std::integral_constant<int, 64>{})
                                   : of_type(std::integral_constant<int, 128>{});
    if (e != hipSuccess) return e;
    if (bias_dtype == kBF16)
      hipLaunchKernelGGL(evo_pair_sum_kernel<bf16>, dim3((n + 1023) / 1024), dim3(256), 0, st, part, (bf16*)db2, n,
                         chunks);
    else
      hipLaunchKernelGGL(evo_pair_sum_kernel<float>, dim3((n + 1023) / 1024), dim3(256), 0, st, part, (float*)db2, n,
                         chunks);
  }
  return hipGetLastError();
}
