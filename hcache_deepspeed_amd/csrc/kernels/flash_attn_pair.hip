// FlashAttention forward over a paged cache, head size 128, by workgroups of 128 query rows: for steps whose 256-row
// workgroups (flash_attn_w64.hip) leave CUs idle or differ in their lengths, as prompts of up to some thousand tokens
// (ops/paged_prefill.py ``prefill_rows`` chooses).
//
// What bounds the 256-row kernel there is its chain: each of its waves has a SIMD to itself and walks all keys, 1.9 us a tile
// of 64, whether a quarter of the CUs work or all. Here two groups of four waves take the tiles of 64 keys in turn, for the
// same 128 rows (32 a wave), and their parts are added through LDS at the end: half the rows and half the tiles a wave. The
// groups share the SIMDs and go round a turn half a turn apart, joined by barriers: while one group multiplies (P.V of its
// tile and S of its next one, 32 MFMAs a wave), the other does its softmax. Fragments are read from LDS two groups of four
// MFMAs ahead. At 32 rows a wave LDS reads are as long as the products; without them, without the softmax and without the
// loads the kernel takes 759 of 943 us at 16,000 tokens (without the softmax 836, without the loads too 768): the products at
// the clock that they leave, 1.38 PFLOP/s, are what it runs at. The groups joined once a turn instead of twice: 998 us; one
// group of MFMAs ahead 977.
#include <algorithm>

#include "flash_attn_shared.h"

namespace {

__device__ __forceinline__ float xor32_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return max3_raw(__uint_as_float(r[0]), __uint_as_float(r[1]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xor32_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Queries are the new tokens of a sequence behind earlier ones, keys and values lie in the paged cache, causal (as in
// attn_fwd_w64_kernel; an entry of the list is 256 new tokens, which two workgroups share here). A kernel of contiguous rows
// made a forward of 2 x 509 tokens 25 -> 16 us, but the training step it is part of 1 % faster only.
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_fwd_pair_kernel(AttnParams p, int n) {
  constexpr int D = 128, BM = 128, KS = 8, DT = 4, TL = 16384, PW = 4;
  __shared__ __attribute__((aligned(1024))) char smem[8 * TL];  // a group: K[2], V[2]
  // By groups of entries: a workgroup a head of each, for its second 128 rows, which see more keys, where it has them, then
  // those for the first rows of such. A group is of a multiple of 32 heads: workgroups go round the XCDs and their 4 shader
  // engines, and empty ones of short entries that come in shorter runs meet the same engines, which then idle (entry by
  // entry, 16 sequences of 16 tokens behind 60, 16 heads, 14.9 us, so 9.4; 64 of 64 tokens, 4 heads 19.7 and 10.5). Larger
  // groups part the halves, of whose keys one finds the other's in L2 (all entries in one, 8 of 256 tokens behind 1,500, 32 /
  // 32 heads 71 -> 88). The heads of a key head are on one XCD.
  const int g = 32 >> min(5, __builtin_ctz(p.hq)), e0 = blockIdx.y * g, run = min(g, n - e0) * p.hq;
  const int later = (int)blockIdx.x >= run, place = blockIdx.x - later * run;
  if (place >= run) return;
  const int at = e0 + place / p.hq, rr = place % p.hq;
  const int hq = p.hq % 8 == 0 ? (rr % 8) * (p.hq / 8) + rr / 8 : rr;
  const int seq = p.blocks[2 * at], first = p.blocks[2 * at + 1];
  const int n_new = p.meta[3 * seq + 1], seen = p.meta[3 * seq + 2];
  const bool two = first + BM < n_new;
  if (first >= n_new || (later && !two)) return;
  const int row0 = first + (two && !later ? BM : 0);
  const int start = p.meta[3 * seq] - seen, len = seen + n_new, q0 = seen + row0;
  const int* table = p.tables + (int64_t)seq * p.max_blocks;
  const int hk = hq / (p.hq / p.hkv);
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w = wv & 3, grp = wv >> 2;
  const int wq_lo = q0 + 32 * w, wq_hi = wq_lo + 31, myq = wq_lo + (lane & 31);
  const float c = p.scale * kLog2e;
  int klo, khi;
  key_span(p, myq, len, klo, khi);
  bf16x8 qf[KS];
  {
    const bf16* qp = p.q + (int64_t)(start + min(myq, len - 1)) * p.sq + (int64_t)hq * D + 8 * h;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const bf16x8*>(qp + 16 * ks);
  }
  const int kt_end = (min(q0 + BM, len) + BN - 1) / BN;
  const int kt_begin = p.window > 0 ? max(0, q0 - p.window + 1) / BN : 0;
  // tiles past kt_end_w follow all rows of the wave
  const int kt_end_w = wq_lo >= len ? kt_begin : min(kt_end, wq_hi / BN + 1);
  const int turns = (kt_end - kt_begin + 1) / 2;  // of the group with the first tile

  // a wave's four pieces of a tile: rows 4 (4 w + j) + lane / 16, whose 16-byte pieces lie at c ^ swz(row)
  const int drow = lane >> 4, dcol = 16 * ((lane & 15) ^ (drow << 2));
  // lane i holds the cache slot of tile win + i
  int win = kt_begin, slots = 0;
  auto load_slots = [&](int first) __attribute__((always_inline)) {
    win = first;
    const int per = p.block_size / BN, t = min(first + lane, kt_end - 1), b = t / per;
    slots = table[b] * p.block_size + (t - b * per) * BN;
  };
  load_slots(kt_begin);
  auto source = [&](const bf16* base, int64_t stride, int kt) {
    const int rows = min(BN, len - kt * BN), slot = __builtin_amdgcn_readlane(slots, kt - win);
    return TileSrc{(const char*)(base + (int64_t)slot * stride + (int64_t)hk * D),
                   (int)(((int64_t)(rows - 1) * stride + D) * 2)};
  };
  // tile of turn i of this group; past the end the last tile, which nobody reads
  auto tile_of = [&](int i) { return min(kt_begin + 2 * i + grp, kt_end - 1); };
  auto stage = [&](bool v, int i) __attribute__((always_inline)) {
    const TileSrc src = v ? source(p.v, p.sv, tile_of(i)) : source(p.k, p.sk, tile_of(i));
    char* d = smem + grp * 4 * TL + (v ? 2 * TL : 0) + (i & 1) * TL + w * PW * 1024;
#pragma unroll
    for (int j = 0; j < PW; ++j)
      tile_dma(src, d + j * 1024, (int)(((4 * (w * PW + j) + drow) * (v ? p.sv : p.sk)) * 2) + (dcol ^ 16 * j));
  };
  const uint32_t sbase = (uint32_t)(uintptr_t)smem + grp * 4 * TL;
  const uint32_t kb = sbase + rows_lane_off(0);
  uint32_t vb0, vb1;
  tr_lane_offs(vb0, vb1);
  vb0 += sbase + 2 * TL;
  vb1 += sbase + 2 * TL;

  f32x16 o[DT], s[2];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = f32x16{};
  bf16x8 pb[4];
  float m = -INFINITY, muse = 0.f, l = 0.f;  // muse: m, or 0 where all scores so far are minus infinity

  // P.V of one tile and S of the next: eight groups of four fragments, each read while the one before it is multiplied
  auto products = [&](auto PV, auto S, int vbuf, int kbuf) __attribute__((always_inline)) {
    constexpr int first = decltype(PV)::value ? 0 : 4, last = decltype(S)::value ? 8 : 4;
    bf16x8 f[3][4];
    const uint32_t v0 = vb0 + vbuf * TL, v1 = vb1 + vbuf * TL, k = kb + kbuf * TL;
    auto read = [&](auto GC) {
      constexpr int g = decltype(GC)::value;
      static_for<4>([&](auto IC) {
        constexpr int i = decltype(IC)::value;
        if constexpr (g < 4) f[g % 3][i] = tr_x<4096 * (g & 3)>(v0, v1, i);
        else f[g % 3][i] = rows_x<8192 * (i & 1)>(k, 2 * (g - 4) + (i >> 1));
      });
    };
    read(std::integral_constant<int, first>{});
    read(std::integral_constant<int, first + 1>{});
    static_for<8>([&](auto GC) {
      constexpr int g = decltype(GC)::value;
      if constexpr (g >= first && g < last) {
        lds_wait_tie<g + 1 >= last ? 0 : g + 1 < 4 ? 8 : 4>(f[g % 3][0], f[g % 3][1], f[g % 3][2], f[g % 3][3]);
        if constexpr (g + 2 < last) read(std::integral_constant<int, g + 2>{});
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (g < 4) o[i] = mfma(f[g % 3][i], pb[g & 3], o[i]);
          else if (g == 4 && i < 2) s[i] = mfma(f[g % 3][i], qf[0], f32x16{});
          else s[i & 1] = mfma(f[g % 3][i], qf[(2 * (g - 4) + (i >> 1)) & 7], s[i & 1]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    });
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};

  // S of tile kt -> P in bf16, the running maximum and sums. Masked scores are replaced by the power of two that makes 2^28 to
  // 2^29 in the exponent (see attn_fwd_w64_kernel): whatever a key that a row does not see holds, it does not count.
  auto masked_score = [&] { return 0x80000000 | ((127 + 28 + 127 - (__float_as_int(c) >> 23)) << 23); };
  auto softmax = [&](int kt) __attribute__((always_inline)) {
    const int k0 = kt * BN;
    if (k0 + BN > len || k0 + BN - 1 > wq_lo || (p.window > 0 && k0 <= wq_hi - p.window) || wq_hi >= len) {
      const int masked = masked_score();
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int base = k0 + 32 * t + 4 * h, A = base - klo, B = khi - base;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int ar = (r & 3) + 8 * (r >> 2), pen = ((A + ar) | (B - ar)) >> 31;  // -1 outside [lo, hi]
          s[t][r] = __int_as_float((pen & masked) | (~pen & __float_as_int(s[t][r])));
        }
      }
    }
    float t0 = max3_raw(s[0][0], s[0][1], s[0][2]), t1 = max3_raw(s[1][0], s[1][1], s[1][2]);
#pragma unroll
    for (int r = 3; r < 15; r += 2) {
      t0 = max3_raw(t0, s[0][r], s[0][r + 1]);
      t1 = max3_raw(t1, s[1][r], s[1][r + 1]);
    }
    t0 = max3_raw(t0, s[0][15], s[1][15]);
    const float top = xor32_max(max3_raw(t0, t1, t1)) * c;
    if (!__all(top <= m + kDeferThr)) {
      const float next = fmaxf(m, top);
      muse = next == -INFINITY ? 0.f : next;
      const float alpha = fast_exp2(m - muse);
      m = next;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
    }
    float l0 = 0.f, l1 = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        s[t][r] = fast_exp2(__builtin_fmaf(s[t][r], c, -muse));
        s[t][r + 1] = fast_exp2(__builtin_fmaf(s[t][r + 1], c, -muse));
        l0 += s[t][r];
        l1 += s[t][r + 1];
      }
    l += l0 + l1;
    pb[0] = acc_to_b<0>(s[0]);
    pb[1] = acc_to_b<1>(s[0]);
    pb[2] = acc_to_b<0>(s[1]);
    pb[3] = acc_to_b<1>(s[1]);
  };
  auto meet = [] {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  // The groups take turns at the matrix cores: while one multiplies, the other, on the same SIMDs, does its softmax. Turn i
  // of a wave: the softmax of its tile i, then that tile's P.V beside S of the next. Loads of a turn: V of the next tile and
  // K of the one behind it, into the buffers of the last one's. They have a turn to arrive.
  stage(false, 0);
  stage(true, 0);
  if (turns > 1) {
    stage(false, 1);
    asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  if (grp) meet();
  const int mine = max(0, (kt_end_w - kt_begin - grp + 1) / 2);  // tiles of this wave
  if (mine > 0) products(no, yes, 0, 0);
  meet();
  auto stage_next = [&](int i) __attribute__((always_inline)) {
    if (tile_of(i + 2) >= win + 64) load_slots(tile_of(i + 1));
    if (i + 2 < turns) stage(false, i + 2);
    if (i + 1 < turns) stage(true, i + 1);
  };
  // the tiles of the turn's products have arrived for all
  auto arrive = [&](int i) __attribute__((always_inline)) {
    if (i + 2 < turns) asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else if (i + 1 < turns) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  auto turn = [&](int i, auto S, auto STEADY) __attribute__((always_inline)) {  // STEADY: with all of a turn's loads
    if constexpr (STEADY) {
      if (tile_of(i + 2) >= win + 64) load_slots(tile_of(i + 1));
      stage(false, i + 2);
      stage(true, i + 1);
      softmax(tile_of(i));
      asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    } else {
      stage_next(i);
      softmax(tile_of(i));
      arrive(i);
    }
    __builtin_amdgcn_s_setprio(1);
    products(yes, S, i & 1, (i + 1) & 1);
    __builtin_amdgcn_s_setprio(0);
    meet();
  };
  int i = 0;
  for (const int n = min(mine - 1, turns - 2); i < n; ++i) turn(i, yes, yes);
  for (; i + 1 < mine; ++i) turn(i, yes, no);
  if (mine > 0) turn(i++, no, no);
  for (; i < turns; ++i) {  // the others' tiles
    stage_next(i);
    arrive(i);
    meet();
  }
  if (!grp) meet();
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // the second group's part to the first
  l = xor32_sum(l);
  float* part = reinterpret_cast<float*>(smem) + w * (16 * DT * 64);
  float* sums = reinterpret_cast<float*>(smem) + 4 * (16 * DT * 64) + w * 128;
  if (grp) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<f32x4*>(part + ((dt * 4 + r / 4) * 64 + lane) * 4) = f32x4{o[dt][r], o[dt][r + 1], o[dt][r + 2], o[dt][r + 3]};
    sums[lane] = m;
    sums[64 + lane] = l;
  }
  __syncthreads();
  if (grp || myq >= len) return;
  const float m1 = sums[lane], l1 = sums[64 + lane], top = fmaxf(m, m1);
  const float a0 = m == -INFINITY ? 0.f : fast_exp2(m - top), a1 = m1 == -INFINITY ? 0.f : fast_exp2(m1 - top);
  l = l * a0 + l1 * a1;
  // A part that does not count may hold anything (values of masked keys). A sum that is not a number, of a NaN or of plus
  // infinity, and a row that sees minus infinity alone, whose sum is 0 or of masked keys, come out NaN, as softmax gives them.
  const float inv = top <= __int_as_float(masked_score()) * c ? NAN : 1.f / l;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(part + ((dt * 4 + r / 4) * 64 + lane) * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[dt][r + e] = (a0 > 0.f ? o[dt][r + e] * a0 : 0.f) + (a1 > 0.f ? x[e] * a1 : 0.f);
    }
  bf16* op = p.o + (int64_t)(start + myq) * p.so + (int64_t)hq * D;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) store_row_block<D>(op, o[dt], dt, h, inv);
}

}  // namespace

// n: entries of 256 new tokens
int hds_attn_fwd_pair_paged_launch(const void* params, size_t params_bytes, int n, int hq, hipStream_t st) {
  if (params_bytes != sizeof(AttnParams)) return hipErrorInvalidValue;
  const int g = 32 >> std::min(5, __builtin_ctz(hq));
  hipLaunchKernelGGL(attn_fwd_pair_kernel, dim3(2 * g * hq, (n + g - 1) / g), dim3(512), 0, st,
                     *static_cast<const AttnParams*>(params), n);
  return hipGetLastError();
}
