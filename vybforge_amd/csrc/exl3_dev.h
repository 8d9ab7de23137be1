// EXL3 4-bpw trellis device helpers shared by the fused GEMM (exl3.hip) and the grouped MoE
// experts (moe_exl3.hip): the lane windows of a 16x16 tile's stream, the mcg hash decode through
// the tile-slot composition table, and the 128-point FWHT across a wave. Format and decode:
// native/exl3/README.md:24-49, native/exl3/exl3_ref.py:1-120 (see exl3.hip's header).
#pragma once

#include "common.h"

namespace vybdq {

#include "exl3_slots.inc"

constexpr float kRScale = 0.08838834764831845f;  // 1/sqrt(128)

// bits [o, o+32) of the 192-bit lane window w[0..5] (o is a constant after unrolling)
__device__ __forceinline__ uint32_t win_extract(const uint32_t (&w)[6], int o) {
  const int i = o >> 5, s = o & 31;
  if (s == 0) return w[i];
  if (i == 5) return w[5] >> s;
  return __builtin_amdgcn_alignbit(w[i + 1], w[i], s);
}

// mcg hash of the 16-bit window in half HI of d (the other half is ignored): x = w * 0xCBAC1FED
// mod 2^32 from two full-rate 16 x 16-bit products, c = (w * 0xCBAC) << 16 (the multiply writes
// its low 16 bits to the high half through its SDWA destination select) and x = w * 0x1FED + c
// (v_mad_u32_u16, whose op_sel takes the window from either half). Written out because the
// compiler would merge the products into one quarter-rate 32-bit multiply, or shift and add
// separately.
template <bool HI>
__device__ __forceinline__ uint32_t mcg_hash(uint32_t d) {
  uint32_t c, x;
  if constexpr (HI) {
    asm("v_mul_u32_u24_sdwa %0, %1, %2 dst_sel:WORD_1 dst_unused:UNUSED_PAD src0_sel:WORD_1 src1_sel:DWORD"
        : "=v"(c) : "v"(d), "s"(0xCBACu));
    asm("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(x) : "v"(d), "s"(0x1FEDu), "v"(c));
  } else {
    asm("v_mul_u32_u24_sdwa %0, %1, %2 dst_sel:WORD_1 dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:DWORD"
        : "=v"(c) : "v"(d), "s"(0xCBACu));
    asm("v_mad_u32_u16 %0, %1, %2, %3" : "=v"(x) : "v"(d), "s"(0x1FEDu), "v"(c));
  }
  return x;
}

// The mcg hash of a window (its low 16 bits; higher bits are ignored) up to the two fp16 halves
// (before they are added).
__device__ __forceinline__ uint32_t decode_window_halves(uint32_t w) {
  return (mcg_hash<false>(w) & 0x8FFF8FFFu) ^ 0x3B603B60u;
}

// Lane slot q's window hashed up to the two fp16 halves. A one-piece window at a 16-bit boundary
// is hashed straight from its stream dword; other one-piece windows are funnel-extracted without
// a mask (the hash reads only the low 16 bits); two-piece windows are assembled from their masks.
__device__ __forceinline__ uint32_t slot_halves(const uint32_t (&w)[6], int q) {
  const int o = kExl3SlotOff0[q];
  const bool one = kExl3SlotOff1[q] < 0 && kExl3SlotMask0[q] == 0xffffu;
  if (one && (o & 15) == 0) {
    const uint32_t x = (o & 16) ? mcg_hash<true>(w[o >> 5]) : mcg_hash<false>(w[o >> 5]);
    return (x & 0x8FFF8FFFu) ^ 0x3B603B60u;
  }
  if (one) return decode_window_halves(win_extract(w, o));
  // A two-piece window whose first piece runs to the end of its stream dword and whose second
  // piece starts a dword is one funnel shift of those two dwords (the second above the first).
  const unsigned m0 = kExl3SlotMask0[q];
  const int n = __builtin_popcount(m0), o1 = kExl3SlotOff1[q];
  if (o1 >= 0 && m0 == (1u << n) - 1 && (o & 31) + n == 32 && ((o1 + n) & 31) == 0 &&
      kExl3SlotMask1[q] == (0xffffu & ~m0))
    return decode_window_halves(__builtin_amdgcn_alignbit(w[(o1 + n) >> 5], w[o >> 5], o & 31));
  uint32_t x = win_extract(w, o) & kExl3SlotMask0[q];
  if (kExl3SlotOff1[q] >= 0) x |= win_extract(w, kExl3SlotOff1[q]) & kExl3SlotMask1[q];
  return decode_window_halves(x);
}

// The 32 values of lane j: val[q] = row q of column j (q < 16), row q-16 of column j+8. Both
// halves of a hash lie in [0.125, 2), so their float32 sum is exact and one fp16 add rounds it as
// the reference's float32-sum-then-round does.
__device__ __forceinline__ void lane_decode(const uint32_t (&w)[6], _Float16 (&val)[32]) {
#pragma unroll
  for (int q = 0; q < 32; ++q) {
    const h2 v = __builtin_bit_cast(h2, slot_halves(w, q));
    val[q] = v[0] + v[1];
  }
}

// Load tile `tile`'s chunk for lane j (of the 8 lanes sharing it) and build the lane window.
__device__ __forceinline__ void lane_window(const uint16_t *__restrict__ trellis, int64_t tile, int j,
                                            uint32_t (&w)[6]) {
  const u4 c = *reinterpret_cast<const u4 *>(trellis + tile * 64 + 8 * j);
  w[0] = 0;  // stream dword 4j-2: no window reads it (checked by the generator)
  w[2] = c[0];
  w[3] = c[1];
  w[4] = c[2];
  w[5] = c[3];
  // stream dword 4j-1 = lane j-1's last chunk dword (lane 7's for j = 0)
  const int lane = threadIdx.x & 63;
  const int src = (lane & ~7) | ((lane - 1) & 7);
  w[1] = __shfl(c[3], src, 64);
}

// The lane window from an already loaded chunk c: dword 1 is lane j-1's last chunk dword (lane
// 7's for j = 0), taken by DPP row shifts (lane - 1, or lane + 7 for j = 0).
__device__ __forceinline__ void chunk_window(const u4 c, uint32_t (&w)[6]) {
  const int j = threadIdx.x & 7;
  const int prev = __builtin_amdgcn_update_dpp(0, static_cast<int>(c[3]), DPP_ROW_SHR + 1, 0xf, 0xf, false);
  const int wrap = __builtin_amdgcn_update_dpp(0, static_cast<int>(c[3]), DPP_ROW_SHL + 7, 0xf, 0xf, false);
  w[0] = 0;
  w[1] = static_cast<uint32_t>(j == 0 ? wrap : prev);
  w[2] = c[0];
  w[3] = c[1];
  w[4] = c[2];
  w[5] = c[3];
}

// ---- trellis straight into matrix-core operands -------------------------------------------------
//
// A tile's stream dword 4 j + i (i = 0..3 of lane chunk j, its predecessor above it) holds the
// windows of rows 2 i, 2 i + 1, 2 i + 8, 2 i + 9 of column j (shifts 28, 24, 20, 16) and of column
// j + 8 (shifts 12, 8, 4, 0): the four words of either column, two fp16 halves each, are a lane's
// whole B operand of v_mfma_f32_16x16x32_f16 (k' = 8 group + 2 row + half). So nothing is
// regrouped through LDS and nothing is added or packed on the VALU: the matrix core adds x lo + x hi in
// float32. Shifts s and s + 16 are the two halves of one funnel shift, so eight windows take three
// of them. Instructions per weight: 2 hash products, 1 mask and xor, 3/8 windows = 3.4 for the decode; 4.0 with the
// neighbours' dwords, the operands of x and the matrix instructions (8 per 32 weights of a lane).

// the eight windows of dword d (predecessor p), hashed up to their fp16 halves: a = column j, b = column j + 8
__device__ __forceinline__ void dword_halves(uint32_t p, uint32_t d, u4 &a, u4 &b) {
  auto fin = [](uint32_t x) { return (x & 0x8FFF8FFFu) ^ 0x3B603B60u; };
  const uint32_t w12 = __builtin_amdgcn_alignbit(p, d, 12), w8 = __builtin_amdgcn_alignbit(p, d, 8),
                 w4 = __builtin_amdgcn_alignbit(p, d, 4);
  a = u4{fin(mcg_hash<true>(w12)), fin(mcg_hash<true>(w8)), fin(mcg_hash<true>(w4)), fin(mcg_hash<true>(d))};
  b = u4{fin(mcg_hash<false>(w12)), fin(mcg_hash<false>(w8)), fin(mcg_hash<false>(w4)), fin(mcg_hash<false>(d))};
}

constexpr int kExl3Step = 4;  // k-blocks of 16 rows per step of exl3_mma_run

// A workgroup barrier for LDS alone: waits for this wave's LDS accesses, not for its loads in flight
// (the release fence of __syncthreads() may wait for those).
__device__ __forceinline__ void exl3_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}

// One wave: acc += x' (at most 16 rows) times `nsteps` steps of 64 k of 128 columns (eight tiles per
// k-block). Lane l: k-block l >> 4 of the step, chunk l & 7 of the tile pair's tile (l >> 3) & 1, so
// each 16-byte load instruction covers 256 contiguous bytes of four k-blocks, the four pairs of a
// step whole 1 KB runs. `base`: the first step's first tile (wave-uniform); `kstride`: uint16 from
// one k-block to the next; aload(st, v): step st's 16 x' values (k-block l >> 4 of the step) of row
// l & 15 (any finite or other values for rows past the group: they reach only outputs that are not
// stored), a step ahead if AHEAD (x' in memory) or at the step (x' in LDS); ready() runs between the
// first trellis loads and the first aload (it may stage x' in LDS and wait for it: the trellis loads
// stay in flight across an exl3_barrier). acc[2 c + h][r] = z[row 4 (l >> 4) + r][exl3_mma_col(c, h, l)].
// A step of loads (4 KB per wave) is in flight per lane; each slot is refilled right after its use,
// pinned by scheduling barriers (sunk to the end of the step it would leave no load in flight). Two steps in flight
// (114 VGPRs, four waves per SIMD) measured 3% slower, both where this form has five waves per SIMD (up to 8 rows) and where
// the partials of 16 rows (33 KB of LDS) leave four workgroups per CU, one wave of each per SIMD.
template <bool AHEAD, class Ready, class ALoad>
__device__ __forceinline__ void exl3_mma_run(const uint16_t *__restrict__ base, int64_t kstride, int nsteps,
                                             const Ready &ready, const ALoad &aload, f4 (&acc)[8]) {
  if (nsteps <= 0) {
    ready();
    return;
  }
  const int lane = threadIdx.x & 63, n = lane & 15;
  const uint16_t *lp = base + (lane >> 4) * kstride + 8 * n;
  // Steps in flight. (A loop over steps alone is the same program, but the compiler then peels the last one: 0.5 to 1.8% slower.)
  constexpr int R = 1;
  u4 ring[R][4], xr[AHEAD ? R : 1][2];
  auto wload = [&](int st, int c) {
    const int sc = st < nsteps ? st : nsteps - 1;  // in range: re-read the last
    return *reinterpret_cast<const u4 *>(lp + kExl3Step * kstride * sc + 128 * c);
  };
#pragma unroll
  for (int d = 0; d < R; ++d)
#pragma unroll
    for (int c = 0; c < 4; ++c) ring[d][c] = wload(d, c);
  __builtin_amdgcn_sched_barrier(0);
  ready();
  if constexpr (AHEAD) {
#pragma unroll
    for (int d = 0; d < R; ++d) aload(d < nsteps ? d : nsteps - 1, xr[d]);
  }
  auto step = [&](int st, u4 (&rw)[4], u4 (&rx)[2]) {
    if constexpr (!AHEAD) aload(st, rx);
    // A of dword i: rows 2 i, 2 i + 1, 2 i + 8, 2 i + 9 of the lane's k-block, each value twice
    h8 a[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      a[i] = __builtin_bit_cast(h8, u4{__builtin_amdgcn_perm(rx[0][i], rx[0][i], 0x01000100u),
                                       __builtin_amdgcn_perm(rx[0][i], rx[0][i], 0x03020302u),
                                       __builtin_amdgcn_perm(rx[1][i], rx[1][i], 0x01000100u),
                                       __builtin_amdgcn_perm(rx[1][i], rx[1][i], 0x03020302u)});
    if constexpr (AHEAD) aload(st + R < nsteps ? st + R : nsteps - 1, rx);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      uint32_t w[6];
      chunk_window(rw[c], w);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        u4 b0, b1;
        dword_halves(w[i + 1], w[i + 2], b0, b1);
        acc[2 * c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], __builtin_bit_cast(h8, b0), acc[2 * c], 0, 0, 0);
        acc[2 * c + 1] =
            __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], __builtin_bit_cast(h8, b1), acc[2 * c + 1], 0, 0, 0);
      }
      rw[c] = wload(st + R, c);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int st = 0;
  for (; st + R <= nsteps; st += R) {
#pragma unroll
    for (int d = 0; d < R; ++d) step(st + d, ring[d], xr[AHEAD ? d : 0]);
  }
}

// column (of the 128) of accumulator 2 c + h in lane l
__device__ __forceinline__ int exl3_mma_col(int c, int h, int l) {
  return 32 * c + 16 * ((l >> 3) & 1) + (l & 7) + 8 * h;
}

// the wave's accumulators to its rows of the workgroup's partials [4 waves][rows][kExl3RedStride];
// rows past B are not written
constexpr int kExl3RedStride = 132;  // 4 floats of padding: the four row groups fall on different banks
__device__ __forceinline__ void exl3_mma_store(const f4 (&acc)[8], float *red, int B) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int b = 4 * (lane >> 4) + r;
    if (b < B)
#pragma unroll
      for (int q = 0; q < 8; ++q) red[b * kExl3RedStride + exl3_mma_col(q >> 1, q & 1, lane)] = acc[q][r];
  }
}

// ---- 128-point FWHT across a wave (2 elements per lane) -------------------------------------

// The value of lane ^ M. M = 1, 2: a quad permutation; M = 4, 8: a row shift each way, picked by
// the lane's bit M (both on the VALU); M = 16, 32: ds_bpermute.
template <int M>
__device__ __forceinline__ float xor_lane(float v, bool upper) {
  const int b = __builtin_bit_cast(int, v);
  if constexpr (M == 1) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, b, DPP_QUAD_XOR1, 0xf, 0xf, false));
  } else if constexpr (M == 2) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, b, DPP_QUAD_XOR2, 0xf, 0xf, false));
  } else if constexpr (M == 4 || M == 8) {
    const int hi = __builtin_amdgcn_update_dpp(0, b, DPP_ROW_SHL + M, 0xf, 0xf, false);  // lane + M
    const int lo = __builtin_amdgcn_update_dpp(0, b, DPP_ROW_SHR + M, 0xf, 0xf, false);  // lane - M
    return __builtin_bit_cast(float, upper ? lo : hi);
  } else {
    return __shfl_xor(v, M, 64);
  }
}

template <int M>
__device__ __forceinline__ void fwht_stage(float &a0, float &a1, int lane) {
  const bool upper = (lane & M) != 0;
  const float p0 = xor_lane<M>(a0, upper), p1 = xor_lane<M>(a1, upper);
  a0 = upper ? p0 - a0 : a0 + p0;
  a1 = upper ? p1 - a1 : a1 + p1;
}

__device__ __forceinline__ void fwht128_wave(float &a0, float &a1) {
  const int lane = threadIdx.x & 63;
  float t0 = a0 + a1, t1 = a0 - a1;
  a0 = t0;
  a1 = t1;
  fwht_stage<1>(a0, a1, lane);
  fwht_stage<2>(a0, a1, lane);
  fwht_stage<4>(a0, a1, lane);
  fwht_stage<8>(a0, a1, lane);
  fwht_stage<16>(a0, a1, lane);
  fwht_stage<32>(a0, a1, lane);
}

}  // namespace vybdq
