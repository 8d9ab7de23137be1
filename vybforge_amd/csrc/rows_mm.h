// GEMM on packed rows at a few X rows (batched or speculative decode), all six GGUF types, gfx950.
//
// Y[m, n] = RS[m, n] + sum_k X[m, k] * W[n, k],  M <= 64
//
// Bound: the weights' bytes, read once. A workgroup owns a K range of a few super-blocks (256 k) and walks
// tiles of BN weight rows over it:
//  - its X rows are brought into LDS once, in matrix-core operand order (an A operand is one
//    conflict-free 16-byte read per lane), every (row, super-block) scaled into fp16 range by a power of two;
//  - the weights stream through NS stages of one super-block of a tile's rows, copied by direct-to-LDS loads
//    of whole row runs in 16-byte chunks (a lane loading its own unit's window straight from memory
//    touches a line per lane, which kept the address unit busy half of the time), one barrier per
//    stage;
//  - with the K range split, float32 partials are summed in split order by a second launch.
// Lane l decodes unit g = l >> 4 (64 weights, the decode GEMV's units and windows) of weight row l & 15
// into B operands of v_mfma_f32_16x16x32_f16: operand j of a super-block takes 8 weights of each of the
// row's four units. What is common to a super-block stays out of the operands: they hold the exact
// integers sc q (Q4_K, Q5_K: at most 1953), sc (q - 32) (Q6_K: rounded above 2048 only) or
// (2 s + 1) grid (IQ2_S: at most 1333), one packed fma per two weights, and the super-block's float32
// scale multiplies the accumulated sums. The mins of Q4_K / Q5_K are one operand more: the
// sub-blocks' 6-bit mins against their sums of x, split into three fp16 terms. So the weights of these
// types are not rounded at all. q4_0 / Q8_0 have a scale per 32: their operands are d q, one fp16 product.
//
// Measured with the reduce launch, 24 rows bf16, 17408 x 5120 and 5120 x 17408: Q4_K 26.1 and 26.5 us (65 and 136 on the
// 64-row tiles of kqgemm.hip), Q6_K 32.6 and 33.4 (72 and 177), q4_0 23.6 and 24.0 (47 and 86). The loop
// itself streams weights at 4.6 TB/s; the rest is the start (X), the last round of tiles and the
// reduce (~5 us). Non-finite activations give what the sum over k gives: where the mins are subtracted apart from the
// products (Q4_K, Q5_K), an infinity would meet zeros and infinities that the weight itself is not, so a row's
// super-block that holds one is staged as zeros under an infinite scale, and where a tile then holds NaNs, those rows are
// left to the end: their infinities (and NaNs) times whole weights.
#pragma once
#include "gemv_dev.h"

namespace vybdq {

struct RowsArgs {
  const uint8_t *W;
  int64_t rowbytes;
  const void *X;
  int M, N, SB;         // SB: super-blocks (256 k) per row
  int splits, sps;      // splits of K, super-blocks per split
  int tiles, ns;        // column tiles; LDS stages (2..4)
  void *Y;
  int ydt;
  int64_t ldy;
  const void *RS;
  float *part;          // splits > 1: float32 partials [splits][M][N]
};

// k offset within a super-block of run h (32 weights) of unit g
template <bool Q6>
__host__ __device__ constexpr int rows_run_elem(int g, int h) {
  return Q6 ? 128 * (g >> 1) + 64 * h + 32 * (g & 1) : 64 * g + 32 * h;
}

template <int FMT> struct RowsFmt {
  static constexpr int SBB = FMT == FMT_Q4_0 ? 144 : FMT == FMT_Q8_0 ? 272 : FMT == FMT_Q4_K ? 144 : FMT == FMT_Q5_K ? 176
                                                                                : FMT == FMT_Q6_K   ? 210 : 82;
  static constexpr bool ALIGNED = SBB % 16 == 0;
  // 16-byte chunks that cover a super-block: super-blocks of 2-byte alignment start at most 14 bytes in
  static constexpr int C = ALIGNED ? SBB / 16 : (SBB + 14 + 15) / 16;
  static constexpr bool MINS = FMT == FMT_Q4_K || FMT == FMT_Q5_K;
  static constexpr bool SCALED = FMT != FMT_Q4_0 && FMT != FMT_Q8_0;  // a float32 scale per super-block
  static constexpr int OPS = MINS ? 9 : 8;                           // A operands per 16 rows and super-block
};

__device__ __forceinline__ h2 rows_h2(float v) { return h2{static_cast<_Float16>(v), static_cast<_Float16>(v)}; }
__device__ __forceinline__ uint32_t rows_bits(h2 v) { return __builtin_bit_cast(uint32_t, v); }

// The 6-bit scales and mins of sub-blocks 2 g and 2 g + 1 (get_scale_min_k4), as bytes 0 and 1 of each; both forms
// formed, one selected
__device__ __forceinline__ void rows_scales_k4(const uint32_t s0, const uint32_t s1, const uint32_t s2, int g, uint32_t &sc,
                                               uint32_t &mn) {
  const uint32_t sh = 16 * (g & 1), a = s0 >> sh, b = s1 >> sh, c = s2 >> sh;
  const bool lo = g < 2;
  sc = lo ? a & 0x3F3Fu : (c & 0x0F0Fu) | ((a >> 2) & 0x3030u);
  mn = lo ? b & 0x3F3Fu : ((c >> 4) & 0x0F0Fu) | ((b >> 2) & 0x3030u);
}

// bytes A and B of v (below 256) as fp16
template <int A, int B>
__device__ __forceinline__ h2 rows_bytes(uint32_t v) {
  constexpr uint32_t sel = 0x04000400u | A | (B << 16);
  return __builtin_bit_cast(h2, __builtin_amdgcn_perm(C64, v, sel)) - rows_h2(1024.0f);
}

// Run h of unit g from its windows as 16 packed fp16 pairs in k order (see the head of the file)
template <int FMT>
__device__ __forceinline__ void rows_run(const uint32_t (&dw)[Fmt<FMT>::PAIR_DWORDS], int g, int h, uint32_t sc6,
                                         const uint2 *lgrid, uint32_t (&out)[16]) {
  if constexpr (FMT == FMT_Q4_0 || FMT == FMT_Q8_0) {
    constexpr int QDW = Fmt<FMT>::QDW;
    uint32_t q[QDW];
#pragma unroll
    for (int t = 0; t < QDW; ++t) q[t] = h == 0 ? __builtin_amdgcn_alignbit(dw[t + 1], dw[t], 16) : dw[QDW + 1 + t];
    const _Float16 d = __builtin_bit_cast(_Float16, static_cast<uint16_t>(h == 0 ? dw[0] : dw[QDW] >> 16));
    const h2 dd = {d, d}, off = rows_h2(-Fmt<FMT>::CORR);
    h2 wv[16];
    unpack_block<FMT, VYBDQ_Q4_GGML>(q, wv);
#pragma unroll
    for (int i = 0; i < 16; ++i) out[i] = rows_bits((wv[i] + off) * dd);
  } else if constexpr (FMT == FMT_Q4_K || FMT == FMT_Q5_K) {
    // (1024 + q) sc - 1024 sc: both terms and the result are exact fp16 values; Q4_K's high nibbles stay
    // in place, (1024 + 16 q) sc / 16 - 64 sc
    constexpr int QS = FMT == FMT_Q4_K ? 4 : 12;
    const bool hi = FMT == FMT_Q4_K && h == 1;
    const h2 s1 = h == 0 ? rows_bytes<0, 0>(sc6) : rows_bytes<1, 1>(sc6);
    const h2 s = hi ? s1 * rows_h2(0.0625f) : s1, o = s * rows_h2(-1024.0f);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      uint32_t v;
      if (hi) v = dw[QS + t] & 0xF0F0F0F0u;
      else v = h == 0 ? (dw[QS + t] & 0x0F0F0F0Fu) : ((dw[QS + t] >> 4) & 0x0F0F0F0Fu);
      if constexpr (FMT == FMT_Q5_K) v |= ((dw[4 + t] >> (2 * g + h)) & 0x01010101u) << 4;
      h2 a, b;
      bytes_to_h2(v, a, b);
      out[2 * t] = rows_bits(__builtin_elementwise_fma(a, s, o));
      out[2 * t + 1] = rows_bits(__builtin_elementwise_fma(b, s, o));
    }
  } else if constexpr (FMT == FMT_Q6_K) {
    const uint32_t part = g & 1, sh = dw[22], hs = 4 * h + 2 * part;
    const uint32_t scw = __builtin_amdgcn_alignbit(dw[19 + h], dw[18 + h], sh);
    const h2 s0 = rows_h2(static_cast<float>(static_cast<int8_t>(__builtin_amdgcn_ubfe(scw, 16 * part, 8))));
    const h2 s1 = rows_h2(static_cast<float>(static_cast<int8_t>(__builtin_amdgcn_ubfe(scw, 16 * part + 8, 8))));
    const h2 off = rows_h2(-1056.0f);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const uint32_t ql = __builtin_amdgcn_alignbit(dw[t + 1], dw[t], sh);
      const uint32_t qh = __builtin_amdgcn_alignbit(dw[10 + t], dw[9 + t], sh);
      const uint32_t v = (h == 0 ? (ql & 0x0F0F0F0Fu) : ((ql >> 4) & 0x0F0F0F0Fu)) | (((qh >> hs) & 0x03030303u) << 4);
      h2 a, b;
      bytes_to_h2(v, a, b);
      out[2 * t] = rows_bits((a + off) * (t < 4 ? s0 : s1));
      out[2 * t + 1] = rows_bits((b + off) * (t < 4 ? s0 : s1));
    }
  } else {
    // groups 8 g + 4 h + l of 8 weights: grid entry (bytes, LDS) times 2 s + 1, signs XORed in
    const uint32_t sh = dw[9];
    const uint32_t ix = __builtin_amdgcn_alignbit(dw[1 + h], dw[h], sh);
    const uint32_t sg = __builtin_amdgcn_alignbit(dw[4 + h], dw[3 + h], sh);
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      const uint32_t idx = __builtin_amdgcn_ubfe(ix, 8 * l, 8) | (__builtin_amdgcn_ubfe(dw[6], 8 * h + 2 * l, 2) << 8);
      const uint2 e = lgrid[idx];
      const uint32_t sgn = __builtin_amdgcn_ubfe(sg, 8 * l, 8);
      const float sc = static_cast<float>(2 * __builtin_amdgcn_ubfe(dw[7], 8 * h + 4 * (l >> 1), 4) + 1);
      const h2 s = rows_h2(sc), o = rows_h2(-1024.0f * sc);
      h2 p[4];
      bytes_to_h2(e.x, p[0], p[1]);
      bytes_to_h2(e.y, p[2], p[3]);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t s2 = __builtin_amdgcn_ubfe(sgn, 2 * k, 2);  // sign bits 2k, 2k + 1 -> bits 15, 31
        out[4 * l + k] = rows_bits(__builtin_elementwise_fma(p[k], s, o)) ^ (((s2 << 15) | (s2 << 30)) & 0x80008000u);
      }
    }
  }
}

constexpr int kRowsGrid = 1024 * 8;  // IQ2_S: the grid as bytes, at the start of LDS

template <int FMT, int MF, int NW> struct RowsShape {
  using F = RowsFmt<FMT>;
  static constexpr int BN = 16 * NW;
  static constexpr int JW = BN * F::C / 64;  // direct-to-LDS loads per stage (64 chunks each)
  static constexpr int PER = (JW + NW - 1) / NW;  // most per wave
  static constexpr int STAGE = JW * 1024;
  static constexpr int XSB = MF * (F::OPS * 1024 + 64);  // X of a super-block: operands, then row scales
  static constexpr int TAB = FMT == FMT_IQ2_S ? kRowsGrid : 0;
  static_assert(BN * F::C % 64 == 0, "whole loads");
};

typedef unsigned short us2 __attribute__((ext_vector_type(2)));

template <int XDT> struct RowsX { u4 r[XDT == VYBDQ_F32 ? 2 : 1]; };

// Whether row R of the workgroup has a marked super-block (scale infinite, operands zero) in its K range
template <int FMT, int MF>
__device__ __forceinline__ bool rows_marked(const char *xs, int nst, int R) {
  using F = RowsFmt<FMT>;
  constexpr int XSB = MF * (F::OPS * 1024 + 64);
  for (int b = 0; b < nst; ++b)
    if (!(reinterpret_cast<const float *>(xs + b * XSB + MF * F::OPS * 1024)[R] < __builtin_inff())) return true;
  return false;
}

// value of row, col: this K range's partial, or the output
__device__ __forceinline__ void rows_store(const RowsArgs &a, int row, int64_t col, float v) {
  if (a.splits > 1) {
    a.part[(static_cast<int64_t>(blockIdx.y) * a.M + row) * a.N + col] = v;
    return;
  }
  const int64_t i = static_cast<int64_t>(row) * a.ldy + col;
  switch (a.ydt) {
    case VYBDQ_F32: store_elem<VYBDQ_F32>(a.Y, a.RS, i, v); break;
    case VYBDQ_F16: store_elem<VYBDQ_F16>(a.Y, a.RS, i, v); break;
    case VYBDQ_BF16: store_elem<VYBDQ_BF16>(a.Y, a.RS, i, v); break;
    default: store_elem<VYBDQ_F64>(a.Y, a.RS, i, v); break;
  }
}

// The marked rows of a tile, whose accumulators are NaN: their non-finite activations times whole weights (the other
// terms are finite), stored. All lanes of the wave; column col, unit g, split super-blocks sb0 .. sb0 + nst.
template <int FMT, int XDT, int MF>
__device__ __forceinline__ void rows_non_finite(const RowsArgs &a, const char *xs, int sb0, int nst, int m0, int64_t col, int g) {
  using F = RowsFmt<FMT>;
  constexpr int XSB = MF * (F::OPS * 1024 + 64);
#pragma unroll 1
  for (int R = 0; R < 16 * MF && m0 + R < a.M; ++R) {
    if (!rows_marked<FMT, MF>(xs, nst, R)) continue;
    float s = 0.f;
#pragma unroll 1
    for (int b = 0; b < nst; ++b) {
      if (reinterpret_cast<const float *>(xs + b * XSB + MF * F::OPS * 1024)[R] < __builtin_inff()) continue;
      const uint8_t *sb = a.W + col * a.rowbytes + static_cast<int64_t>(sb0 + b) * F::SBB;
      const uint32_t *hd = reinterpret_cast<const uint32_t *>(sb);
      const float d = half_bits_to_f32(hd[0] & 0xffffu), dmin = half_bits_to_f32(hd[0] >> 16);
      uint32_t sc6, mn6;
      rows_scales_k4(hd[1], hd[2], hd[3], g, sc6, mn6);
      const int64_t e0 = ((m0 + R) * static_cast<int64_t>(a.SB) + sb0 + b) * 256 + 64 * g;
#pragma unroll 1
      for (int i = 0; i < 64; ++i) {
        const float x = load_elem<XDT>(a.X, e0 + i);
        if (fabsf(x) < __builtin_inff()) continue;
        const int h = i >> 5, l = i & 31;
        uint32_t q = (sb[(FMT == FMT_Q4_K ? 16 : 48) + 32 * g + l] >> (4 * h)) & 15u;
        if constexpr (FMT == FMT_Q5_K) q |= ((sb[16 + l] >> (2 * g + h)) & 1u) << 4;
        s += x * fmaf(d * static_cast<float>((sc6 >> (8 * h)) & 0xffu), static_cast<float>(q),
                      -dmin * static_cast<float>((mn6 >> (8 * h)) & 0xffu));
      }
    }
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    if (g == 0) rows_store(a, m0 + R, col, s);
  }
}

template <int FMT, int XDT, int MF, int NW, bool GR = false>
__global__ void __launch_bounds__(64 * NW) k_rows_mm(const RowsArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  using Sh = RowsShape<FMT, MF, NW>;
  using F = RowsFmt<FMT>;
  constexpr int PD = Fmt<FMT>::PAIR_DWORDS, PER = Sh::PER;
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int sb0 = blockIdx.y * a.sps, m0 = GR ? blockIdx.z * 16 * MF : 0;  // K range, first row
  const int nst = min(a.sps, a.SB - sb0), NS = a.ns;
  const int ntile = (a.tiles - static_cast<int>(blockIdx.x) + static_cast<int>(gridDim.x) - 1) / static_cast<int>(gridDim.x);
  const int total = ntile * nst;
  char *xs = smem + Sh::TAB, *st0 = xs + a.sps * Sh::XSB;

  // 1. X of (m-fragment, super-block) task q: lane = row n, 16-byte chunk 4 cc + g of the super-block
  const int64_t K = static_cast<int64_t>(a.SB) * 256;
  auto xload = [&](int q, RowsX<XDT> (&v)[8]) {
    const int m = q % MF, sb = sb0 + q / MF, row = min(m0 + 16 * m + n, a.M - 1);
    const int64_t e = row * K + sb * 256 + 8 * g;
#pragma unroll
    for (int cc = 0; cc < 8; ++cc) {
      const u4 *p = reinterpret_cast<const u4 *>(static_cast<const char *>(a.X) + (e + 32 * cc) * (XDT == VYBDQ_F32 ? 4 : 2));
      v[cc].r[0] = p[0];
      if constexpr (XDT == VYBDQ_F32) v[cc].r[1] = p[1];
    }
  };
  auto xval = [](const RowsX<XDT> &k, int i) {
    if constexpr (XDT == VYBDQ_F32) return __uint_as_float(k.r[i >> 2][i & 3]);
    else return __uint_as_float(i & 1 ? k.r[0][i >> 1] & 0xffff0000u : k.r[0][i >> 1] << 16);
  };
  auto xstage = [&](int q, const RowsX<XDT> (&v)[8]) {
    float amax = 0.f;
    if constexpr (XDT == VYBDQ_F32) {
#pragma unroll
      for (int cc = 0; cc < 8; ++cc)
#pragma unroll
        for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(xval(v[cc], i)));
    } else {
      // magnitudes of 16-bit floats order as integers; a NaN only makes its own block's scale its own
      us2 mx = {0, 0};
#pragma unroll
      for (int cc = 0; cc < 8; ++cc)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = __builtin_elementwise_max(mx, __builtin_bit_cast(us2, v[cc].r[0][i] & 0x7fff7fffu));
      const uint32_t m = mx[0] > mx[1] ? mx[0] : mx[1];
      amax = XDT == VYBDQ_F16 ? half_bits_to_f32(m) : __uint_as_float(m << 16);
    }
    amax = fmaxf(amax, __shfl_xor(amax, 16, 64));
    amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
    float inv;
    const float sc = block_scale(amax, inv);
    const bool inf = F::MINS && amax == __builtin_inff();
    char *base = xs + (q / MF) * Sh::XSB + (q % MF) * (F::OPS * 1024);
    if (g == 0) reinterpret_cast<float *>(xs + (q / MF) * Sh::XSB + MF * F::OPS * 1024)[16 * (q % MF) + n] = inf ? amax : sc;
#pragma unroll
    for (int cc = 0; cc < 8; ++cc) {  // block cc of the super-block; this lane's chunk: quarter g
      u4 o;
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        h2 p;
        if constexpr (XDT == VYBDQ_F16) {
          // exact up to float16's subnormals, as through float32; 2^-e may be past float16's range
          const h2 x = __builtin_bit_cast(h2, static_cast<uint32_t>(v[cc].r[0][i]));
          p = h2{static_cast<_Float16>(static_cast<float>(x[0]) * inv), static_cast<_Float16>(static_cast<float>(x[1]) * inv)};
        } else {
          p = h2{static_cast<_Float16>(xval(v[cc], 2 * i) * inv), static_cast<_Float16>(xval(v[cc], 2 * i + 1) * inv)};
        }
        o[i] = __builtin_bit_cast(uint32_t, p);
        if constexpr (F::MINS) s = __builtin_amdgcn_fdot2(p, rows_h2(1.0f), s, false);
      }
      // unit and run of block cc
      constexpr bool Q6 = FMT == FMT_Q6_K;
      const int u = Q6 ? 2 * (cc >> 2) + (cc & 1) : cc >> 1, h = Q6 ? (cc >> 1) & 1 : cc & 1;
      *reinterpret_cast<u4 *>(base + (4 * h + g) * 1024 + (n + 16 * u) * 16) = o;
      if constexpr (F::MINS) {
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
        s *= 0.03125f;
        const _Float16 t0 = static_cast<_Float16>(s);
        const float r1 = s - static_cast<float>(t0);
        const _Float16 t1 = static_cast<_Float16>(r1);
        const _Float16 t2 = static_cast<_Float16>(r1 - static_cast<float>(t1));
        if (g == 0) {
          _Float16 *p = reinterpret_cast<_Float16 *>(base + 8 * 1024 + (n + 16 * u) * 16) + 3 * h;
          p[0] = t0;
          p[1] = t1;
          p[2] = t2;
          if (h == 1) {
            p[3] = static_cast<_Float16>(0.f);
            p[4] = static_cast<_Float16>(0.f);
          }
        }
      }
    }
    if constexpr (F::MINS) {
      asm volatile("" ::: "memory");  // stored after the values above
      if (inf) {  // this lane's operands and sums again, as zeros
        for (int j = 0; j < 8; ++j) *reinterpret_cast<u4 *>(base + (4 * (j & 1) + g) * 1024 + (n + 16 * (j >> 1)) * 16) = u4{0u, 0u, 0u, 0u};
        *reinterpret_cast<u4 *>(base + 8 * 1024 + (n + 16 * g) * 16) = u4{0u, 0u, 0u, 0u};
      }
    }
  };

  // 2. weight stages: load j = wave + NW u of a stage; this lane's chunk is chunk % C of row chunk / C
  const int nj = (Sh::JW - wave + NW - 1) / NW;  // PER or PER - 1
  uint32_t off[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int q = 64 * (wave + NW * u) + lane;
    off[u] = static_cast<uint32_t>((q / F::C) * a.rowbytes) + (F::ALIGNED ? 16 * (q % F::C) : 0);
  }
  const int64_t wend = static_cast<int64_t>(a.N) * a.rowbytes - 16;  // the matrix's last 16-byte chunk
  int it_tile = blockIdx.x, it_sb = 0, it_buf = 0;  // next stage to issue
  auto issue = [&] {
    char *buf = st0 + it_buf * Sh::STAGE;
    const int64_t tb = static_cast<int64_t>(it_tile) * Sh::BN * a.rowbytes;  // a multiple of 16
    const uint32_t so = static_cast<uint32_t>(sb0 + it_sb) * F::SBB;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      if (u < PER - 1 || u < nj) {
        const int j = wave + NW * u;
        if constexpr (F::ALIGNED) {
          lds_dma16_s(a.W + tb + so, off[u], buf + 1024 * j);
        } else {
          // chunks past a super-block of the last row stay inside the matrix
          const uint32_t left = wend - tb < 0xfffffff0 ? static_cast<uint32_t>(wend - tb) : 0xfffffff0u;
          const uint32_t o = ((off[u] + so) & ~15u) + 16 * ((64 * j + lane) % F::C);
          lds_dma16_s(a.W + tb, o < left ? o : left, buf + 1024 * j);
        }
      }
    }
    it_buf = it_buf + 1 < NS ? it_buf + 1 : 0;
    if (++it_sb == nst) {
      it_sb = 0;
      it_tile += gridDim.x;
    }
  };
  auto wait_later = [&](int later) {  // all but the loads of `later` stages have arrived
    auto vm = [](auto k) {
      constexpr int V = decltype(k)::value;
      static_assert(V < 64, "vmcnt range");
      __builtin_amdgcn_s_waitcnt((V & 15) | ((V >> 4) << 14) | (7 << 4) | (15 << 8));
    };
    constexpr int P1 = PER > 0 ? PER - 1 : 0;
    if (later >= 2) {
      if (nj == PER) vm(std::integral_constant<int, 2 * PER>{});
      else vm(std::integral_constant<int, 2 * P1>{});
    } else if (later == 1) {
      if (nj == PER) vm(std::integral_constant<int, PER>{});
      else vm(std::integral_constant<int, P1>{});
    } else {
      vm(std::integral_constant<int, 0>{});
    }
  };
  auto bar = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  };
  {
    const int ntask = MF * nst;
    RowsX<XDT> v[8];
    if (wave < ntask) xload(wave, v);
    __builtin_amdgcn_sched_barrier(0);
    for (int i = 0; i < NS - 1 && i < total; ++i) issue();
    __builtin_amdgcn_sched_barrier(0);
    if (wave < ntask) xstage(wave, v);
    for (int q = wave + NW; q < ntask; q += NW) {
      xload(q, v);
      xstage(q, v);
    }
  }
  const uint2 *lgrid = reinterpret_cast<const uint2 *>(smem);
  if constexpr (FMT == FMT_IQ2_S) {
    const uint2 *grid = reinterpret_cast<const uint2 *>(kIq2sGrid);
    for (int i = threadIdx.x; i < 1024; i += 64 * NW) reinterpret_cast<uint2 *>(smem)[i] = grid[i];
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's LDS stores, before the first stage's barrier

  f4 acc[MF];
#pragma unroll
  for (int m = 0; m < MF; ++m) acc[m] = f4{0.f, 0.f, 0.f, 0.f};
  const int row0 = wave * 16 + n;  // this lane's weight row within the tile
  int tile = blockIdx.x, sbl = 0, cb = 0;
  bool fix = false;  // a tile had rows of marked super-blocks
  for (int z = 0; z < total; ++z) {
    wait_later(min(NS - 2, total - 1 - z));
    bar();
    if (z + NS - 1 < total) issue();  // into the buffer of stage z - 1, which every wave has left
    const char *buf = st0 + cb * Sh::STAGE;
    const char *xb = xs + sbl * Sh::XSB + 16 * lane;
    const f4 *xsc = reinterpret_cast<const f4 *>(xs + sbl * Sh::XSB + MF * F::OPS * 1024);
    uint32_t dw[PD], sc6 = 0, mn6 = 0;
    int sub = 0;
    if constexpr (!F::ALIGNED) sub = (row0 * static_cast<int>(a.rowbytes) + (sb0 + sbl) * F::SBB) & 15;
    load_unit<FMT>(reinterpret_cast<const uint8_t *>(buf) + row0 * (16 * F::C) + sub, g, dw);
    if constexpr (F::MINS) rows_scales_k4(dw[1], dw[2], dw[3], g, sc6, mn6);
    f4 t[MF];
#pragma unroll
    for (int m = 0; m < MF; ++m) t[m] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint32_t out[16];
      rows_run<FMT>(dw, g, h, sc6, lgrid, out);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const h8 b = __builtin_bit_cast(h8, u4{out[4 * q], out[4 * q + 1], out[4 * q + 2], out[4 * q + 3]});
#pragma unroll
        for (int m = 0; m < MF; ++m) {
          const h8 av = *reinterpret_cast<const h8 *>(xb + (m * F::OPS + 4 * h + q) * 1024);
          t[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, b, t[m], 0, 0, 0);
        }
      }
    }
    // acc += row scale * (d t - dmin u)
    float d = 1.f, dm = 0.f;
    h8 mb{};
    if constexpr (F::MINS) {
      d = half_bits_to_f32(dw[0] & 0xffffu);
      dm = -32.0f * half_bits_to_f32(dw[0] >> 16);
      mb = __builtin_bit_cast(h8, u4{rows_bits(rows_bytes<0, 0>(mn6)), rows_bits(rows_bytes<0, 1>(mn6)),
                                     rows_bits(rows_bytes<1, 1>(mn6)), 0u});
    } else if constexpr (FMT == FMT_Q6_K) {
      d = half_bits_to_f32(dw[21]);
    } else if constexpr (FMT == FMT_IQ2_S) {
      d = half_bits_to_f32(dw[8]) * 0.125f;
    }
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      const f4 sc = xsc[4 * m + g];
      f4 u = f4{0.f, 0.f, 0.f, 0.f};
      if constexpr (F::MINS) {
        const h8 av = *reinterpret_cast<const h8 *>(xb + (m * F::OPS + 8) * 1024);
        u = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, mb, u, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = F::SCALED ? d * t[m][r] : t[m][r];
        if constexpr (F::MINS) v = fmaf(dm, u[r], v);
        acc[m][r] = fmaf(sc[r], v, acc[m][r]);
      }
    }
    cb = cb + 1 < NS ? cb + 1 : 0;
    if (++sbl < nst) continue;
    // acc[m][r] = C[m0 + 16 m + 4 g + r][BN tile + row0]
    const int64_t col = static_cast<int64_t>(tile) * Sh::BN + row0;
    int lim = a.M;
    if constexpr (F::MINS) {
      bool nan = false;
#pragma unroll
      for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) nan |= acc[m][r] != acc[m][r];
      if (__any(nan)) {  // stored here but for the marked rows, which follow the last tile
        fix = true;
        lim = 0;
#pragma unroll 1
        for (int i = 0; i < 4 * MF; ++i) {
          float v = 0.f;
#pragma unroll
          for (int m = 0; m < MF; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) v = i == 4 * m + r ? acc[m][r] : v;
          const int R = 16 * (i >> 2) + 4 * g + (i & 3);
          if (m0 + R < a.M && !rows_marked<FMT, MF>(xs, nst, R)) rows_store(a, m0 + R, col, v);
        }
      }
    }
#pragma unroll
    for (int m = 0; m < MF; ++m) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + 16 * m + 4 * g + r;
        if (row < lim) rows_store(a, row, col, acc[m][r]);
      }
      acc[m] = f4{0.f, 0.f, 0.f, 0.f};
    }
    sbl = 0;
    tile += gridDim.x;
  }
  if constexpr (F::MINS) {
    if (fix) {
      // Arguments and lane are read again, so that nothing here is computed ahead of the tile loop or kept over it: inside
      // the loop, with its values shared, this took 5 to 10% of every call of 49 to 64 rows (Q4_K 17408 x 5120, 64 rows
      // 40.7 us; like this 37.8, without it 37.0).
      const RowsArgs *ap = (const RowsArgs *)__builtin_amdgcn_kernarg_segment_ptr();
      int tid = threadIdx.x;
      char *sm = smem;
      asm volatile("" : "+s"(ap), "+v"(tid), "+v"(sm));
      const int s0 = blockIdx.y * ap->sps;
      for (int t = blockIdx.x; t < ap->tiles; t += gridDim.x)
        rows_non_finite<FMT, XDT, MF>(*ap, sm + Sh::TAB, s0, min(ap->sps, ap->SB - s0), GR ? blockIdx.z * 16 * MF : 0,
                                      static_cast<int64_t>(t) * Sh::BN + (tid >> 6) * 16 + (tid & 15), (tid & 63) >> 4);
    }
  }
}

}  // namespace vybdq
