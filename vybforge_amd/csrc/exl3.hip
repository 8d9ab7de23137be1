// EXL3 4-bpw trellis decode, full dequant and the fused GEMM (batch 1..16), gfx950.
//
// Format (native/exl3/README.md:24-49, native/exl3/exl3_ref.py:1-120): W [K, N] stored as
// 16x16 tiles, trellis uint16 [K/16][N/16][64] (256 nibbles per tile, LSB-first), suh fp16 [K],
// svh fp16 [N]. Tile slot (r, c) takes a 16-bit window of the tile's nibble stream through the
// tile-slot composition table and decodes it with the mcg codebook hash (exllamav3's
// decode_3inst at cb=1, the only codebook the reference implements: native/exl3/exl3_ref.py:19-22,
// native/kernels/exl3.vyb:15-19):
//   x = w * 0xCBAC1FED (mod 2^32);  y = (x & 0x8FFF8FFF) ^ 0x3B603B60;
//   value = fp16(fp16(y.lo) + fp16(y.hi))
// Both halves of y always lie in [0.125, 2), so their float32 sum is exact and one fp16 add
// (round to nearest even) equals the reference's float32-sum-then-round.
// W = diag(suh) (H/sqrt(128)) What (H/sqrt(128)) diag(svh) per 128x128 block, H = Sylvester
// Hadamard-128, so x W = FWHT(FWHT(x * suh)/sqrt(128) What)/sqrt(128) * svh per 128 chunk.
//
// Lane decomposition of the decode-only kernels (exl3_slots.inc, generated and checked by
// gen_exl3_slots.py; the fused GEMM's is in exl3_dev.h): 8 lanes share a tile; lane j owns columns j and j+8 (32 values), loads the tile's 16-byte chunk j (stream
// dwords 4j..4j+3) and takes dword 4j-1 from its neighbour by a shuffle; every window is one or
// two constant-offset funnel extracts of those 5 dwords. A wave covers 8 consecutive tiles along
// N (one 128-column Hadamard block) and reads 1 KB of contiguous trellis per step.
#include "exl3_dev.h"

#include <algorithm>
#include <cstdlib>

namespace vybdq {

// one launch (x rotation per workgroup, output rotation by the last split) up to batch 2; at
// batch 3..16 the per-workgroup rotation of every batch row costs more than the two extra
// launches (batch 16 measured 39 us with k_exl3_xprep / k_exl3_out, 68 us in one launch)
__host__ __device__ constexpr bool exl3_fused(int BP) { return BP <= 2; }
// LDS of the fused GEMM: batch <= 2 the x' stage of a split (fp16, rows exl3_xstride apart), reused
// after the loop for the waves' partials [4][batch rows][kExl3RedStride]; larger batches those alone
__host__ __device__ constexpr int exl3_xstride(int kbs) { return 16 * kbs + 8; }
constexpr size_t kExl3MaxLds = 160 * 1024 - 256;  // dynamic, beside the kernel's static words
static size_t exl3_lds_bytes(int BP, int kbs) {
  const size_t main = exl3_fused(BP) ? static_cast<size_t>(BP) * exl3_xstride(kbs) * 2 : 0;
  const size_t red = static_cast<size_t>(4) * BP * kExl3RedStride * 4;
  return main > red ? main : red;
}

// ---- decode-only: rotated basis What [K, N] ------------------------------------------------

template <int ODT>
__global__ void __launch_bounds__(256) k_exl3_decode(const uint16_t *__restrict__ trellis, void *__restrict__ out,
                                                     int64_t ntiles, int NB) {
  const int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t tile = g >> 3;
  const int j = static_cast<int>(g & 7);
  const int64_t safe = tile < ntiles ? tile : 0;  // every lane joins the shuffle
  uint32_t w[6];
  lane_window(trellis, safe, j, w);
  _Float16 v[32];
  lane_decode(w, v);
  if (tile >= ntiles) return;
  const int64_t kb = tile / NB, nb = tile % NB;
  const int64_t N = static_cast<int64_t>(NB) * 16;
#pragma unroll
  for (int q = 0; q < 32; ++q) {
    const int64_t r = 16 * kb + (q & 15);
    const int64_t c = 16 * nb + j + (q >> 4) * 8;
    store_elem<ODT>(out, nullptr, r * N + c, static_cast<float>(v[q]));
  }
}

// ---- full dequant: W [K, N] = diag(suh) Hs What Hs diag(svh) -------------------------------
// One workgroup per 128x128 block: decode the 64 tiles into LDS (float, rows padded to 129),
// FWHT every row, then every column, scale, store.

template <int ODT>
__global__ void __launch_bounds__(256) k_exl3_dequant(const uint16_t *__restrict__ trellis,
                                                      const _Float16 *__restrict__ suh,
                                                      const _Float16 *__restrict__ svh, void *__restrict__ out,
                                                      int NB) {
  extern __shared__ float blk[];  // [128][129]
  const int bk = blockIdx.y, bn = blockIdx.x;
  const int64_t N = static_cast<int64_t>(NB) * 16;
  for (int task = threadIdx.x; task < 512; task += blockDim.x) {  // 64 tiles x 8 lanes
    const int tl = task >> 3, j = task & 7;
    const int tk = tl >> 3, tn = tl & 7;
    const int64_t tile = static_cast<int64_t>(8 * bk + tk) * NB + (8 * bn + tn);
    uint32_t w[6];
    lane_window(trellis, tile, j, w);
    _Float16 v[32];
    lane_decode(w, v);
#pragma unroll
    for (int q = 0; q < 32; ++q)
      blk[(16 * tk + (q & 15)) * 129 + 16 * tn + j + (q >> 4) * 8] = static_cast<float>(v[q]);
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int row = wave; row < 128; row += 4) {  // column transform: What_row . Hs
    float a0 = blk[row * 129 + 2 * lane], a1 = blk[row * 129 + 2 * lane + 1];
    fwht128_wave(a0, a1);
    blk[row * 129 + 2 * lane] = a0 * kRScale;
    blk[row * 129 + 2 * lane + 1] = a1 * kRScale;
  }
  __syncthreads();
  for (int col = wave; col < 128; col += 4) {  // row transform: Hs . (.)
    float a0 = blk[(2 * lane) * 129 + col], a1 = blk[(2 * lane + 1) * 129 + col];
    fwht128_wave(a0, a1);
    const float sv = static_cast<float>(svh[128 * bn + col]);
    const int64_t r0 = 128 * static_cast<int64_t>(bk) + 2 * lane;
    store_elem<ODT>(out, nullptr, r0 * N + 128 * bn + col, a0 * kRScale * static_cast<float>(suh[r0]) * sv);
    store_elem<ODT>(out, nullptr, (r0 + 1) * N + 128 * bn + col,
                    a1 * kRScale * static_cast<float>(suh[r0 + 1]) * sv);
  }
}

// ---- fused GEMM ------------------------------------------------------------------------------
// grid (N/128 column blocks, S k-splits), 4 waves per workgroup; a split's k-range is whole 128
// chunks.
// 1. x' [BP][k-range] = FWHT(x * suh) / sqrt(128) per 128 chunk. Batch <= 2: computed by the
//    GEMM workgroup itself for its k-range, in LDS; larger batches: by k_exl3_xprep into the
//    workspace (a workgroup would otherwise rotate BP chunks per wave before its first weight).
// 2. z[b][n] over the split's k-range = sum x'[b][k] What[k][n]: each wave a quarter of the
//    k-range on the block's 128 columns (exl3_mma_run: trellis words straight into matrix-core
//    operands, every batch size), the waves' partials summed in LDS in a fixed order. Bound by the
//    hash on the VALU (4.0 instructions per weight, 80% of the issue slots while it runs) and, at one row,
//    by ~8 us per call that do not scale with K (x rotation, arrival, output rotation). K = 5120,
//    N = 17408: batch 16 23 us (29.2 with the decoded words regrouped through LDS, 7.3
//    instructions per weight), batch 1 19.3 (20.5 with one dot product per weight and lane, 5.0).
// 3. y[b][n] = svh[n] * FWHT(sum_s z_s[b][.]) / sqrt(128), sums in split order. Batch <= 2: the
//    last split of a column block to arrive (a per-block arrival counter, reset by that last
//    arrival so the counters stay zero between calls) does it; larger batches: k_exl3_out.
//    The single-launch form publishes the partials with device-coherent stores (written
//    through the XCD's L2) that have completed (s_waitcnt vmcnt(0)) before the arrival is
//    counted, and the last arrival reads them with device-coherent loads issued after the
//    count has returned. An agent-scope release/acquire pair around the count would instead
//    write back and invalidate whole L2s: measured 17 us more per call at batch 1.

template <int XDT>
__global__ void __launch_bounds__(64) k_exl3_xprep(const void *__restrict__ X, const _Float16 *__restrict__ suh,
                                                   _Float16 *__restrict__ xp, int64_t K) {
  const int chunk = blockIdx.x, b = blockIdx.y, lane = threadIdx.x;
  const int64_t k0 = 128 * static_cast<int64_t>(chunk) + 2 * lane;
  float a0 = load_elem<XDT>(X, b * K + k0) * static_cast<float>(suh[k0]);
  float a1 = load_elem<XDT>(X, b * K + k0 + 1) * static_cast<float>(suh[k0 + 1]);
  fwht128_wave(a0, a1);
  xp[b * K + k0] = static_cast<_Float16>(a0 * kRScale);
  xp[b * K + k0 + 1] = static_cast<_Float16>(a1 * kRScale);
}

template <bool FUSED>
__global__ void __launch_bounds__(256, 5) k_exl3_gemm(const uint16_t *__restrict__ trellis, const void *__restrict__ X,
                                                      int xdt, const _Float16 *__restrict__ suh,
                                                      const _Float16 *__restrict__ svh, void *__restrict__ Y, int ydt,
                                                      int B, int BP, const _Float16 *__restrict__ xp,
                                                      float *__restrict__ zpart, uint32_t *__restrict__ arrivals,
                                                      int64_t K, int NB, int kb_per_split) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ int is_last;
  const int g = blockIdx.x, s = blockIdx.y, S = gridDim.y;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int KB = static_cast<int>(K / 16);
  const int kb_begin = s * kb_per_split;
  const int kb_end = min(kb_begin + kb_per_split, KB);
  const int nkb = kb_end - kb_begin;
  // this wave's 64-k steps of the split
  const int nst = nkb / kExl3Step;
  const int st0 = nst * wave / 4, st1 = nst * (wave + 1) / 4;
  const int kb0 = kb_begin + kExl3Step * st0;
  const int64_t kstride = static_cast<int64_t>(NB) * 64;
  const uint16_t *base = trellis + kb0 * kstride + 512 * static_cast<int64_t>(g);
  const int am = lane & 15;
  f4 acc[8];
#pragma unroll
  for (int f = 0; f < 8; ++f) acc[f] = f4{0.f, 0.f, 0.f, 0.f};
  if constexpr (FUSED) {
    // 1. x' rows of this split: [B][16 nkb] fp16 in LDS; wave w rotates the 128-chunks w, w + 4, ...
    // of all rows (batch row cb / nch). The raw x and suh words of its first kXP chunks are read before the
    // trellis ring: loads return in order, so the rotation waits for these alone. (x elements k,
    // k + 1: two f32 words, or one word of two 16-bit halves; suh likewise. Kept raw: converting them
    // here would wait.)
    constexpr int kXP = 2;
    _Float16 *xs = reinterpret_cast<_Float16 *>(smem);
    const int xst = exl3_xstride(kb_per_split), nch = nkb / 8, ntask = B * nch;
    auto x_raw = [&](int cb, uint32_t (&xv)[2], uint32_t &sv) {
      const int b = cb / nch, c = cb - b * nch;
      const int64_t k = 16 * static_cast<int64_t>(kb_begin) + 128 * c + 2 * lane, i = static_cast<int64_t>(b) * K + k;
      if (xdt == VYBDQ_F32) __builtin_memcpy(xv, static_cast<const float *>(X) + i, 8);
      else __builtin_memcpy(xv, static_cast<const uint16_t *>(X) + i, 4);
      __builtin_memcpy(&sv, suh + k, 4);
    };
    auto rotate = [&](int cb, const uint32_t (&xv)[2], uint32_t sv) {  // one 128-chunk, whole wave
      const int b = cb / nch, c = cb - b * nch;
      float a0, a1;
      if (xdt == VYBDQ_F32) { a0 = __uint_as_float(xv[0]); a1 = __uint_as_float(xv[1]); }
      else if (xdt == VYBDQ_F16) { a0 = half_bits_to_f32(xv[0] & 0xffffu); a1 = half_bits_to_f32(xv[0] >> 16); }
      else { a0 = __uint_as_float(xv[0] << 16); a1 = __uint_as_float(xv[0] & 0xffff0000u); }
      a0 *= half_bits_to_f32(sv & 0xffffu);
      a1 *= half_bits_to_f32(sv >> 16);
      fwht128_wave(a0, a1);
      *reinterpret_cast<h2 *>(xs + b * xst + 128 * c + 2 * lane) =
          h2{static_cast<_Float16>(a0 * kRScale), static_cast<_Float16>(a1 * kRScale)};
    };
    uint32_t xw[kXP][2], sw[kXP];
#pragma unroll
    for (int it = 0; it < kXP; ++it)
      if (wave + 4 * it < ntask) x_raw(wave + 4 * it, xw[it], sw[it]);
    __builtin_amdgcn_sched_barrier(0);
    const _Float16 *arow = xs + (am < B ? am : 0) * xst + 16 * (kb0 - kb_begin + (lane >> 4));
    exl3_mma_run<false>(base, kstride, st1 - st0,
                 [&] {
#pragma unroll
                   for (int it = 0; it < kXP; ++it)
                     if (wave + 4 * it < ntask) rotate(wave + 4 * it, xw[it], sw[it]);
                   for (int cb = wave + 4 * kXP; cb < ntask; cb += 4) {
                     uint32_t xv[2], sv;
                     x_raw(cb, xv, sv);
                     rotate(cb, xv, sv);
                   }
                   exl3_barrier();
                 },
                 [&](int st, u4 (&v)[2]) {
                   const u4 *x = reinterpret_cast<const u4 *>(arow + 16 * kExl3Step * st);
                   v[0] = x[0];
                   v[1] = x[1];
                 },
                 acc);
    __syncthreads();  // the partials reuse the stage
  } else {
    const _Float16 *arow = xp + (am < B ? am : 0) * K + 16 * static_cast<int64_t>(kb0 + (lane >> 4));
    exl3_mma_run<true>(base, kstride, st1 - st0,
                 [] {},
                 [&](int st, u4 (&v)[2]) {
                   const u4 *x = reinterpret_cast<const u4 *>(arow + 16 * kExl3Step * st);
                   v[0] = x[0];
                   v[1] = x[1];
                 },
                 acc);
  }

  // 2. this split's partial: the 4 waves (same columns, different k) summed in a fixed order
  float *red = reinterpret_cast<float *>(smem);  // [4][BP][kExl3RedStride]
  const int wst = BP * kExl3RedStride;
  exl3_mma_store(acc, red + wave * wst, B);
  __syncthreads();
  const int64_t N = static_cast<int64_t>(NB) * 16;
  auto zp = [&](int split, int b, int c) {
    return reinterpret_cast<uint32_t *>(zpart) + (static_cast<int64_t>(split) * BP + b) * N + 128 * static_cast<int64_t>(g) + c;
  };
  for (int i = threadIdx.x; i < B * 128; i += blockDim.x) {
    const int b = i / 128, c = i % 128;
    const float *o = red + b * kExl3RedStride + c;
    const float z = ((o[0] + o[wst]) + o[2 * wst]) + o[3 * wst];
    if constexpr (FUSED) __hip_atomic_store(zp(s, b, c), __float_as_uint(z), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *zp(s, b, c) = __float_as_uint(z);
  }
  if constexpr (!FUSED) return;

  // 3. arrival; the last split of the block applies the output rotation
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's partials are performed
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t old = __hip_atomic_fetch_add(arrivals + g, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    is_last = old == static_cast<uint32_t>(S - 1);
    if (is_last) __hip_atomic_store(arrivals + g, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!is_last) return;
  const int b = wave;  // batch <= 2: one row per wave
  if (b >= B) return;
  // the splits' partials (this lane's two columns as one 8-byte word) in groups of 8 independent
  // loads, one round trip per group, added in split order
  float a0 = 0.f, a1 = 0.f;
  for (int s0 = 0; s0 < S; s0 += 8) {
    uint64_t v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (s0 + u < S)
        v[u] = __hip_atomic_load(reinterpret_cast<uint64_t *>(zp(s0 + u, b, 2 * lane)), __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (s0 + u < S) {
        a0 += __uint_as_float(static_cast<uint32_t>(v[u]));
        a1 += __uint_as_float(static_cast<uint32_t>(v[u] >> 32));
      }
  }
  fwht128_wave(a0, a1);
  const int64_t n0 = 128 * static_cast<int64_t>(g) + 2 * lane;
  const float y0 = a0 * kRScale * static_cast<float>(svh[n0]);
  const float y1 = a1 * kRScale * static_cast<float>(svh[n0 + 1]);
  if (ydt == VYBDQ_F32) { store_elem<VYBDQ_F32>(Y, nullptr, b * N + n0, y0); store_elem<VYBDQ_F32>(Y, nullptr, b * N + n0 + 1, y1); }
  else if (ydt == VYBDQ_F16) { store_elem<VYBDQ_F16>(Y, nullptr, b * N + n0, y0); store_elem<VYBDQ_F16>(Y, nullptr, b * N + n0 + 1, y1); }
  else { store_elem<VYBDQ_BF16>(Y, nullptr, b * N + n0, y0); store_elem<VYBDQ_BF16>(Y, nullptr, b * N + n0 + 1, y1); }
}

// 3. (batch > 2) y[b][n] = svh[n] * FWHT(sum_s zpart[s][b][.]) / sqrt(128)

template <int YDT>
__global__ void __launch_bounds__(64) k_exl3_out(const float *__restrict__ zpart, const _Float16 *__restrict__ svh,
                                                 void *__restrict__ Y, int BP, int S, int64_t N) {
  const int blk = blockIdx.x, b = blockIdx.y, lane = threadIdx.x;
  const int64_t n0 = 128 * static_cast<int64_t>(blk) + 2 * lane;
  // the splits' partials in groups of 8 independent 8-byte loads, added in split order
  float a0 = 0.f, a1 = 0.f;
  for (int s0 = 0; s0 < S; s0 += 8) {
    f2 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (s0 + u < S) v[u] = *reinterpret_cast<const f2 *>(zpart + (static_cast<int64_t>(s0 + u) * BP + b) * N + n0);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (s0 + u < S) {
        a0 += v[u][0];
        a1 += v[u][1];
      }
  }
  fwht128_wave(a0, a1);
  store_elem<YDT>(Y, nullptr, b * N + n0, a0 * kRScale * static_cast<float>(svh[n0]));
  store_elem<YDT>(Y, nullptr, b * N + n0 + 1, a1 * kRScale * static_cast<float>(svh[n0 + 1]));
}

// ---- host --------------------------------------------------------------------------------

static int exl3_bp(int64_t B) { return B <= 1 ? 1 : B <= 2 ? 2 : B <= 4 ? 4 : B <= 8 ? 8 : 16; }

// K-splits: whole 128 chunks (the x rotation is done per chunk), and from 256 k on a multiple of 256
// k, one 64-k step for each of the four waves. The product is bound by the decode on the VALU, so the
// time follows the k-blocks that the fullest CU decodes: ceil(workgroups / CUs) * kbs (at batch <= 2, 8 k-blocks cost as
// 16: two of the waves idle), plus a little per workgroup, per k-block of x rotated before the first step (batch <= 2) and per split of
// partials written and read back, which at batch <= 2 the last arrival reads alone (K = 2048, N = 5120, batch 1: 4 splits
// of 32 k-blocks 7.7 us, 8 of 16 8.2, 16 of 8 10.6; K = 4096, N = 1536: 8 splits 8.2, 16 9.4). Measured, batch 16: K = 5120, N = 17408: 5 splits (3 workgroups of
// 64 k-blocks a CU) 25.8 us per call, 4 (3 x 80) 27.5, 7 (4 x 48) 26.2, 10 (6 x 32) 27.3; K = 17408, N = 5120:
// 12 (2 x 96) 26.6, 17 (3 x 64) 28.1, 10 (2 x 112) 28.2, 14 (3 x 80) 29.6; K = 9216, N = 3072: 9 (1 x 64)
// 17.6, 12 (2 x 48) 20.0. Batch 1, K = 17408: 12 splits 22.6, 10 24.4, 7 27.3 us.
struct Exl3Split {
  int S;    // splits
  int kbs;  // 16-row k-blocks per split (a multiple of 8)
};
static Exl3Split exl3_splits(int64_t K, int64_t N, int BP) {
  const int KB = static_cast<int>(K / 16);
  const int64_t groups = N / 128;
  auto shape = [&](int S) {
    int kbs = (KB + S - 1) / S;
    kbs = kbs > 8 ? (kbs + 15) / 16 * 16 : 8;
    return Exl3Split{(KB + kbs - 1) / kbs, kbs};
  };
  const int64_t cus = device_cu_count();
  Exl3Split best = shape(1);
  int64_t best_cost = -1;
  for (int S = 1; S <= 16; ++S) {
    const Exl3Split c = shape(S);
    if (exl3_lds_bytes(BP, c.kbs) > kExl3MaxLds) continue;
    const int64_t rounds = (groups * c.S + cus - 1) / cus, steps = 8 * (c.kbs > 16 ? c.kbs : 16);
    const int64_t cost = exl3_fused(BP) ? rounds * (steps + 8) + 3 * BP * c.kbs + 32 * c.S : rounds * (8 * c.kbs + 48) + 8 * c.S;
    if (best_cost < 0 || cost < best_cost) best_cost = cost, best = c;
  }
  if (const char *e = tuning_env("VYBDQ_EXL3_SPLITS")) {  // tuning override
    const Exl3Split c = shape(atoi(e) > 0 ? atoi(e) : 1);
    if (exl3_lds_bytes(BP, c.kbs) <= kExl3MaxLds) best = c;
  }
  return best;
}

// The sizes the entry takes: x' rows of one of at most 16 k-splits (a grid of 2048 workgroups) within
// 160 KB, beside 40 KB of tiles above batch 2. (The kernel itself needs less.)
static bool exl3_size_ok(int64_t K, int64_t N, int BP) {
  const int64_t KB = K / 16, groups = N / 128;
  int64_t S = exl3_fused(BP) ? (KB + 23) / 24 : (2048 + groups - 1) / groups;
  if (exl3_fused(BP) && S > (groups < 2048 ? 2048 / groups : 1)) S = groups < 2048 ? 2048 / groups : 1;
  S = S > 16 ? 16 : S;
  S = S > KB / 4 ? KB / 4 : S;
  const int64_t kbs = ((KB + S - 1) / S + 7) / 8 * 8;
  return exl3_fused(BP) ? BP * 16 * kbs * 4 <= 160 * 1024 : BP * (16 * kbs + 8) * 2 + 40960 <= 160 * 1024;
}

// workspace: per-column-block arrival counters (zero between calls), x' (batch > 2), partials
static int64_t exl3_arrival_bytes(int64_t N) { return ((N / 128 * 4 + 255) / 256) * 256; }
static int64_t exl3_xp_bytes(int BP, int64_t K) { return exl3_fused(BP) ? 0 : ((BP * K * 2 + 255) / 256) * 256; }

static int64_t exl3_ws_bytes(int64_t B, int64_t K, int64_t N) {
  const int BP = exl3_bp(B);
  return exl3_arrival_bytes(N) + exl3_xp_bytes(BP, K) + static_cast<int64_t>(exl3_splits(K, N, BP).S) * BP * N * 4;
}

}  // namespace vybdq

using namespace vybdq;

static int exl3_check(uint64_t trellis, int64_t K, int64_t N, int codebook) {
  VYBDQ_REQUIRE(trellis, VYBDQ_ERR_ARG, "null trellis");
  VYBDQ_REQUIRE(codebook == VYBDQ_EXL3_MCG, VYBDQ_ERR_ARG,
                "unsupported codebook: only mcg (1) is implemented, as in the reference");
  VYBDQ_REQUIRE(K > 0 && N > 0 && K % 16 == 0 && N % 16 == 0, VYBDQ_ERR_SHAPE, "K and N must be positive multiples of 16");
  VYBDQ_REQUIRE((trellis & 15) == 0, VYBDQ_ERR_ALIGN, "trellis must be 16-byte aligned");
  VYBDQ_REQUIRE(N / 16 < (1 << 30) && K / 16 < (1 << 30), VYBDQ_ERR_SHAPE, "too many tiles");
  return VYBDQ_OK;
}

extern "C" int vybdq_exl3_decode_tiles(uint64_t trellis, uint64_t out, int64_t K, int64_t N, int codebook,
                                       int out_dt, uint64_t stream) {
  int rc = exl3_check(trellis, K, N, codebook);
  if (rc) return rc;
  VYBDQ_REQUIRE(out, VYBDQ_ERR_ARG, "null out");
  VYBDQ_REQUIRE(out_dt == VYBDQ_F32 || out_dt == VYBDQ_F16 || out_dt == VYBDQ_F64, VYBDQ_ERR_ARG,
                "out_dt must be F32, F16 or F64");
  const int NB = static_cast<int>(N / 16);
  const int64_t ntiles = (K / 16) * NB;
  const unsigned grid = static_cast<unsigned>((ntiles * 8 + 255) / 256);
  hipStream_t s = as_stream(stream);
  const auto *t = reinterpret_cast<const uint16_t *>(trellis);
  void *o = reinterpret_cast<void *>(out);
#define L(ODT) hipLaunchKernelGGL((k_exl3_decode<ODT>), dim3(grid), dim3(256), 0, s, t, o, ntiles, NB)
  if (out_dt == VYBDQ_F32) L(VYBDQ_F32); else if (out_dt == VYBDQ_F16) L(VYBDQ_F16); else L(VYBDQ_F64);
#undef L
  return check_launch("vybdq_exl3_decode_tiles");
}

extern "C" int vybdq_dequant_exl3(uint64_t trellis, uint64_t suh, uint64_t svh, uint64_t out, int64_t K, int64_t N,
                                  int codebook, int out_dt, uint64_t stream) {
  int rc = exl3_check(trellis, K, N, codebook);
  if (rc) return rc;
  VYBDQ_REQUIRE(suh && svh && out, VYBDQ_ERR_ARG, "null suh, svh or out");
  VYBDQ_REQUIRE(K % 128 == 0 && N % 128 == 0, VYBDQ_ERR_SHAPE, "K and N must be multiples of 128");
  VYBDQ_REQUIRE(out_dt == VYBDQ_F32 || out_dt == VYBDQ_F16 || out_dt == VYBDQ_F64, VYBDQ_ERR_ARG,
                "out_dt must be F32, F16 or F64");
  const int NB = static_cast<int>(N / 16);
  const dim3 grid(static_cast<unsigned>(N / 128), static_cast<unsigned>(K / 128));
  const size_t lds = 128 * 129 * 4;
  hipStream_t s = as_stream(stream);
  const auto *t = reinterpret_cast<const uint16_t *>(trellis);
  const auto *su = reinterpret_cast<const _Float16 *>(suh);
  const auto *sv = reinterpret_cast<const _Float16 *>(svh);
  void *o = reinterpret_cast<void *>(out);
#define L(ODT)                                                                                             \
  do {                                                                                                     \
    static std::atomic<uint64_t> raised{0};                                                                \
    const int rc = ensure_lds_limit(reinterpret_cast<const void *>(&k_exl3_dequant<ODT>),                  \
                                    static_cast<int>(lds), raised, "vybdq_dequant_exl3");                  \
    if (rc) return rc;                                                                                     \
    hipLaunchKernelGGL((k_exl3_dequant<ODT>), grid, dim3(256), lds, s, t, su, sv, o, NB);                 \
  } while (0)
  if (out_dt == VYBDQ_F32) L(VYBDQ_F32); else if (out_dt == VYBDQ_F16) L(VYBDQ_F16); else L(VYBDQ_F64);
#undef L
  return check_launch("vybdq_dequant_exl3");
}

// also what every smaller batch needs (its K splits may be more), so that one workspace serves them all
extern "C" int64_t vybdq_exl3_workspace_size(int64_t B, int64_t K, int64_t N) {
  if (B < 1 || B > 16 || K <= 0 || N <= 0 || K % 128 || N % 128) return -1;
  int64_t need = exl3_ws_bytes(B, K, N);
  for (int64_t b = 1; b < B; b *= 2) need = std::max(need, exl3_ws_bytes(b, K, N));
  return need;
}

template <bool FUSED>
static void exl3_gemm_launch(const uint16_t *t, const void *X, int xdt, const _Float16 *su, const _Float16 *sv,
                             void *Y, int ydt, int B, int BP, const _Float16 *xp, float *zp, uint32_t *arr, int64_t K,
                             int NB, const Exl3Split &sp, hipStream_t s) {
  const size_t lds = exl3_lds_bytes(BP, sp.kbs);  // at most kExl3MaxLds (exl3_splits; exl3_size_ok: some split fits)
  if (lds > 64 * 1024) {
    static std::atomic<uint64_t> raised{0};
    if (ensure_lds_limit(reinterpret_cast<const void *>(&k_exl3_gemm<FUSED>), kExl3MaxLds, raised, "exl3 gemm"))
      return;  // the launch below then fails and check_launch reports it
  }
  hipLaunchKernelGGL((k_exl3_gemm<FUSED>), dim3(static_cast<unsigned>(NB / 8), static_cast<unsigned>(sp.S)),
                     dim3(256), lds, s, t, X, xdt, su, sv, Y, ydt, B, BP, xp, zp, arr, K, NB, sp.kbs);
}

extern "C" int vybdq_exl3_gemm(uint64_t trellis, uint64_t suh, uint64_t svh, uint64_t X, uint64_t Y, int64_t B,
                               int64_t K, int64_t N, int codebook, int x_dt, int y_dt, uint64_t ws,
                               int64_t ws_bytes, uint64_t stream) {
  int rc = exl3_check(trellis, K, N, codebook);
  if (rc) return rc;
  VYBDQ_REQUIRE(suh && svh && X && Y, VYBDQ_ERR_ARG, "null suh, svh, X or Y");
  VYBDQ_REQUIRE(B >= 1 && B <= 16, VYBDQ_ERR_SHAPE, "B must be in [1, 16]");
  VYBDQ_REQUIRE(K % 128 == 0 && N % 128 == 0, VYBDQ_ERR_SHAPE, "K and N must be multiples of 128");
  VYBDQ_REQUIRE(dt_valid_in(x_dt), VYBDQ_ERR_ARG, "x_dt must be F32, F16 or BF16");
  VYBDQ_REQUIRE(dt_valid_in(y_dt), VYBDQ_ERR_ARG, "y_dt must be F32, F16 or BF16");
  VYBDQ_REQUIRE(ws && (ws & 255) == 0, VYBDQ_ERR_WORKSPACE, "workspace must be non-null and 256-byte aligned");
  VYBDQ_REQUIRE(ws_bytes >= exl3_ws_bytes(B, K, N), VYBDQ_ERR_WORKSPACE,
                "workspace smaller than vybdq_exl3_workspace_size");
  const int BP = exl3_bp(B);
  const Exl3Split sp = exl3_splits(K, N, BP);
  VYBDQ_REQUIRE(exl3_size_ok(K, N, BP), VYBDQ_ERR_SHAPE,
                "K too large for one split's x' stage in LDS at this batch");
  const int NB = static_cast<int>(N / 16);
  hipStream_t s = as_stream(stream);
  auto *arr = reinterpret_cast<uint32_t *>(ws);
  auto *xp = reinterpret_cast<_Float16 *>(ws + exl3_arrival_bytes(N));
  auto *zp = reinterpret_cast<float *>(ws + exl3_arrival_bytes(N) + exl3_xp_bytes(BP, K));
  const auto *su = reinterpret_cast<const _Float16 *>(suh);
  const auto *sv = reinterpret_cast<const _Float16 *>(svh);
  const auto *t = reinterpret_cast<const uint16_t *>(trellis);
  const void *x = reinterpret_cast<const void *>(X);
  void *y = reinterpret_cast<void *>(Y);
  const int b = static_cast<int>(B);
  if (!exl3_fused(BP)) {
    const dim3 gx(static_cast<unsigned>(K / 128), static_cast<unsigned>(B));
    VYBDQ_DISPATCH_IN(x_dt, XDT, hipLaunchKernelGGL((k_exl3_xprep<XDT>), gx, dim3(64), 0, s, x, su, xp, K));
  }
  if (exl3_fused(BP)) exl3_gemm_launch<true>(t, x, x_dt, su, sv, y, y_dt, b, BP, xp, zp, arr, K, NB, sp, s);
  else exl3_gemm_launch<false>(t, x, x_dt, su, sv, y, y_dt, b, BP, xp, zp, arr, K, NB, sp, s);
  if (!exl3_fused(BP)) {
    const dim3 go(static_cast<unsigned>(N / 128), static_cast<unsigned>(B));
    VYBDQ_DISPATCH_IN(y_dt, YDT, hipLaunchKernelGGL((k_exl3_out<YDT>), go, dim3(64), 0, s, zp, sv, y, BP, sp.S, N));
  }
  return check_launch("vybdq_exl3_gemm");
}
