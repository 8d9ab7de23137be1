// Prefill GEMM of many X rows: the packed matrix expanded to fp16 once, then a plain fp16 tile GEMM, gfx950.
//
// Y[m, n] = RS[m, n] + sum_k X[m, k] * W[n, k]
//
// The fused tile bodies (mmq.h, kqgemm.hip) decode every weight once per 128 X rows, on the VALU between the
// matrix-core instructions: at 1999 rows 16 times, and the kernel is bound by that (650 to 740 TFLOP/s,
// Q6_K and IQ2_S 480 to 540). From a few hundred rows it is cheaper to decode each weight once into the
// caller's workspace (k_wide_expand: bound by memory, packed bytes in, 2 bytes per weight out) and to
// multiply fp16 by fp16 (k_wide_mm). Every weight is the decode's F16 value: exact in float32, one rounding.
//
// k_wide_mm: tiles of BM (128, 192 or 256) x 256, K step 64, eight waves (2 x 4) of BM/2 x 64 on
// v_mfma_f32_32x32x16_f16, both operands staged by direct-to-LDS loads of whole 128-byte lines, two
// stages, one barrier per step. A row's eight 16-byte chunks are stored at chunk ^ (row & 7), so the eight
// lanes of a read phase fall on distinct banks. Bound by LDS and the matrix cores together (per step and CU 2048
// matrix-core cycles against 1536 of operand reads and 512 of stage writes at BM = 256) and by the clock
// under that load. Alone, fp16 X, float32 Y: 1999 x 17408 x 5120 397 us (898 TFLOP/s, BM = 192; 431 at
// 256, 526 at 128), 1999 x 5120 x 17408 383 us (930, BM = 256), 512 x 17408 x 5120 106 us (862). Issuing the next
// stage's loads between the k16 steps instead of at once: 421 / 395 us and 433 / 397 us (256 / 192); raised wave
// priority around the matrix-core instructions: 2 to 5% slower.
#include "gemv_dev.h"

#include <cstdlib>

namespace vybdq {

typedef float f16v __attribute__((ext_vector_type(16)));

// ---- expand -------------------------------------------------------------------------------------

// 8 consecutive weights: chunk e of 8 weights of the block (q4_0, Q8_0: 32 weights) or super-block (256) at sb
template <int FMT>
__device__ __forceinline__ u4 expand8(const uint8_t *sb, int e) {
  auto ld8 = [](const uint8_t *p, uint32_t (&v)[2]) { __builtin_memcpy(v, p, 8); };
  auto ldh = [](const uint8_t *p) {
    uint16_t h;
    __builtin_memcpy(&h, p, 2);
    return half_bits_to_f32(h);
  };
  auto pack = [](const float (&w)[8]) {
    u4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = __builtin_bit_cast(uint32_t, h2{static_cast<_Float16>(w[2 * i]), static_cast<_Float16>(w[2 * i + 1])});
    return o;
  };
  auto byte = [](const uint32_t (&v)[2], int i) { return (v[i >> 2] >> (8 * (i & 3))) & 0xffu; };
  float w[8];
  uint32_t v[2];
  if constexpr (FMT == FMT_Q4_0) {
    const float d = ldh(sb);
    ld8(sb + 2 + 8 * (e & 1), v);
#pragma unroll
    for (int i = 0; i < 2; ++i) v[i] = (v[i] >> (4 * (e >> 1))) & 0x0F0F0F0Fu;
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = d * static_cast<float>(static_cast<int>(byte(v, i)) - 8);
  } else if constexpr (FMT == FMT_Q8_0) {
    const float d = ldh(sb);
    ld8(sb + 2 + 8 * e, v);
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = d * static_cast<float>(static_cast<int8_t>(byte(v, i)));
  } else if constexpr (FMT == FMT_Q4_K || FMT == FMT_Q5_K) {
    constexpr int QS = FMT == FMT_Q4_K ? 16 : 48;
    const int j = e >> 2, l = 8 * (e & 3);  // sub-block, first weight in it
    const u4a4 h = *reinterpret_cast<const u4a4 *>(sb);
    float sc, mn;
    scale_min_k4(h[1], h[2], h[3], j, sc, mn);
    const float ds = half_bits_to_f32(h[0] & 0xffffu) * sc, dm = half_bits_to_f32(h[0] >> 16) * mn;
    ld8(sb + QS + 32 * (j >> 1) + l, v);
#pragma unroll
    for (int i = 0; i < 2; ++i) v[i] = (v[i] >> (4 * (j & 1))) & 0x0F0F0F0Fu;
    if constexpr (FMT == FMT_Q5_K) {
      uint32_t b[2];
      ld8(sb + 16 + l, b);
#pragma unroll
      for (int i = 0; i < 2; ++i) v[i] |= ((b[i] >> j) & 0x01010101u) << 4;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = fmaf(ds, static_cast<float>(byte(v, i)), -dm);
  } else if constexpr (FMT == FMT_Q6_K) {
    const int hf = e >> 4, q = (e >> 2) & 3, l = 8 * (e & 3);  // half, 32-weight run of it, first weight
    uint32_t b[2];
    ld8(sb + 64 * hf + 32 * (q & 1) + l, v);
    ld8(sb + 128 + 32 * hf + l, b);
    const float ds = ldh(sb + 208) * static_cast<float>(static_cast<int8_t>(sb[192 + 8 * hf + 2 * q + (l >> 4)]));
#pragma unroll
    for (int i = 0; i < 2; ++i) v[i] = ((v[i] >> (4 * (q >> 1))) & 0x0F0F0F0Fu) | (((b[i] >> (2 * q)) & 0x03030303u) << 4);
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = ds * static_cast<float>(static_cast<int>(byte(v, i)) - 32);
  } else {
    const int ib = e >> 2, l = e & 3;  // sub-block, group of 8 in it
    const unsigned long long grid = kIq2sGrid[sb[2 + e] | (((sb[66 + ib] >> (2 * l)) & 3) << 8)];
    v[0] = static_cast<uint32_t>(grid);
    v[1] = static_cast<uint32_t>(grid >> 32);
    const uint32_t sgn = sb[34 + e], nib = (sb[74 + ib] >> (4 * (l >> 1))) & 15u;
    const float dl = ldh(sb) * (0.5f + static_cast<float>(nib)) * 0.25f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float x = dl * static_cast<float>(byte(v, i));
      w[i] = (sgn >> i) & 1u ? -x : x;
    }
  }
  return pack(w);
}

template <int FMT>
__global__ void __launch_bounds__(256) k_wide_expand(const uint8_t *__restrict__ W, u4 *__restrict__ out, int64_t n8) {
  constexpr int CPB = is_kquant<FMT>() ? 32 : 4;  // 8-weight chunks per block
  constexpr int BB = FMT == FMT_Q4_0 ? 18 : FMT == FMT_Q8_0 ? 34 : FMT == FMT_Q4_K ? 144 : FMT == FMT_Q5_K ? 176 : FMT == FMT_Q6_K ? 210 : 82;
  constexpr int U = 4;  // chunks per thread, their loads independent
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * (256 * U) + threadIdx.x;
  u4 o[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t i = i0 + 256 * u < n8 ? i0 + 256 * u : n8 - 1;
    o[u] = expand8<FMT>(W + (i / CPB) * BB, static_cast<int>(i % CPB));
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (i0 + 256 * u < n8) out[i0 + 256 * u] = o[u];
}

// ---- fp16 x fp16 --------------------------------------------------------------------------------

struct WideArgs {
  const _Float16 *A, *B;  // X [M][K], W [N][K]
  const float *xscale;    // per X row (null: 1)
  int M, N, K;
  int m_tiles, units;
  void *Y;
  int ydt;
  int64_t ldy;
  const void *RS;
};

template <int MF>
__global__ void __launch_bounds__(512, 2) k_wide_mm(const WideArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int BM = 64 * MF, PER = (BM + 256) / 64, STAGE = (BM + 256) * 128;
  int u = blockIdx.x;
  if (a.units % 8 == 0) u = (u & 7) * (a.units >> 3) + (u >> 3);  // workgroups are dealt to the 8 XCDs in turn
  const int m0 = u % a.m_tiles * BM, n0 = u / a.m_tiles * 256;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int wm = wave >> 2, wn = wave & 3;
  const uint32_t rb = static_cast<uint32_t>(a.K) * 2;
  const char *Ab = reinterpret_cast<const char *>(a.A) + static_cast<int64_t>(m0) * rb;
  const char *Bb = reinterpret_cast<const char *>(a.B) + static_cast<int64_t>(n0) * rb;
  // load j = wave + 8 i of a stage: rows 8 j .. + 8 of the tile's X rows, then its W rows (rows past the ends
  // re-read the last one: they reach only outputs that are not stored)
  uint32_t off[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int r = 8 * (wave + 8 * i) + (lane >> 3), c = (lane & 7) ^ (lane >> 3);
    const int row = r < BM ? min(r, a.M - 1 - m0) : min(r - BM, a.N - 1 - n0);
    off[i] = static_cast<uint32_t>(row) * rb + 16 * c;
  }
  auto issue = [&](int k, char *buf) {
#pragma unroll
    for (int i = 0; i < PER; ++i) lds_dma16_s((8 * (wave + 8 * i) < BM ? Ab : Bb) + 128 * static_cast<int64_t>(k), off[i], buf + 1024 * (wave + 8 * i));
  };
  f16v acc[MF][2];
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[m][n][r] = 0.f;
  // operand of k16 step s: row lane & 31, chunk 2 s + (lane >> 5)
  const int lo = (lane & 31) * 128 + (((lane >> 5) ^ (lane & 7)) * 16);
  const int ao = wm * (BM / 2) * 128, bo = (BM + wn * 64) * 128;
  const int nk = a.K / 64;
  issue(0, smem);
  for (int i = 0; i < nk; ++i) {
    const char *buf = smem + (i & 1) * STAGE;
    __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));  // vmcnt(0): this wave's loads of stage i
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    if (i + 1 < nk) issue(i + 1, smem + ((i + 1) & 1) * STAGE);  // every wave has left stage i - 1
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const char *p = buf + (lo ^ (32 * s));
      h8 av[MF], bv[2];
#pragma unroll
      for (int m = 0; m < MF; ++m) av[m] = *reinterpret_cast<const h8 *>(p + ao + 4096 * m);
#pragma unroll
      for (int n = 0; n < 2; ++n) bv[n] = *reinterpret_cast<const h8 *>(p + bo + 4096 * n);
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int m = 0; m < MF; ++m) acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[m], bv[n], acc[m][n], 0, 0, 0);
    }
  }
  // acc[m][n][r] = C[m0 + wm BM / 2 + 32 m + 8 (r / 4) + 4 (lane >> 5) + r % 4][n0 + 64 wn + 32 n + (lane & 31)]
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = m0 + wm * (BM / 2) + 32 * m + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
      if (row >= a.M) continue;
      const float sc = a.xscale ? a.xscale[row] : 1.0f;
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const int col = n0 + wn * 64 + 32 * n + (lane & 31);
        if (col >= a.N) continue;
        const int64_t i = static_cast<int64_t>(row) * a.ldy + col;
        const float v = acc[m][n][r] * sc;
        switch (a.ydt) {
          case VYBDQ_F32: store_elem<VYBDQ_F32>(a.Y, a.RS, i, v); break;
          case VYBDQ_F16: store_elem<VYBDQ_F16>(a.Y, a.RS, i, v); break;
          case VYBDQ_BF16: store_elem<VYBDQ_BF16>(a.Y, a.RS, i, v); break;
          default: store_elem<VYBDQ_F64>(a.Y, a.RS, i, v); break;
        }
      }
    }
}

// ---- host -----------------------------------------------------------------------------------------

static int64_t wide_align256(int64_t b) { return (b + 255) / 256 * 256; }

double mmq_plan_us(int wtype, int64_t M, int64_t N, int64_t K);
double kq2_plan_us(int64_t M, int64_t N, int64_t K);

// Row fragments of 64 per tile (2, 3 or 4), or 0 where the fused bodies are the better choice: this path's estimate has
// to be 7% below the fused body's. This path: expand, rounds of 256 tiles by the measured time of a K step (idle and full
// chip; more once the expanded matrix leaves the 256 MB cache), the conversion of X. The fused body: its own planner's
// estimate, scaled, plus the conversion of X and the outputs. Fitted over 14 row counts from 256 to 4096 x 11 shapes, standard
// deviation 3 to 8% on either side (a flat rate per type misses by up to 35%: fused, Q8_0 4096 x 5120 x 17408 runs at
// 900 TFLOP/s, 2000 x 17408 x 5120 at 655); of 924 measured calls none that is taken is the slower one, and the choice is within 0.7%
// of the best one in the mean (up to 15% left: q4_0 3500 x 12288 x 4096, 25600 x 5120 Q5_K at 1400 rows). Measured, fused / here: 17408 x 5120 at 2000 rows q4_0 490 / 489 us (not taken), Q8_0 545 / 474,
// Q4_K 531 / 472, Q6_K 634 / 476; 5120 x 17408 Q8_0 413 / 474 (not taken), Q6_K 639 / 492; 25600 x 5120 Q8_0 662 / 734 (not taken),
// at 600 rows Q6_K 307 / 338 (not taken). Calls under 50 us stay fused. At most 2^29 weights (1 GiB of workspace).
static int wide_plan(int wtype, int64_t M, int64_t N, int64_t K) {
  if (M < 128 || M >= (1 << 24) || K % 256 || K >= (1 << 22) || N % 64 || N * K > (int64_t(1) << 29) || M * K >= (int64_t(1) << 31))
    return 0;
  double bpw, f[4];  // bytes per weight; fused: planner's us, constant, us per 10^6 elements of X and of Y
  switch (wtype) {
    case 2: bpw = 0.5625, f[0] = 0.511, f[1] = 11.2, f[2] = 0.69, f[3] = 2.86; break;
    case 8: bpw = 1.0625, f[0] = 0.620, f[1] = 13.8, f[2] = 0.58, f[3] = 2.45; break;
    case 12: bpw = 0.5625, f[0] = 0.566, f[1] = 12.9, f[2] = 1.02, f[3] = 2.90; break;
    case 13: bpw = 0.6875, f[0] = 0.661, f[1] = 14.1, f[2] = 0.96, f[3] = 2.76; break;
    case 14: bpw = 0.8203, f[0] = 0.826, f[1] = 18.4, f[2] = 0.73, f[3] = 0.49; break;
    case 22: bpw = 0.3203, f[0] = 0.797, f[1] = 16.9, f[2] = 0.43, f[3] = 0.91; break;
    default: return 0;
  }
  const double nk = 1e-6 * static_cast<double>(N) * static_cast<double>(K), mk = 1e-6 * static_cast<double>(M) * static_cast<double>(K);
  struct Cost {  // us per MB expanded; per K step and round; per K step and full chip, out of cache; per round; constant; per 10^6 of X
    double exp, step, full, cold, round, fixed, x;
  };
  constexpr Cost cost[3] = {{0.148, 0.738, 0.325, 0.283, 10.8, 14.5, 0.06}, {0.123, 1.032, 0.342, 0.206, 18.6, 13.9, 0.17},
                            {0.151, 1.238, 0.317, 0.168, 31.9, 7.1, 0.38}};
  const int64_t cus = device_cu_count();
  int best = 0;
  double best_t = -1;
  for (int mf = 2; mf <= 4; ++mf) {
    const Cost &c = cost[mf - 2];
    const int64_t units = (M + 64 * mf - 1) / (64 * mf) * ((N + 255) / 256);
    const double rounds = static_cast<double>((units + cus - 1) / cus), full = static_cast<double>(units) / static_cast<double>(cus);
    const double t = nk * (2 + bpw) * c.exp + static_cast<double>(K / 64) * (rounds * c.step + full * (c.full + (nk > 120 ? c.cold : 0))) +
                     rounds * c.round + c.fixed + c.x * mk;
    if (best_t < 0 || t < best_t) best_t = t, best = mf;
  }
  if (const char *e = tuning_env("VYBDQ_WIDE")) {  // 0: never, 2..4: that tile height
    const int h = atoi(e);
    return h >= 2 && h <= 4 ? h : 0;
  }
  const double fused = f[0] * (wtype >= 14 ? kq2_plan_us(M, N, K) : mmq_plan_us(wtype, M, N, K)) + f[1] + f[2] * mk +
                       f[3] * 1e-6 * static_cast<double>(M) * static_cast<double>(N);
  return fused > 50 && best_t < (fused > 500 ? 0.98 : 0.93) * fused ? best : 0;
}

// workspace: [fp16 weights][fp16 copy of X][X row scales]
static int64_t wide_bytes(int64_t M, int64_t N, int64_t K) {
  return wide_align256(N * K * 2) + wide_align256(M * K * 2) + wide_align256(M * 4);
}

int64_t wide_mm_workspace_size(int wtype, int64_t M, int64_t N, int64_t K) {
  return wide_plan(wtype, M, N, K) ? wide_bytes(M, N, K) : 0;
}

int x_rows_to_f16(const void *X, int xdt, int64_t M, int64_t K, void *xh, float *xscale, hipStream_t s);

template <int FMT>
static void wide_expand(const uint8_t *W, u4 *out, int64_t n8, hipStream_t s) {
  hipLaunchKernelGGL((k_wide_expand<FMT>), dim3(static_cast<unsigned>((n8 + 1023) / 1024)), dim3(256), 0, s, W, out, n8);
}

template <int MF>
static int wide_launch(WideArgs &a, hipStream_t s) {
  constexpr int BM = 64 * MF, LDS = 2 * (BM + 256) * 128;
  static std::atomic<uint64_t> raised{0};
  const int rc = ensure_lds_limit(reinterpret_cast<const void *>(&k_wide_mm<MF>), LDS, raised, "gemm (many rows)");
  if (rc) return rc;
  a.m_tiles = (a.M + BM - 1) / BM;
  a.units = a.m_tiles * ((a.N + 255) / 256);
  hipLaunchKernelGGL((k_wide_mm<MF>), dim3(static_cast<unsigned>(a.units)), dim3(512), LDS, s, a);
  return check_launch("gemm (many rows)");
}

// Returns 1 when the call does not take this path (rule, or no workspace of wide_mm_workspace_size bytes).
int wide_mm_gemm(int wtype, const void *W, const void *X, int xdt, void *Y, int ydt, int64_t M, int64_t N, int64_t K,
                 int64_t ldy, const void *RS, void *ws, int64_t ws_bytes, hipStream_t s) {
  if (!ws || ws_bytes < wide_bytes(M, N, K)) return 1;
  const int mf = wide_plan(wtype, M, N, K);
  if (!mf) return 1;
  char *base = static_cast<char *>(ws);
  char *xh = base + wide_align256(N * K * 2);
  float *sc = reinterpret_cast<float *>(xh + wide_align256(M * K * 2));
  WideArgs a{};
  a.A = static_cast<const _Float16 *>(X);
  if (xdt != VYBDQ_F16) {
    const int rc = x_rows_to_f16(X, xdt, M, K, xh, sc, s);
    if (rc) return rc;
    a.A = reinterpret_cast<const _Float16 *>(xh);
    a.xscale = sc;
  }
  const uint8_t *w = static_cast<const uint8_t *>(W);
  u4 *wh = reinterpret_cast<u4 *>(base);
  const int64_t n8 = N * K / 8;
  switch (wtype) {
    case 2: wide_expand<FMT_Q4_0>(w, wh, n8, s); break;
    case 8: wide_expand<FMT_Q8_0>(w, wh, n8, s); break;
    case 12: wide_expand<FMT_Q4_K>(w, wh, n8, s); break;
    case 13: wide_expand<FMT_Q5_K>(w, wh, n8, s); break;
    case 14: wide_expand<FMT_Q6_K>(w, wh, n8, s); break;
    default: wide_expand<FMT_IQ2_S>(w, wh, n8, s); break;
  }
  const int rc = check_launch("gemm (many rows) expand");
  if (rc) return rc;
  a.B = reinterpret_cast<const _Float16 *>(base);
  a.M = static_cast<int>(M);
  a.N = static_cast<int>(N);
  a.K = static_cast<int>(K);
  a.Y = Y;
  a.ydt = ydt;
  a.ldy = ldy;
  a.RS = RS;
  return mf == 2 ? wide_launch<2>(a, s) : mf == 3 ? wide_launch<3>(a, s) : wide_launch<4>(a, s);
}

}  // namespace vybdq
