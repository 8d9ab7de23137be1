// Host side of the GEMM at a few X rows (rows_mm.h): plan, dispatch and the split reduce.
#include "rows_mm.h"

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>

namespace vybdq {

constexpr int kRowsMaxSplits = 40;  // K splits: above, the partials outweigh the weights

// the float32 partials of a K split summed in split order and stored with the residual
template <int ODT>
__global__ void __launch_bounds__(256) k_rows_reduce(const RowsArgs a) {
  const int64_t n4 = a.N / 4, total = a.M * n4, stride = static_cast<int64_t>(a.M) * a.N;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= total) return;
  const int64_t row = i / n4, c = 4 * (i % n4);
  const float *p = a.part + row * a.N + c;
  f4 v = f4{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < a.splits; s0 += 8) {  // eight loads in flight, added in split order
    f4 t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = *reinterpret_cast<const f4 *>(p + (s0 + u < a.splits ? s0 + u : 0) * stride);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (s0 + u < a.splits) v = v + t[u];
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) store_elem<ODT>(a.Y, a.RS, row * a.ldy + c + u, v[u]);
}

struct RowsPlan {
  // waves (16 weight rows each), K splits, super-blocks per split, workgroups per split and row group, stages, X row
  // fragments per workgroup, row groups
  int NW, splits, sps, nwg, ns, MF, groups;
};

// One workgroup fits a CU; the plan minimises the stages of the busiest CU (a stage's bytes at the 18.5 GB/s a CU gets of HBM)
// plus a workgroup's start (X staging) and the split partials, written and read back. Up to 32 X rows it has 16 waves (256
// weight rows a tile) or 8: with 8 (two per SIMD) a wave's decode waits on its own LDS reads and matrix-core chains, 8%; with 16
// a K range that leaves LDS two stages has one barely in flight, 10% (but not Q6_K, whose decode hides it). Forced, 8 / 16 waves,
// 17408 x 5120 at 8 rows: q4_0 20.7 / 20.4 us, Q8_0 24.9 / 27.0, Q4_K 21.3 / 20.0, Q5_K 23.5 / 22.3, Q6_K 29.3 / 25.7, IQ2_S 27.7 / 25.2;
// at 24 rows 24.5 / 23.7, 29.7 / 37.3, 25.9 / 25.0, 28.0 / 27.5, 32.7 / 32.6, 34.7 / 31.8; 4096 x 4096 at 24 rows Q4_K 12.7 / 13.6, Q6_K
// 13.7 / 14.6; 34816 x 5120 Q4_K 42.4 / 38.6. Over 660 such calls the choice is 0.4% off the better one in the mean, 10% at the
// worst (8 waves for Q4_K there). Above 32 rows the accumulators need the registers of 8 waves.
// Up to 2^22 weights the chip is idle and a workgroup's own chain counts, which grows with its X rows (LDS reads of the
// operands, staging): every 16 rows get workgroups of their own (W again from L2), of 8 waves (twice the workgroups of 16), and a
// stage costs its latency.
// 64 rows, X all in one workgroup / in groups of 16: 512 x 512 q4_0 9.4 / 5.5 us, Q4_K 11.8 / 6.4, IQ2_S 10.8 / 7.3; 1024 x
// 1024 8.2 / 6.7, 10.1 / 7.7, 9.2 / 7.9; 2048 x 2048 10.6 / 9.3, 12.4 / 10.2, 10.9 / 10.6; 2560 x 2560 12.8 / 12.0, 14.5 / 12.6 but IQ2_S
// 14.1 / 14.2 (its decode is repeated per group). (The unscaled tiles of the calls without a workspace: 512 x 512 5.3, 7.9, 8.7;
// Q8_0, whose decode is short, 5.2 against 5.9 here.) Only plans whose partials
// fit ws_bytes are looked at. VYBDQ_ROWS_PLAN="sps,nwg[,groups]" overrides
// the split (and whether rows are grouped: 1 or more); ignored where it does not fit.
template <int FMT>
static RowsPlan rows_plan(int M, int64_t N, int64_t K, int64_t ws_bytes) {
  using F = RowsFmt<FMT>;
  const int SB = static_cast<int>(K / 256), MT = (M + 15) / 16, cus = device_cu_count(), tab = FMT == FMT_IQ2_S ? kRowsGrid : 0;
  RowsPlan best{};
  double best_t = -1;
  int fs = 0, fn = 0, fg = 0;
  if (const char *e = tuning_env("VYBDQ_ROWS_PLAN"))
    if (sscanf(e, "%d,%d,%d", &fs, &fn, &fg) < 2 || fs < 1 || fn < 1) fs = fn = fg = 0;
  if (fs > SB) fs = SB;
  for (;; fs = fg = 0) {
    const bool small = fg ? fg > 1 : MT > 1 && N * K <= (1 << 22);
    const int groups = small ? MT : 1, MF = MT / groups, xsb = MF * (F::OPS * 1024 + 64);
    for (int NW = MF <= 2 && !small ? 16 : 8; NW >= 4; NW /= 2) {
      const int BN = 16 * NW, tiles = static_cast<int>(N / BN), stage = BN * F::C * 16;
      if (N % BN || (NW == 4 && N % 128 == 0)) continue;  // 4 waves only where 8 do not divide N
      for (int sps = fs ? fs : 1; sps <= SB && sps <= (fs ? fs : 32); ++sps) {
        const int splits = (SB + sps - 1) / sps;
        int ns = (160 * 1024 - tab - sps * xsb) / stage;
        if (ns < 2) break;
        ns = ns > 4 ? 4 : ns;
        if (splits > kRowsMaxSplits || (splits > 1 && splits * M * N * 4 > ws_bytes)) continue;
        int nwg = cus / (splits * groups) > 0 ? cus / (splits * groups) : 1;
        if (fs) nwg = fn;
        nwg = nwg < tiles ? nwg : tiles;
        const int wgs = splits * groups * nwg, rounds = (wgs + cus - 1) / cus, stages = (tiles + nwg - 1) / nwg * sps;
        const double part = splits * M * static_cast<double>(N) / 1.0e6;
        double t;
        if (small) {
          t = rounds * stages * (FMT == FMT_Q6_K || FMT == FMT_IQ2_S ? 1.85 : 1.2) + static_cast<double>(wgs) / cus;
          if (splits > 1) t += 2.0 + 1.5 * part;
        } else {
          t = rounds * (stages * stage / 18.5e3 * (ns == 2 && FMT != FMT_Q6_K ? 1.1 : 1.0) + 2.5 + 0.2 * sps * MF);
          if (NW < 16 && MF <= 2) t *= 1.08;
          if (splits > 1) t += 4.0 + 2.0 * part;
        }
        if (best_t < 0 || t < best_t) {
          best_t = t;
          best = {NW, splits, sps, nwg, ns, MF, groups};
        }
      }
    }
    if (!fs || best.splits) return best;  // splits = 0: no plan fits (an override that does not fit: plan without it)
  }
}

bool rows_mm_supported(int wtype, int64_t M, int64_t N, int64_t K) {
  return M >= 1 && M <= 64 && K % 256 == 0 && K < (int64_t(1) << 22) && N % 64 == 0 &&
         (wtype == 2 || wtype == 8 || wtype == 12 || wtype == 13 || wtype == 14 || wtype == 22);
}

// the plan of a type id
static RowsPlan rows_plan_ty(int wtype, int M, int64_t N, int64_t K, int64_t ws_bytes) {
  switch (wtype) {
    case 2: return rows_plan<FMT_Q4_0>(M, N, K, ws_bytes);
    case 8: return rows_plan<FMT_Q8_0>(M, N, K, ws_bytes);
    case 12: return rows_plan<FMT_Q4_K>(M, N, K, ws_bytes);
    case 13: return rows_plan<FMT_Q5_K>(M, N, K, ws_bytes);
    case 14: return rows_plan<FMT_Q6_K>(M, N, K, ws_bytes);
    default: return rows_plan<FMT_IQ2_S>(M, N, K, ws_bytes);
  }
}

// Workspace: the split partials of M rows and of every smaller count, so that one workspace serves a batch that shrinks
// (at least 256 bytes where the shape is taken, so that a caller has one). Within 16 row counts a plan's estimate is
// a constant plus a term in splits times rows, so its splits only fall as rows are added: those of the first count bound
// the rest.
int64_t rows_mm_workspace_size(int wtype, int64_t M, int64_t N, int64_t K) {
  if (!rows_mm_supported(wtype, M, N, K)) return 0;
  int64_t need = 0;
  for (int64_t m = 1; m <= M; m += 16) {
    const int64_t splits = rows_plan_ty(wtype, static_cast<int>(m), N, K, INT64_MAX).splits, last = m + 15 < M ? m + 15 : M;
    if (splits > 0) need = std::max(need, splits > 1 ? splits * last * N * 4 : 256);
  }
  return need;
}

template <int FMT, int XDT, int MF, int NW, bool GR = false>
static int rows_launch(const RowsArgs &a, const RowsPlan &p, hipStream_t s) {
  using Sh = RowsShape<FMT, MF, NW>;
  static std::atomic<uint64_t> raised{0};
  const int rc = ensure_lds_limit(reinterpret_cast<const void *>(&k_rows_mm<FMT, XDT, MF, NW, GR>), 160 * 1024, raised,
                                  "gemm (few rows)");
  if (rc) return rc;
  const size_t lds = Sh::TAB + static_cast<size_t>(p.sps) * Sh::XSB + static_cast<size_t>(p.ns) * Sh::STAGE;
  hipLaunchKernelGGL((k_rows_mm<FMT, XDT, MF, NW, GR>), dim3(static_cast<unsigned>(p.nwg), static_cast<unsigned>(p.splits),
                     static_cast<unsigned>(p.groups)), dim3(64 * NW), lds, s, a);
  return check_launch("gemm (few rows)");
}

template <int FMT, int XDT, int MF>
static int rows_launch_p(const RowsArgs &a, const RowsPlan &p, hipStream_t s) {
  if constexpr (MF == 1) {
    if (p.groups > 1) return p.NW == 8 ? rows_launch<FMT, XDT, 1, 8, true>(a, p, s) : rows_launch<FMT, XDT, 1, 4, true>(a, p, s);
  }
  if constexpr (MF <= 2) {
    if (p.NW == 16) return rows_launch<FMT, XDT, MF, 16>(a, p, s);
  }
  if (p.NW == 8) return rows_launch<FMT, XDT, MF, 8>(a, p, s);
  return rows_launch<FMT, XDT, MF, 4>(a, p, s);
}

template <int FMT, int XDT>
static int rows_launch_x(const RowsArgs &a, const RowsPlan &p, hipStream_t s) {
  switch (p.MF) {
    case 1: return rows_launch_p<FMT, XDT, 1>(a, p, s);
    case 2: return rows_launch_p<FMT, XDT, 2>(a, p, s);
    case 3: return rows_launch_p<FMT, XDT, 3>(a, p, s);
    default: return rows_launch_p<FMT, XDT, 4>(a, p, s);
  }
}

template <int FMT>
static int rows_run_fmt(RowsArgs &a, int xdt, void *ws, int64_t ws_bytes, hipStream_t s) {
  const int64_t K = static_cast<int64_t>(a.SB) * 256;
  const RowsPlan p = rows_plan<FMT>(a.M, a.N, K, ws_bytes);
  if (p.splits == 0) return 1;
  a.rowbytes = unit_row_bytes<FMT>(K / 64);
  a.splits = p.splits;
  a.sps = p.sps;
  a.ns = p.ns;
  a.tiles = a.N / (16 * p.NW);
  a.part = static_cast<float *>(ws);
  int rc = VYBDQ_OK;
  VYBDQ_DISPATCH_IN(xdt, XDT, rc = rows_launch_x<FMT, XDT>(a, p, s));
  return rc;
}

// Returns 1 when the call does not fit (shape, W not 16-byte aligned).
int rows_mm_gemm(int wtype, const void *W, const void *X, int xdt, void *Y, int ydt, int64_t M, int64_t N, int64_t K,
                 int64_t ldy, const void *RS, void *ws, int64_t ws_bytes, hipStream_t s) {
  if (!rows_mm_supported(wtype, M, N, K) || (reinterpret_cast<uintptr_t>(W) & 15)) return 1;
  RowsArgs a{};
  a.W = static_cast<const uint8_t *>(W);
  a.X = X;
  a.M = static_cast<int>(M);
  a.N = static_cast<int>(N);
  a.SB = static_cast<int>(K / 256);
  a.Y = Y;
  a.ydt = ydt;
  a.ldy = ldy;
  a.RS = RS;
  int rc;
  switch (wtype) {
    case 2: rc = rows_run_fmt<FMT_Q4_0>(a, xdt, ws, ws_bytes, s); break;
    case 8: rc = rows_run_fmt<FMT_Q8_0>(a, xdt, ws, ws_bytes, s); break;
    case 12: rc = rows_run_fmt<FMT_Q4_K>(a, xdt, ws, ws_bytes, s); break;
    case 13: rc = rows_run_fmt<FMT_Q5_K>(a, xdt, ws, ws_bytes, s); break;
    case 14: rc = rows_run_fmt<FMT_Q6_K>(a, xdt, ws, ws_bytes, s); break;
    default: rc = rows_run_fmt<FMT_IQ2_S>(a, xdt, ws, ws_bytes, s); break;
  }
  if (rc || a.splits == 1) return rc;
  const unsigned grid = static_cast<unsigned>((M * N / 4 + 255) / 256);
  VYBDQ_DISPATCH_OUT(ydt, ODT, hipLaunchKernelGGL((k_rows_reduce<ODT>), dim3(grid), dim3(256), 0, s, a));
  return check_launch("gemm (few rows) split reduce");
}

}  // namespace vybdq
