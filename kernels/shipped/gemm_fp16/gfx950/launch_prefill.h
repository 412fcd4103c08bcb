// launch_prefill.h -- the launchers of the interleaved prefill kernel (k_gemm_ilv): template
// definitions, instantiated by launch_prefill.hip for the ladder's rows (prefill.inc) -- or by
// any other translation unit built with the same scheduler flag (the plugin's tuning
// harness instantiates its candidates from this header).
#pragma once
#include "launch.h"

namespace tempo {
namespace gen {

template <int BM, int BN, int BK, int WM, int WN, int STAGES, int GROUP, int XCD, int RSP,
          int SW, int MINKT>
hipError_t launch_ilv(const GemmParams& p, hipStream_t s, const Workspace& w) {
  const int nm = (p.M + BM - 1) / BM;
  const int nn = p.N / BN;
  const int splits = split_count(nm * nn, p.K / BK, SW, MINKT);
  const size_t bytes = splits > 1 ? (size_t)splits * p.M * p.N * sizeof(float) : 0;
  if (w.need) {
    *w.need = bytes;
    return hipSuccess;
  }
  const dim3 blk(WM * WN * 64);
  if (splits == 1) {
    hipLaunchKernelGGL((k_gemm_ilv<BM, BN, BK, WM, WN, STAGES, GROUP, XCD, RSP, 0>),
                       dim3(nm * nn), blk, 0, s, p.A, p.B, p.C, p.M, p.N, p.K, p.lda, p.ldb,
                       p.ldc, static_cast<float*>(nullptr), 1, p.N);
    return hipGetLastError();
  }
  if constexpr (SW > 0) {
    hipError_t werr = hipSuccess;
    const Lease ws = workspace_for(w, bytes, s, &werr);
    if (!ws.ptr) return werr;
    hipLaunchKernelGGL((k_gemm_ilv<BM, BN, BK, WM, WN, STAGES, GROUP, XCD, RSP, 1>),
                       dim3(nm * nn * splits), blk, 0, s, p.A, p.B, p.C, p.M, p.N, p.K, p.lda, p.ldb,
                       p.ldc, ws.ptr, splits, p.N);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_reduce(ws.ptr, splits, p.M, p.N, p.C, p.ldc, s);
  }
  return hipErrorInvalidConfiguration;  // not reached: splits == 1 where SW == 0
}

// Fused gate/up (EPI = 1): p.N is the output width and B holds 2N rows (gate, then up); each
// tile covers BN/2 output columns.  No split-K, no workspace.  `up`: the row of the first up row
// relative to B (p.N for a launch over all output columns).
template <int BM, int BN, int BK, int WM, int WN, int STAGES, int GROUP, int XCD, int RSP>
hipError_t launch_ilv_gu_part(const GemmParams& p, hipStream_t s, int up) {
  const int nm = (p.M + BM - 1) / BM;
  const int nn = p.N / (BN / 2);
  hipLaunchKernelGGL((k_gemm_ilv<BM, BN, BK, WM, WN, STAGES, GROUP, XCD, RSP, 0, 1>),
                     dim3(nm * nn), dim3(WM * WN * 64), 0, s, p.A, p.B, p.C, p.M, p.N, p.K, p.lda,
                     p.ldb, p.ldc, static_cast<float*>(nullptr), 1, up);
  return hipGetLastError();
}

// The fused gate/up row with the output columns in two parts: where the last round of tiles
// (BN/2 output columns each) is at most a quarter full, the whole rounds run on the leading
// columns and the remaining columns on TBM x TBN/2-column tiles -- four or more times as many --
// as a launch of their own; both parts read their up rows p.N rows past their gate rows.
template <int BM, int BN, int BK, int WM, int WN, int STAGES, int GROUP, int XCD, int RSP,
          int TBM, int TBN, int TBK, int TWM, int TWN, int TSTAGES>
hipError_t launch_ilv_gu_tail(const GemmParams& p, hipStream_t s, const Workspace& w) {
  static_assert(BN % TBN == 0 && (BM * BN) / (TBM * TBN) >= 4, "tail tiles of a quarter or less");
  if (w.need) {
    *w.need = 0;
    return hipSuccess;
  }
  constexpr int CUS = 256, BNO = BN / 2;
  const int nm = (p.M + BM - 1) / BM, nn = p.N / BNO;
  const int tiles = nm * nn, whole = tiles / CUS * CUS;
  if (whole == 0 || whole % nm || whole / nm == nn || 4 * (tiles - whole) > CUS)
    return launch_ilv_gu_part<BM, BN, BK, WM, WN, STAGES, GROUP, XCD, RSP>(p, s, p.N);
  const int n0 = whole / nm * BNO;
  GemmParams a = p, b = p;
  a.N = n0;
  b.N = p.N - n0;
  b.B = p.B + (long)n0 * p.ldb;
  b.C = p.C + n0;
  const hipError_t e = launch_ilv_gu_part<BM, BN, BK, WM, WN, STAGES, GROUP, XCD, RSP>(a, s, p.N);
  if (e != hipSuccess) return e;
  return launch_ilv_gu_part<TBM, TBN, TBK, TWM, TWN, TSTAGES, GROUP, XCD, RSP>(b, s, p.N);
}

// ---- PLAN rows --------------------------------------------------------------------------------
// One tile of plan.inc: unsplit (gate_up: with the fused epilogue), or its partial sums into ws.
template <int BM, int BN, int BK, int WM, int WN, int STAGES, int GROUP, int XCD, int RSP, int SPL>
hipError_t run_plan_tile(const GemmParams& p, hipStream_t s, float* ws, int splits, bool gate_up) {
  if (splits == 1 && gate_up)
    return launch_ilv_gu_part<BM, BN, BK, WM, WN, STAGES, GROUP, XCD, RSP>(p, s, p.N);
  if (splits == 1) return launch_ilv<BM, BN, BK, WM, WN, STAGES, GROUP, XCD, RSP, 0, 0>(p, s, Workspace{});
  if constexpr (SPL) {
    const int cols = gate_up ? 2 * p.N : p.N;  // the plain product over the gate and the up rows
    hipLaunchKernelGGL((k_gemm_ilv<BM, BN, BK, WM, WN, STAGES, GROUP, XCD, RSP, 1>),
                       dim3((unsigned)((p.M + BM - 1) / BM) * (cols / BN) * splits),
                       dim3(WM * WN * 64), 0, s, p.A, p.B, p.C, p.M, cols, p.K, p.lda, p.ldb, p.ldc,
                       ws, splits, cols);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return gate_up ? launch_reduce_gu(ws, splits, p.M, p.N, p.C, p.ldc, s)
                   : launch_reduce(ws, splits, p.M, p.N, p.C, p.ldc, s);
  }
  return hipErrorInvalidConfiguration;  // not reached: the plan splits only tiles that can be
}

template <int GROUP, int XCD, int RSP>
hipError_t run_plan(const GemmParams& p, hipStream_t s, float* ws, const TilePlan& pl, bool gate_up) {
  switch (pl.tile) {
#define TEMPO_TILE(i, bm, bn, bk, wm, wn, st, split) \
  case i:                                           \
    return run_plan_tile<bm, bn, bk, wm, wn, st, GROUP, XCD, RSP, split>(p, s, ws, pl.splits, gate_up);
#include "plan.inc"
#undef TEMPO_TILE
  }
  return hipErrorInvalidConfiguration;
}

// plan_tiles over `cols` weight rows, but for 192 x 256 tiles (5) whose tile rows make whole raster
// groups of 8 and a ragged one: those run at 0.82 to 1.05 PFLOP/s, whatever their round's fill, where
// 256 x 256 tiles (2) in whole groups reach 1.1.  So from K = 3584 on the 256-row tiles take what the
// 192-row ones would need longer for at 1 PFLOP/s, and what leaves their own last round of whole
// groups at most 48 tiles (us, 256 rows against 192: (2048, 11008, 11008) 478, 539; (2048, 11264,
// 13824) 582, 660; (2048, 9216, 12288) 491, 516; (2048, 17408, 11008) 724, 871; (2048, 9472, 14080)
// 570, 644; (2048, 9728, 4352) 177, 187; where they stay:
// (2048, 10240, 3584) 162, 141; in whole groups: (3000, 11008, 11008) 819, 628).
// Fused gate/up (cols = 2N): at M <= 128 a split has to be 10 % ahead of the best unsplit tile, whose
// short last round costs less than a whole one ((74, 17408, 3840) 66 us unsplit, 71 in three splits);
// and where the gate and the up panel lie an odd number of 128 rows of a multiple of 8 KiB apart, the
// 192-row tiles give way to 256 rows ((700, 14464, 4096) 189 against 230).
inline TilePlan ilv_plan(const GemmParams& p, int cols, bool split) {
  TilePlan pl = plan_tiles(kPlanTiles, kPlanTables, 0, p.M, cols, p.K, split);
  if (cols != p.N && p.M <= 128 && pl.splits > 1) {
    const TilePlan flat = plan_tiles(kPlanTiles, kPlanTables, 0, p.M, cols, p.K, false);
    if (flat.tile >= 0 && pl.us > 0.9 * flat.us) pl = flat;
  }
  if (cols != p.N && pl.tile == 5 && pl.splits == 1 && p.N % 256 && p.ldb % 4096 == 0) pl.tile = 2;
  const int nm5 = (p.M + 191) / 192, nm = (p.M + 255) / 256;
  if (pl.tile != 5 || pl.splits != 1 || p.K < 3584 || p.K % 64 || nm5 < 8 || nm5 % 8 == 0) return pl;
  double rate = 0;
  for (const TileRate& r : plan_table(kPlanTables, p.M).rate)
    if (r.tile == 2) rate = r.us[0];
  const double us = tile_us(plan_table(kPlanTables, p.M), rate, 256, 256, 64, p.M, cols, p.K, 1);
  const int rest = (int)((long)nm * (cols / 256) % 256);
  if (2e-9 * p.M * cols * p.K > us || (nm % 8 == 0 && rest > 0 && rest <= 48)) {
    pl.tile = 2;
    pl.us = us;
  }
  return pl;
}

template <int GROUP, int XCD, int RSP>
hipError_t launch_ilv_planned(const GemmParams& p, hipStream_t s, const Workspace& w, bool gate_up) {
  const int cols = gate_up ? 2 * p.N : p.N;
  TilePlan pl = ilv_plan(p, cols, true);
  const size_t bytes = pl.splits > 1 ? (size_t)pl.splits * p.M * cols * sizeof(float) : 0;
  if (w.need) {
    *w.need = bytes;
    return hipSuccess;
  }
  Lease ws;
  if (bytes) {
    hipError_t err = hipSuccess;
    ws = workspace_to_gain(w, bytes, 0, s, &err);
    if (!ws.ptr) pl = ilv_plan(p, cols, false);  // unsplit
  }
  return run_plan<GROUP, XCD, RSP>(p, s, ws.ptr, pl, gate_up);
}

template <int GROUP, int XCD, int RSP>
hipError_t launch_ilv_plan(const GemmParams& p, hipStream_t s, const Workspace& w) {
  return launch_ilv_planned<GROUP, XCD, RSP>(p, s, w, false);
}

template <int GROUP, int XCD, int RSP>
bool plan_instead(const GemmParams& p, hipStream_t s, const Workspace& w, const OwnRow& own,
                  hipError_t* e) {
  constexpr int kLd = 0x7fffffff / (2 * 256);
  if (p.lda > kLd || p.ldb > kLd) return false;
  const TilePlan pl = plan_tiles(kPlanTiles, kPlanTables, 0, p.M, p.N, p.K, true);
  if (pl.tile < 0) return false;
  const TileDims& d = kPlanTiles[pl.tile];
  const double wgs = (double)((p.M + d.bm - 1) / d.bm) * (p.N / d.bn) * pl.splits;
  const double us = std::max(pl.us + own.wg * wgs, own.weights * 1e-6 * p.N * p.K);
  if (us >= (pl.splits > 1 ? own.ahead_split : own.ahead) * own.us) return false;
  const size_t bytes = pl.splits > 1 ? (size_t)pl.splits * p.M * p.N * sizeof(float) : 0;
  *e = hipSuccess;
  if (w.need) {
    *w.need = bytes;
    return true;
  }
  Lease ws;
  if (bytes) {
    ws = workspace_to_gain(w, bytes, own.bytes, s, e);
    if (!ws.ptr) return false;
  }
  *e = run_plan<GROUP, XCD, RSP>(p, s, ws.ptr, pl, false);
  return true;
}

template <int BM, int BN, int BK, int WM, int WN, int STAGES, int GROUP, int XCD, int RSP,
          int SW, int MINKT, int RATE100>
hipError_t launch_ilv_or_plan(const GemmParams& p, hipStream_t s, const Workspace& w) {
  const int splits = split_count((p.M + BM - 1) / BM * (p.N / BN), p.K / BK, SW, MINKT);
  hipError_t e = hipSuccess;
  const OwnRow own = {tile_us(plan_table(kPlanTables, p.M), RATE100 * 0.01, BM, BN, BK, p.M, p.N, p.K,
                              splits),
                      splits > 1 ? (size_t)splits * p.M * p.N * sizeof(float) : 0, 0.95, 0.95};
  if (plan_instead<GROUP, XCD, RSP>(p, s, w, own, &e)) return e;
  return launch_ilv<BM, BN, BK, WM, WN, STAGES, GROUP, XCD, RSP, SW, MINKT>(p, s, w);
}

// Fused gate/up: the plan over the 2N rows of B, or the output columns in two parts
// (launch_ilv_gu_tail, one more launch: 3) where that is estimated ahead.
template <int GROUP, int XCD, int RSP>
hipError_t launch_ilv_plan_gu(const GemmParams& p, hipStream_t s, const Workspace& w) {
  const int nm = (p.M + 255) / 256, tiles = nm * (p.N / 128), whole = tiles / 256 * 256;
  if (p.M > 128 && p.N % 128 == 0 && whole > 0 && whole % nm == 0 && whole < tiles &&
      4 * (tiles - whole) <= 256) {
    const TilePlan pl = ilv_plan(p, 2 * p.N, true);
    double r256 = 0, r128 = 0;
    for (const TileRate& r : plan_table(kPlanTables, 1 << 30).rate) {
      if (r.tile == 2) r256 = r.us[0];
      if (r.tile == 0 && r128 == 0) r128 = r.us[0];
    }
    const double us = (whole / 256 * r256 + r128) * p.K * 1e-3 + 3;
    if (us < pl.us)
      return launch_ilv_gu_tail<256, 256, 64, 2, 2, 2, GROUP, XCD, RSP, 128, 128, 64, 2, 2, 3>(p, s, w);
  }
  return launch_ilv_planned<GROUP, XCD, RSP>(p, s, w, true);
}

}  // namespace gen
}  // namespace tempo
