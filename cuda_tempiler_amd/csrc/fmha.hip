// fmha.hip -- translation unit of the causal FMHA forward (kernel: the plugin skeleton
// tempo/plugins/gfx950/skeletons/fmha_fwd/kernel.hip, compiled here in its own namespace).
#include "fmha_api.h"

#include <limits.h>
#include <stdint.h>

#include <algorithm>

namespace tempo_fmha {
#include "common/cdna4.h"
#include "fmha_fwd/kernel.hip"
#include "fmha_fwd/rows.hip"

bool applicable(const TempoFmhaParams& p) {
  if (!p.Q || !p.K || !p.V || !p.O) return false;
  if (p.B <= 0 || p.H <= 0 || p.Hkv <= 0 || p.Sq <= 0 || p.Sk <= 0) return false;
  if (p.H % p.Hkv != 0) return false;
  if (p.D != 128 && p.D != 256) return false;
  // d contiguous with 16-byte aligned rows (strides in elements)
  const long s[] = {p.q_ss, p.q_sh, p.q_sb, p.k_ss, p.k_sh, p.k_sb,
                    p.v_ss, p.v_sh, p.v_sb, p.o_ss, p.o_sh, p.o_sb};
  for (long x : s)
    if (x % 8 != 0) return false;
  const uintptr_t ptrs[] = {(uintptr_t)p.Q, (uintptr_t)p.K, (uintptr_t)p.V, (uintptr_t)p.O};
  for (uintptr_t x : ptrs)
    if (x % 16 != 0) return false;
  if ((long)p.Sq * p.q_ss > (1L << 40)) return false;
  if ((long)((p.Sq + 127) / 128) * p.H * p.B >= (1L << 31)) return false;
  if ((long)p.Sq * (p.H / p.Hkv) >= (1L << 31) - 256) return false;  // packed rows (O > 500 GB)
  // key/value rows of one block are addressed with 32-bit byte offsets from the block's first row
  if (p.k_ss > (1L << 24) || p.v_ss > (1L << 24)) return false;
  return true;
}

// How a call runs: on k_fmha_rows (all packed rows of a (batch, KV head) fit one 32-row tile) or
// on k_fmha_fwd with `kg` key groups per workgroup; its key blocks in ranges of `chunk` (one
// workgroup each; INT_MAX: not cut), merged by k_fmha_combine over `splits` ranges.  `hg`: head groups
// of k_fmha_fwd, Hkv (packed) or H; `apart`: H is the better one where keys are not cut.
struct Plan {
  bool rows;
  int kg, chunk, splits, hg;
  bool apart;
};

static int tile_rows(const Plan& pl) { return pl.rows ? 32 : fmha::BQ; }

// workspace: [splits][rows] fp32 O of D, then [splits][rows] pairs (reference, sum)
static size_t ws_bytes(const TempoFmhaParams& p, const Plan& pl) {
  if (pl.splits <= 1) return 0;
  return (size_t)pl.splits * p.B * p.H * p.Sq * (p.D + 2) * sizeof(float);
}

// The plan of a call.  The rates below are microseconds on MI355X, measured over grids of 8 to
// 2048 workgroups and 128 to 32768 keys; they only order the alternatives.
//   * Rows: a workgroup passes 4 blocks (128 keys) in 1.0 (D = 128) or 2.1 (D = 256), and a cut
//     costs the second kernel (3) and its pass over the ranges (0.25 each).  256 workgroups
//     stream at the HBM's rate, so a cut never asks for a second round: at 8 sequences x 8 KV
//     heads x 4096 keys, D = 128, 4 ranges take 27.1, 1 range 49.1, 8 ranges 28.4.  At D = 256 more
//     than 16 rows over at most 4 blocks (one a wave) stay on tiles: 8 rows of 4 heads over 96
//     keys 9.3 here, 8.3 there.
//   * Tiles, D = 128: workgroups of two key groups where the grid leaves CUs with at most two
//     workgroups and the longest tile has 16 key blocks or more -- 120 against 134 at 256 tiles of
//     203 blocks, 84 against 98 at 512 causal tiles of up to 128 -- else one group, two
//     workgroups per CU (291 against 330 at 2048 tiles of 64 blocks, 12 against 18 at 512 of 3).
//   * Tiles, cut: while ranges x tiles fit one round of the CUs and the blocks saved (0.47 each,
//     1.07 at D = 256) pay for the partial results: written, read and merged at 4.5 TB/s plus
//     3.5 (5 at D = 256) for the second kernel (512 rows over 8192 keys, 16 heads, D = 256: 96
//     against 265; 2 x 158 rows over 235 keys, 2 heads, D = 256: 18.5 cut, 16.9 whole).
//   * Tiles of one head each where a round of the CUs holds them, they have few key blocks and no
//     cut pays.  Either form is its longest tile -- 0.65 (D = 128) or 1.3 a block, and its rows' Q and
//     O, which pass the tile's CU at 40 GB/s -- and the key blocks all its tiles bring in, 0.034 or
//     0.068 a MB: 4 x 38 rows x 104 keys, 8 heads, 2 KV heads, D = 256: 14.3 packed, 10.6 apart;
//     32 x 107 x 107, 8 heads, 1 KV head: 14.9 packed, 18.5 apart.  Of 6694 random calls of both
//     forms 73 take over 3 % more than packed and 24 than apart (693 and none by the longest tile
//     alone, counted as whole).
static Plan plan(const TempoFmhaParams& p) {
  constexpr int kCus = 256;
  const int G = p.H / p.Hkv;
  const long R = (long)p.Sq * G, bh = (long)p.B * p.Hkv;
  const int L = p.causal ? fmha::fmha_tile_blocks<true>(0, (int)R, (int)R, G, p.Sq, p.Sk)
                         : fmha::fmha_tile_blocks<false>(0, (int)R, (int)R, G, p.Sq, p.Sk);
  Plan pl = {R <= 32 && (p.D == 128 || R <= 16 || L > 4), 1, INT_MAX, 1, p.Hkv, false};
  const long tiles = bh * (pl.rows ? 1 : (R + fmha::BQ - 1) / fmha::BQ);
  if (!pl.rows && p.D == 128 && tiles <= 2 * kCus && L >= 16) pl.kg = 2;
  const double blk = p.D == 128 ? 0.47 : 1.07;
  const int nq = (p.Sq + fmha::BQ - 1) / fmha::BQ;
  double gain = 0;  // of tiles of one head over packed ones, where they are the better
  if (!pl.rows && pl.kg == 1 && G > 1 && L <= 16 && (long)p.B * p.H * nq <= kCus) {
    auto form = [&](int rows, int g, long groups) {  // `groups` times the tiles of `rows` rows
      double longest = 0;
      long blocks = 0;
      for (int r0 = 0; r0 < rows; r0 += fmha::BQ) {
        const int n = rows - r0 < fmha::BQ ? rows - r0 : fmha::BQ;
        const int l = p.causal ? fmha::fmha_tile_blocks<true>(r0, n, rows, g, p.Sq, p.Sk)
                               : fmha::fmha_tile_blocks<false>(r0, n, rows, g, p.Sq, p.Sk);
        longest = std::max(longest, l * (p.D == 128 ? 0.65 : 1.3) + n * p.D * 1.56e-4);
        blocks += l;
      }
      return longest + (p.D == 128 ? 0.034 : 0.068) * groups * blocks * 128 * p.D * 1e-6;
    };
    gain = form((int)R, G, bh) - form(p.Sq, 1, (long)p.B * p.H);
    pl.apart = gain > 0;
  }
  if (2 * tiles > kCus) {
    if (pl.apart) pl.hg = p.H;
    return pl;
  }
  const double rows = (double)bh * R;
  auto cost = [&](int n) {
    const int c = (L + n - 1) / n;
    if (pl.rows)
      return (c + 3) / 4 * (p.D == 128 ? 1.0 : 2.1) + (n > 1 ? 3 + 0.25 * n : 0);
    return c * blk + (n > 1 ? (p.D == 128 ? 3.5 : 5.0) + n * rows * p.D * 8 / 4.5e6 : 0);
  };
  int best = 1;
  for (int n = 2; n <= 64 && n * tiles <= kCus && 4 * n <= L; ++n)
    if (cost(n) < cost(best)) best = n;
  if (pl.apart && (best == 1 || gain - 1 >= cost(1) - cost(best))) {  // (1: the estimates' error)
    pl.hg = p.H;
    return pl;
  }
  if (best > 1) {
    pl.chunk = (L + best - 1) / best;
    pl.splits = (L + pl.chunk - 1) / pl.chunk;
  }
  return pl;
}

// The same call without a workspace.
static Plan whole(const TempoFmhaParams& p) {
  Plan pl = plan(p);
  if (pl.splits > 1 && pl.apart) pl.hg = p.H;
  pl.chunk = INT_MAX;
  pl.splits = 1;
  return pl;
}

template <int D, bool CAUSAL>
static hipError_t run(const TempoFmhaParams& p, const Plan& pl, float* ws, hipStream_t s) {
  const int hg = pl.rows ? p.Hkv : pl.hg, R = p.Sq * (p.H / hg), BQ = tile_rows(pl);
  // one workgroup per (key range, tile of rows, head group, batch); heaviest causal tile first
  const dim3 grid((unsigned)((R + BQ - 1) / BQ) * hg * p.B * pl.splits), blk(pl.rows ? 256 : 256 * pl.kg);
  const float scale_log2 = p.scale * 1.4426950408889634f;
  float* const ml = ws ? ws + (size_t)pl.splits * p.B * p.H * p.Sq * D : nullptr;
  auto go = [&](auto kernel, auto... last) {
    hipLaunchKernelGGL(kernel, grid, blk, 0, s, static_cast<const _Float16*>(p.Q),
                       static_cast<const _Float16*>(p.K), static_cast<const _Float16*>(p.V),
                       static_cast<_Float16*>(p.O), p.LSE, p.B, p.H, p.Hkv, p.Sq, p.Sk, scale_log2,
                       p.q_sb, p.q_ss, p.q_sh, p.k_sb, p.k_ss, p.k_sh, p.v_sb, p.v_ss, p.v_sh,
                       p.o_sb, p.o_ss, p.o_sh, pl.chunk, ws, ml, last...);
  };
  if (pl.rows)
    go(fmha::k_fmha_rows<D, CAUSAL>);
  else if (D == 128 && pl.kg == 2)
    go(fmha::k_fmha_fwd<D, CAUSAL, D == 128 ? 2 : 1>, hg, p.H / hg, hg / p.Hkv);
  else
    go(fmha::k_fmha_fwd<D, CAUSAL, 1>, hg, p.H / hg, hg / p.Hkv);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || pl.splits <= 1) return e;
  const long rows = (long)p.B * p.H * p.Sq;
  hipLaunchKernelGGL((fmha::k_fmha_combine<D, CAUSAL>), dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s,
                     ws, ml, static_cast<_Float16*>(p.O), p.LSE, p.B, p.H, p.Hkv, p.Sq, p.Sk, BQ,
                     pl.chunk, p.o_sb, p.o_ss, p.o_sh);
  return hipGetLastError();
}

static hipError_t dispatch(const TempoFmhaParams& p, const Plan& pl, float* ws, hipStream_t s) {
  if (p.D == 256)
    return p.causal ? run<256, true>(p, pl, ws, s) : run<256, false>(p, pl, ws, s);
  return p.causal ? run<128, true>(p, pl, ws, s) : run<128, false>(p, pl, ws, s);
}

size_t workspace_bytes(const TempoFmhaParams& p) {
  return applicable(p) ? ws_bytes(p, plan(p)) : 0;
}

hipError_t launch(const TempoFmhaParams& p, void* ws, size_t bytes, hipStream_t s) {
  if (!applicable(p)) return hipErrorInvalidConfiguration;
  Plan pl = plan(p);
  if (ws_bytes(p, pl) > (ws ? bytes : 0) || reinterpret_cast<uintptr_t>(ws) % 16 != 0) pl = whole(p);
  return dispatch(p, pl, static_cast<float*>(ws), s);
}
}  // namespace tempo_fmha
