// mk_plan.h — which kernel runs a call, on which tiles, in how many parts: the
// host's choices, from sizes alone (no HIP headers, so that they can be checked
// without a GPU).
#pragma once
#include <stdint.h>

#include <algorithm>

#include "mk_map.h"

namespace mk {

// ---------------------------------------------------------------------------
// The small-tile kernel (mk_gemm_small.hip)
// ---------------------------------------------------------------------------

struct GemmSmallPlan {
  int tile, bm, bn;  // index into kTiles, and its shape
  int grid, split;   // workgroups, and parts of each tile along K
  double us;         // estimated time
};
// What a K-split may use: workspace words and bytes for its partial tiles.
struct SmallSpace {
  int64_t words, tile_bytes;
};
// The fold of a reduce epilogue: `rows` rows with `peers` partials each
// (peers < 0: no such epilogue).
struct SmallFold {
  int peers;
  int64_t rows;
};

// The tile shapes and what they cost, in us.  A launch of g tiles runs in
// rounds of per_cu x CUs workgroups (what fits the LDS of a CU together), each
//   round + stages x slope(x),   x = the round's workgroups per CU,
// slope = one + load x while no CU holds two, else two + more (x - 1): a full
// chip clocks lower and shares its caches.  `start` comes once, `meet` when
// the parts of a tile have to meet.  Fitted to N(0, 1/K) operands at 40 shapes
// of 128 .. 10240 rows, 256 .. 8192 columns and 256 .. 8192 K on one MI355X.
// The two-stage rings (128 x 128 at 64 KB, 64 x 64 at 32 KB) hide one tile's
// first loads and its store behind its neighbours on the CU, which is worth
// more than a deeper ring when many short tiles follow each other:
// 10240x6656x512 takes 82 us with them, 107 with one 128 KB ring per CU.
struct TileCost {
  int bm, bn, per_cu;
  bool fold_only;
  double start, round, one, load, two, more, meet;
};
constexpr TileCost kTiles[] = {
    {64, 64, 3, false, 1.8, 1.2, 0.235, 0.0, 0.33, 0.125, 7.0},
    {128, 64, 2, false, 0.7, 1.6, 0.380, 0.0, 0.60, 0.02, 7.0},
    {128, 128, 1, false, 3.0, 1.0, 0.410, 0.14, 0.0, 0.0, 10.0},
    {192, 128, 1, false, 3.0, 2.0, 0.470, 0.33, 0.0, 0.0, 10.0},
    {128, 256, 1, false, 2.5, 2.3, 0.620, 0.28, 0.0, 0.0, 14.0},
    {128, 128, 2, false, 3.0, 2.0, 0.530, 0.05, 0.717, 0.245, 10.0},
    {64, 64, 5, true, 0.8, 2.2, 0.300, 0.0, 0.31, 0.155, 7.0},
};
// fold_only, the 32 KB ring of the last: its many workgroups hide a fold's loads
// (whole ReduceScatters, against the 128 x 128 tiles at 64 KB: 4096x4096x256 of
// world 16 40.4 us / 44.2, 2048x2304x32 of world 8 16.0 / 17.6, 4096x2048x128 of
// world 16 23.4 / 27.6; the 64 x 64 tiles at 48 KB are level with it), but a plain
// product of tall tiles thrashes L2 with them (5504x768x896 18.5 us, 14.5 with
// the 128 x 128 tiles at 64 KB).

inline double rounds_cost(const TileCost& c, int64_t g, double stages, int cus) {
  const int64_t full = (int64_t)c.per_cu * cus;
  auto round = [&](int64_t n) {
    const double x = (double)n / cus;
    return c.round + stages * (n > cus ? c.two + c.more * (x - 1) : c.one + c.load * x);
  };
  return c.start + (double)(g / full) * round(full) + (g % full ? round(g % full) : 0.0);
}

// Estimated us of folding `tiles` tiles, `at_once` workgroups at a time: the
// chip takes 7 TB/s of partials beside its products, one workgroup 60 GB/s.
inline double fold_cost(const SmallFold& f, double tiles, double tile_elems, double at_once) {
  if (f.peers <= 0) return 0.0;
  const double chip = tiles * tile_elems * 2 * f.peers / 7e6, one = tile_elems * 2 * f.peers / 0.06e6;
  const double own = one * (double)(int64_t)((tiles + at_once - 1) / at_once);
  return chip > own ? chip : own;
}

// The tile and split with the least estimated time; false: no tile fits.
inline bool plan_gemm_small(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int cus, const SmallSpace& ws,
                            const SmallFold& fold, GemmSmallPlan* plan) {
  // offsets from 2^31 up read as zeros, so both buffer windows end below it
  if (K * ldb * 2 >= (1LL << 31)) return false;
  const int64_t nk = (K + 63) / 64;
  const bool reduce = fold.peers >= 0;
  bool found = false;
  for (int i = 0; i < (int)(sizeof kTiles / sizeof kTiles[0]); ++i) {
    const TileCost& c = kTiles[i];
    if (c.fold_only && !reduce) continue;
    if (M % c.bm || N % c.bn || (reduce && 256 % c.bm) || (int64_t)c.bm * lda * 2 >= (1LL << 31)) continue;
    const int64_t nt = (M / c.bm) * (N / c.bn);
    if (nt * nk >= (1LL << 31)) continue;
    for (int s = 1; s <= 4; ++s) {
      const int64_t g = nt * s;
      if (s > 1 && (reduce || g > cus || nk < 4 * s || nt + g > ws.words || g * c.bm * c.bn * 4 > ws.tile_bytes))
        break;
      double t = rounds_cost(c, g, (double)((nk + s - 1) / s), cus) + (s > 1 ? c.meet : 0.0);
      if (reduce) t += fold_cost(fold, (double)fold.rows / c.bm * (N / c.bn), (double)c.bm * c.bn, c.per_cu * cus);
      if (!found || t < plan->us) {
        found = true;
        *plan = {i, c.bm, c.bn, (int)g, s, t};
      }
    }
  }
  return found;
}

// ---------------------------------------------------------------------------
// The persistent kernel (mk_gemm.hip)
// ---------------------------------------------------------------------------

inline double persistent_round(double tiles, double stages, int cus) {
  return 3.8 + stages * (0.24 + 0.55 * tiles / cus);
}

// Parts along K (1..4) for `rest` 256 x 256 tiles of a last round on `cus`
// workgroups, and its estimated us: splitting fills the idle CUs, which then
// clock lower, and costs the parts' exchange, about 13 us for two of them.
// Measured, whole against split tail: 10240x2048x1024 (64 tiles) 54 against
// 80 us, 16384x6656x416 (128) 122 against 137, 16384x3584x3584 (128) equal,
// 9216x2048x3584 (32) 153 against 146, 16384x3584x8192 (128) 745 against 735.
// With the reduce epilogue the exchange costs 35 to 90 us (its registers spill
// beside the fold: 16384x3584x3584, 128 tiles, 406 whole and 480 split with the
// partials staged in the launch; 10240x2048x1024, 64 tiles, 84 and 127), so
// only a K of about 14000 and more is split there: 10240x2048, world 8, K 14336
// 680 whole, 539 split; K 28672 1339 and 971; 9216x2048 (32), world 4, K 14336
// 658 and 514; 16384x3584 (128), world 8, K 28672 2792 and 2581.
inline int tail_split(int64_t rest, int64_t K, int cus, bool reduce, double* us) {
  const double stages = (double)K / 32;
  int best = 1;
  double t = persistent_round((double)rest, stages, cus);
  for (int s = 2; s <= 4 && rest * s <= cus && K / 32 >= 4 * s; ++s) {
    const double ts = persistent_round((double)(rest * s), stages / s, cus) + (reduce ? 80.0 : 10.0 + 1.5 * s);
    if (ts < t) {
      t = ts;
      best = s;
    }
  }
  if (us) *us = t;
  return best;
}

// Estimated us of the persistent kernel on `tiles` 256 x 256 tiles (split:
// with a workspace for the K-split of its tail).  Fitted like the tile table:
// 4096^3 106-118 measured, 8192x8192x512 71, 8192x3584x8192 382.
inline double persistent_cost(int64_t tiles, int64_t K, int cus, bool split) {
  const double stages = (double)K / 32;
  double t = 5.0 + (double)(tiles / cus) * persistent_round(cus, stages, cus);
  const int64_t rest = tiles % cus;
  if (rest && split && tiles > cus) {
    double tail;
    tail_split(rest, K, cus, false, &tail);
    t += tail;
  } else if (rest) {
    t += persistent_round((double)rest, stages, cus);
  }
  return t;
}

// Parts along K of each of the R < n_cons tiles in the persistent kernel's last
// round, bm rows each: as many as fit, up to 4 and with at least 4 K stages,
// for the expert GEMMs, which stream weights; as tail_split finds best for
// dense 256-row tiles.
inline int tail_parts(int R, int64_t K, int bm, int n_cons, bool reduce) {
  if (R == 0) return 1;
  if (bm == 256) return tail_split(R, K, n_cons, reduce, nullptr);
  return (int)std::min<int64_t>(std::min(4, n_cons / R), (K / 32) / 4);
}

// The tail of `tiles` tiles may be split: the workspace is there and holds the
// partial tiles.
inline bool tail_fits(int64_t tiles, int64_t K, int bm, int cus, const SmallSpace& ws) {
  const int rest = (int)(tiles % cus);
  return ws.words > 0 && (int64_t)rest * (tail_parts(rest, K, bm, cus, false) - 1) * bm * 256 * 4 <= ws.tile_bytes;
}

// ---------------------------------------------------------------------------
// Which of the two
// ---------------------------------------------------------------------------

// A product with no tile, wave count or grid named.  false: none of the small
// tiles fits, or the persistent kernel's 256-row tiles do and are estimated to
// be faster.
inline bool gemm_runs_small(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int cus, const SmallSpace& ws,
                            GemmSmallPlan* plan) {
  if (!plan_gemm_small(M, N, K, lda, ldb, cus, ws, {-1, 0}, plan)) return false;
  const int64_t t256 = M % 256 ? 0 : (M / 256) * (N / 256);
  if (2 * t256 > cus && persistent_cost(t256, K, cus, tail_fits(t256, K, 256, cus, ws)) <= plan->us) return false;
  // An odd number of 128-row blocks, a last round of 128 x 256 tiles that can be
  // split along K, and a K long enough for it (the more rounds, the less the
  // last one weighs): the persistent kernel.  us, its time against the small
  // tiles': 264 tiles K 4096 104 / 102, 5504 120 / 122, 14336 284 / 306; 289 of
  // 256 columns 4096 103 / 126, 14336 331 / 526; 345 K 4384 112 / 117, 13472 336 /
  // 478; 536 K 15072 551 / 673; 595 K 4928 216 / 189, 10656 432 / 546; 820 K 5408
  // 306 / 342; 1050 K 4832 356 / 344; 1090 K 13856 1011 / 1115.  A fuller last
  // round gains nothing (418 tiles K 10016 333 / 330, 472 K 14688 483 / 442).
  // Over 267 such shapes the choice costs 0.7 % in the mean, 2.2 % when the line
  // was at 320 tiles of K 4096 and more.
  const int64_t t128 = (M / 128) * (N / 256), rounds = t128 / cus, rest = t128 % cus;
  return !(M % 256 && rounds && rest && 20 * rest <= 9 * cus && K >= 1000 * (rounds + 3) &&
           tail_fits(t128, K, 128, cus, ws));
}

struct FusedPlan {
  bool small;  // the small-tile kernel runs, by `plan`
  bool first;  // the blocks are staged by a launch of their own before
  GemmSmallPlan plan;
};

// A fused launch of M x N x K that may run as a sequence: the staging of its
// `blocks` blocks on every CU, then a GEMM that waits for nothing.  Results do
// not depend on the choice (every output is the same K-ordered sum).
// fold.peers < 0: AllGather; second_copy: the blocks hold a two-shot
// all-reduce's reduced slices too; small_ok: the small-tile kernel can serve
// the call's done flags.
//
// The persistent kernel's workgroups copy between their tiles, which hides
// part of the copy behind others' tiles when there are several rounds and a
// round is longer than its share of the copy.  Staging first was faster (us,
// in the launch -> first) for AllGather below two rounds (12288x1280x2784 114
// -> 100) or K 2048 (16384x3584x1024 146 -> 138; 16384x3584x8192 805 -> 812)
// and for ReduceScatter below K 1024 (16384x8192, world 8: K 512 321 -> 233,
// 1536 453 -> 449, 3584 865 -> 871); the all-reduces, whose fold or second
// copy is spread over all rounds, gained nothing (8192^2, two-shot, K 768 171
// -> 179).  The tiles of the persistent kernel are too large where there are
// few (AllGather 4096x256x4096, world 16: 211 -> 32 with the small ones) and
// where few rows are folded by whole workgroups (ReduceScatter 4096x4096x256,
// world 16: 69 -> 50).
inline FusedPlan plan_fused(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int cus, const SmallFold& fold,
                            int blocks, bool second_copy, bool small_ok) {
  FusedPlan f = {};
  const bool reduce = fold.peers >= 0;
  const int64_t tiles = (M / 256) * (N / 256);
  f.small = small_ok && plan_gemm_small(M, N, K, lda, ldb, cus, {0, 0}, fold, &f.plan);
  if (f.small) {
    double one = persistent_cost(tiles, K, cus, false), sm = f.plan.us;
    if (reduce) {
      // a workgroup of the persistent kernel folds in about two of its rounds
      // when the last is not full; either kernel moves its stores and partials
      // at 2.5 TB/s at most
      const double bytes = 2.0 * N * ((double)M + (double)fold.peers * fold.rows) / 2.5e6;
      const bool partial = tiles > cus && tiles % cus;
      one += (partial ? 2.0 : 1.0) * fold_cost(fold, (double)fold.rows / 256 * (N / 256), 65536.0, cus);
      one = std::max(one, bytes) + (partial ? 14.0 : 7.0);
      sm = std::max(sm, bytes) + 8.0;
    }
    f.small = sm < one;
  }
  f.first = blocks > 0 &&
            (f.small || (reduce ? K < 1024 && !second_copy && fold.rows < M : tiles < 2 * cus || K < 2048));
  return f;
}

}  // namespace mk
