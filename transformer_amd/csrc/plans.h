// The host's choices of grid, tile and split that depend on nothing but sizes: plain C++, so that the tests can ask them.
#pragma once

#include <stdint.h>

namespace mla {

// ---- the attention kernels' grids (prefill_fwd.hip, prefill_bwd.hip)
// Whether a causal attention kernel's grid runs one tile of 128 rows per workgroup, longest first, instead of mirrored
// pairs (tiles r and n - 1 - r of one (b, h), always the same work together).  Pairs start a new round of workgroups for
// any remainder; single tiles fill the chip to the end but start twice as often, without the next tile's prefetch, and
// share less of a (b, h) in L2.  Results are the same bit for bit.  Times in units of a pair's, n_bh (b, h) of n tiles:
//   single tiles: the work over the workgroups that run at once, plus what the starts cost, at least the longest tile;
//   pairs: whole rounds; where two workgroups share a CU, a last round of one per CU takes a fraction of that.
// The constants are fitted, not derived; what they stand for is beside them.  Checked over 150 random sizes of both head
// layouts (14 heads of 64 + 64, 16 of 128 + 64 with shared k_rope; B to 24, T 150 to 8000, B T to 24000), each kernel timed
// in both grids: against pairs everywhere the forward takes 5.0 % less on average (at most 28 % less, 2.5 % more), the
// backward 4.7 % less through dK/dV (21 % less, 0.5 % more) and 1.2 % less through dQ (13 % less, 2.3 % more); against the
// faster grid of each size the rule leaves 1.3 %, 0.1 % and 1.6 %, the most (16 % of a forward, 13 % of a backward) where
// fewer than 256 pairs run one to a CU.  Examples, pairs -> single (us, B x T), forward / whole backward:
//   3 x 3000 180 -> 144 / 530 -> 468;  2 x 2600 76 -> 63 / 263 -> 191;  4 x 2900 148 -> 130 / 450 -> 418;  3 x 1900 60 ->
//   52 / 206 -> 169;  but whole rounds: 12 x 2048 265 -> 279 / 911 -> 990;  4 x 4096 319 -> 320 / 1060 -> 1076.
struct TileGrid {
  int64_t n_bh, n;
  bool square;  // causal from the first key: tile sizes 1 .. n, else alike
  double longest() const { return square ? (double)n / (double)(n + 1) : 0.5; }
  double work() const { return (double)n_bh * (double)n / 2; }
  int64_t pairs() const { return n_bh * ((n + 1) / 2); }
};
inline bool single_tiles_one_per_cu(const TileGrid& g) {  // 256 workgroups at once
  if (g.n < 2) return false;
  const double pair = (double)((g.pairs() + 255) / 256);
  // a start (nothing prefetched) costs a pair's tiles 1 / n of their time; never less than the longest tile
  const double most = g.work() / 256 * (1.0 + 1.0 / (double)g.n), single = most > g.longest() ? most : g.longest();
  return single < 0.97 * pair;  // (what is this close stays in pairs)
}
inline bool single_tiles_two_per_cu(const TileGrid& g) {  // 512, two on a CU
  if (g.n < 2) return false;
  const int64_t rest = g.pairs() % 512;
  // a last round of at most 160 pairs, alone on their CUs: 0.42 of a round of two a CU; to 256, where the dispatcher puts
  // some on one CU, up to 0.67; beyond, a whole round
  const double last = rest == 0 ? 0.0 : rest > 256 ? 1.0 : 0.42 + (rest > 160 ? 0.25 * (double)(rest - 160) / 96 : 0.0);
  const double pair = (double)(g.pairs() / 512) + last;
  // a start costs 0.6 / n (the other workgroup of the CU runs on); the longest tile, alone on its CU at the end, 0.8
  const double most = g.work() / 512 * (1.0 + 0.6 / (double)g.n), low = 0.8 * g.longest();
  return (most > low ? most : low) < 0.95 * pair;
}

// ---- norm_linear.hip's output tiles
constexpr int kNlBK = 32;  // k per stage

struct NlPlan {
  int kind;  // 0 NlWide (+ NlRest), 1 NlHalf, 2 NlSmall
  int64_t n_nt, n_wide, n_rest;
};

// The least of: rounds of 256 workgroups (one per CU) x (the tile's time per stage x stages + what a workgroup takes
// beside them), both fitted to the measured calls (us at M x N x K, wide / half / small tiles): 12288 x 2560 x 1792 129.0 /
// 146.0 / 168.8 (two full rounds of wide tiles), 8192 x 2624 x 2048 132.8 / 127.7 / 140.7, 2735 x 2000 x 1632 57.1 / 36.6 /
// 40.2, 1000 x 2624 x 2048 61.7 / 42.6 / 39.3 (wide tiles leave most of the chip idle).  Small tiles share a CU.
inline NlPlan nl_plan(int64_t M, int64_t N, int64_t K) {
  NlPlan best{};
  double best_t = 1e300;
  const double stages = (double)(K / kNlBK);
  static const int bn[3] = {256, 256, 128}, bm[3] = {256, 128, 128};
  static const double ts[3] = {1.0, 0.6, 0.39}, fixed[3] = {6.0, 4.0, 1.5};
  for (int kind = 0; kind < 3; ++kind) {
    const int64_t mt = (M + bm[kind] - 1) / bm[kind];
    int64_t nt = (N + bn[kind] - 1) / bn[kind], rest = 0;
    if (kind == 0 && nt > 1 && N % 256 != 0 && N % 256 <= 128) {
      --nt;
      rest = mt;
    }
    const int64_t wide = mt * nt;
    // the remainder's tiles fill the last round's free CUs first
    double rounds = (double)((wide + 255) / 256);
    const int64_t over = rest - (int64_t)(rounds * 256 - wide);
    if (over > 0) rounds += 0.6 * (double)((over + 255) / 256);
    const double t = rounds * (stages * ts[kind] + fixed[kind]);
    if (t < best_t) {
      best_t = t;
      best = NlPlan{kind, nt, wide, rest};
    }
  }
  return best;
}

// ---- wgrad.hip's output tiles and token segments
constexpr int kWgSt = 32;  // tokens per stage

struct WgPlan {
  int narrow, S, seg, nt, kt;
  int64_t part_bytes;
};

// The plan of least estimated time: rounds of 256 workgroups (one per CU), each its stages at the measured 1.05 us (wide
// tile: 128 stages of 4096 x 2048 took 124-134 us) or 0.62 us (narrow) plus 4 us of start and stores, and where the
// tokens are cut the second kernel with its partials at 4 TB/s.  Wide tiles stage fewer bytes per product, so they win
// where the weight has enough of them; narrow ones (and more segments) where it has few: 896 x 384 makes 12.
inline WgPlan wg_plan(int64_t M, int64_t N, int64_t K) {
  WgPlan best{};
  double best_t = 1e300;
  const int64_t st = (M + kWgSt - 1) / kWgSt;
  for (int narrow = 0; narrow < 2; ++narrow) {
    const int64_t TN = 256, TK = narrow ? 128 : 256;
    const int64_t nt = (N + TN - 1) / TN, kt = (K + TK - 1) / TK, tiles = nt * kt;
    const double ts = narrow ? 0.62 : 1.05;  // us per stage of a workgroup
    for (int64_t S = 1; S <= 32 && S <= st; ++S) {
      const int64_t per = (st + S - 1) / S;
      if ((st + per - 1) / per != S) continue;  // fewer segments hold the same stages
      const double rounds = (double)((tiles * S + 255) / 256);
      double t = rounds * ((double)per * ts + 4.0);
      const int64_t pb = S > 1 ? tiles * S * TN * TK * 4 : 0;
      if (S > 1) t += 4.0 + (double)pb / 4.0e6;
      if (pb > (256ll << 20)) continue;
      if (t < best_t) {
        best_t = t;
        best = WgPlan{narrow, (int)S, (int)(per * kWgSt), (int)nt, (int)kt, pb};
      }
    }
  }
  return best;
}

}  // namespace mla
