// Work decomposition of the grouped GEMM: which (tile, K range) items a workgroup processes, in which
// order, and which workgroup completes a tile that several workgroups shared along K.  Pure integer
// arithmetic on the problem table.  It runs on the host: fp8gmm_plan_grouped_gemm_launch (plan.cpp) writes the
// schedule out as the work list the kernels read, and the introspection entry points show it to the CPU tests.
#pragma once

#include <stdint.h>

#include <vector>

#include "fp8gmm.h"
#include "tiling.h"

#if defined(__HIPCC__)
#define FP8GMM_HD __host__ __device__ inline __attribute__((always_inline))
#else
#define FP8GMM_HD inline
#endif

namespace fp8gmm {

// ---- tail balancing (stream-K over the remainder of an XCD's tile range) ----
// A range of n tiles on W workgroups takes ceil(n / W) rounds; when the last round is mostly empty the
// remainder tiles are cut along K instead: the region's K = 128 steps are dealt out in equal contiguous
// pieces, up to W of them.  A piece that does not cover
// a whole tile leaves its fp32 accumulators in a workspace slot; a second, small kernel adds the pieces
// of such a tile in K order and runs the normal epilogue.  No workgroup ever waits for another one.
constexpr int kSkMinPairs = 4;        // never cut pieces shorter than this many K = 128 steps
constexpr int kSkMaxPieces = 8;       // average pieces per tile the region may be cut into
constexpr int kSkMaxRounds = 24;      // with more full rounds than this the tail cannot cost enough to share it
// What sharing costs, in K = 128 steps of time: kSkFixupLaunch for the second launch, which completes the shared tiles
// (5 us: the gap between two launches), and kSkPerSlot / 100 per workspace slot of an XCD while all eight of them share - a
// slot is 256 KB to write and to read again, 4 MB for the chip.  Measured with the pieces forced, 8 experts, K = 4096, 10
// remainder tiles on 32 workgroups: 2 pieces a tile 147 us, 3 154, 32 pieces over the ten tiles (40 slots) 161, not
// shared 146; 6 tiles: 135, 136 and, 5 pieces a tile, 139, 141 (36 slots), not shared 138 (to the rule a draw: not shared);
// K = 14336, 8 tiles: 2, 3 or 4 pieces 5536 - 5555 us for an MLP's step, not shared 5608; one XCD of the eight sharing 4
// tiles of 17 steps: 17 pieces 164 us for a layer's step, 12 164, 8 171, not shared 171.  Three quarters of a step per slot
// fit these figures better, but over the 181 launches of drawn layers that would then be planned otherwise 43 got faster
// and 42 slower by more than 3 %, 0.9 % faster in the mean: the price stays.  With the GELU epilogue to apply, a shared tile
// costs kSkGeluPerTile / 100 steps more.
constexpr int kSkFixupLaunch = 4;
constexpr int kSkPerSlot = 100;
constexpr int kSkGeluPerTile = 150;
constexpr int kPartialBytes = BM * BN * 4;  // one slot: the fp32 accumulators of one tile
constexpr int kTileOverhead = 4;      // fixed cost of a tile (epilogue, switch) in K = 128 steps, measured
constexpr int kSlotsPerWg = 2;        // a piece that starts inside a tile, one that ends inside a tile

struct Sched {
  const fp8gmm_gemm_problem* probs;
  int nprob, total_tiles;
  int wgs;                     // workgroups per XCD
  int range_begin, range_end;  // tiles of this XCD
  int dp_rounds;               // workgroup j takes tile dp_tile(j, i) of rounds i < dp_rounds
  int sk_begin;                // first tile of the stream-K region (== range_end: none)
  int sk_wgs;                  // workgroups that take a piece of the region
  int64_t sk_c0, sk_cost;      // cost before the region, cost of the region (K = 128 steps)
  int64_t total_cost;          // cost of all tiles
  bool halves;                 // the remainder [sk_begin, range_end) in tiles of half height, two per tile (sk_wgs is 0)
  bool gelu;                   // completing a shared tile includes the GELU epilogue
};

FP8GMM_HD int problem_end_tile(const Sched& s, int p) {
  return (p + 1 < s.nprob) ? s.probs[p + 1].tile_begin : s.total_tiles;
}
// last problem whose first tile is <= tile
FP8GMM_HD int problem_of_tile(const Sched& s, int tile) {
  int lo = 0, hi = s.nprob - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (s.probs[mid].tile_begin <= tile) lo = mid; else hi = mid - 1;
  }
  return lo;
}
// A tile of problem p costs ceil(k / 128) main-loop steps (1 for k = 0: its epilogue still has to run).
FP8GMM_HD int64_t tile_cost(const Sched& s, int p) {
  const int c = (s.probs[p].k + 127) / 128;
  return (int64_t)(c > 0 ? c : 1);
}
// Work before `tile` (0 <= tile <= total_tiles) when every tile counts its K steps plus `ov` steps of fixed
// overhead; cost_begin is the plan's prefix sum of the K steps alone.  ov = 0 is the unit in which tiles are
// cut along K; ov = kTileOverhead is the weight that balances the XCD ranges.
FP8GMM_HD int64_t work_before(const Sched& s, int tile, int ov) {
  const int p = problem_of_tile(s, tile);
  return (int64_t)s.probs[p].cost_begin + (int64_t)ov * s.probs[p].tile_begin +
         (int64_t)(tile - s.probs[p].tile_begin) * (tile_cost(s, p) + ov);
}
FP8GMM_HD int64_t cost_before(const Sched& s, int tile) { return work_before(s, tile, 0); }
// the tile that holds work offset c: work_before(t) <= c < work_before(t + 1); total_tiles past the end
FP8GMM_HD int tile_holding_work(const Sched& s, int64_t c, int ov) {
  if (c >= s.total_cost + (int64_t)ov * s.total_tiles) return s.total_tiles;
  int lo = 0, hi = s.nprob - 1;  // last problem whose prefix is <= c: it is not empty, as c < the total
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((int64_t)s.probs[mid].cost_begin + (int64_t)ov * s.probs[mid].tile_begin <= c) lo = mid; else hi = mid - 1;
  }
  const int64_t before = (int64_t)s.probs[lo].cost_begin + (int64_t)ov * s.probs[lo].tile_begin;
  return s.probs[lo].tile_begin + (int)((c - before) / (tile_cost(s, lo) + ov));
}
FP8GMM_HD int tile_holding_cost(const Sched& s, int64_t c) { return tile_holding_work(s, c, 0); }
// first tile whose preceding work is >= c (total_tiles if there is none)
FP8GMM_HD int first_tile_at_work(const Sched& s, int64_t c, int ov) {
  if (c <= 0) return 0;
  const int t = tile_holding_work(s, c, ov);
  if (t >= s.total_tiles) return s.total_tiles;
  return work_before(s, t, ov) == c ? t : t + 1;
}

// first tile of XCD x's range (x = 8: the end of the last one)
FP8GMM_HD int range_start(const Sched& s, int x) {
  const int64_t total_work = s.total_cost + (int64_t)kTileOverhead * s.total_tiles;
  return first_tile_at_work(s, (total_work * x + kNumXcd - 1) / kNumXcd, kTileOverhead);
}
// Striding takes a range of n tiles full + 1 rounds, sharing the remainder full + rem / W: worth a thought when that saves
// a twelfth of the launch by this count.  Measured, sharing returns about half of what the count promises (workgroups do
// not finish their rounds in step, so part of a last round is hidden anyway), and it costs the second launch and a
// round trip of the partial sums through memory: config 2's 4.25 rounds (15 % by the count) gain 6.5 %, launches
// of 14 rounds with a short tail (4 - 6.5 % by the count; the reference's example layer) lost 1 % of their step.
FP8GMM_HD bool remainder_may_share(int n_tiles, int W) {
  const int full = n_tiles / W, rem = n_tiles % W;
  return rem != 0 && full <= kSkMaxRounds && (int64_t)(W - rem) * 12 >= (int64_t)W * (full + 1);
}

// The tile that workgroup j of the XCD takes in round i of the strided part.  The position inside the round
// rotates from round to round: how fast a workgroup's steps run depends on where its tile sits in the round's
// 8 x 4 block (which operand slabs it shares with its neighbours, which memory channels those fall into - up to
// 6 % between columns of a weight-gradient problem), and a workgroup that kept one position for the whole launch
// would finish that much earlier or later than the others.
constexpr int kRoundRotation = 5;  // coprime to every workgroup count in use (multiples of 8 per XCD: 32, 38, ...)
FP8GMM_HD int dp_tile(const Sched& s, int j, int i) {
  return s.range_begin + s.wgs * i + (j + kRoundRotation * i) % s.wgs;
}

// ---- a last round of tiles of half height ----
// A remainder of at most half a round leaves half of the workgroups without a tile while the others run a whole one.  Cut
// into two items of half height (FP8GMM_ITEM_HALF_HEIGHT) it takes them kHalfStep / 100 of a step's time per K step and
// kHalfTile / 100 steps for the result and the switch; no partial sums, no second launch.  Measured on launches of one
// contraction that the tile rules leave to this tile, halves against whole tiles: less than a round, 0.65 - 0.8 of the time
// with up to 4 tiles on 32 workgroups, 0.75 - 0.95 with up to 16; a round and a bit 0.88 - 0.95, two 0.95, more 0.97 - 1.
// A range that may share is asked first, against whole tiles: what it then shares took 0.92 of the time that it took in halves
// (K = 14336, 4.25 rounds: 735 us against 761, whole tiles 771; remainders that are most of the launch 0.6 - 0.9), and halves
// are for what sharing does not pay for (K = 4096, 2.25 rounds: 136 us, whole tiles and shared 144).
// With the GELU an item stores three bytes per value: beyond kHalfGeluTiles / 16 of a round, halves of short contractions lose
// (12 tiles of 4 - 12 steps 1.03 - 1.15, 16 of 3 steps 1.23 of the time of whole ones), and from kHalfGeluSteps on they gain
// 2 - 12 %.  With the GELU's derivative, which reads the pre-activation, they take 0.55 - 0.98, with one launch of 15 losing.
// Against the plans without halves: 150 launches, three quarters of them with the GELU, 0.933 of the time in the mean, the worst
// 1.03; 120 with the derivative 0.77 (1.05); 150 weight gradients of skewed splits 0.989 (1.025).
constexpr int kHalfStep = 95;
constexpr int kHalfTile = 300;
constexpr int kHalfMaxRounds = 12;    // with more full rounds than this a last round is not worth the look
constexpr int kHalfGeluTiles = 5;
constexpr int kHalfGeluSteps = 32;
inline int64_t half_tile_x100(int64_t steps) { return steps * kHalfStep + kHalfTile; }
FP8GMM_HD bool remainder_may_halve(int n_tiles, int W, int64_t steps, int epilogue) {
  const int rem = n_tiles % W;
  return rem != 0 && 2 * rem <= W && n_tiles / W <= kHalfMaxRounds &&
         (!(epilogue & FP8GMM_EPI_GELU) || 16 * rem <= kHalfGeluTiles * W || steps >= kHalfGeluSteps);
}
// Workgroup j's item of the round behind `full` whole ones: which tile of the remainder, and which half of it.
FP8GMM_HD int half_position(int wgs, int j, int full) { return (j + kRoundRotation * full) % wgs; }

// One way to share a remainder: so many equal pieces, and the workspace slots that they leave.
struct SkSplit {
  int pieces, slots;
};
// The remainder of an XCD's range, the ways to share it, and when the range's last workgroup is through, from the launch's
// start and in hundredths of a K = 128 step: with whole tiles, and with each split but for its partial sums.
struct SkRemainder {
  int begin, tiles;      // first tile, how many
  int64_t c0, cost;      // cost before it, its own
  int n_splits;          // 0: not worth a thought
  SkSplit split[kSkMaxPieces];
  int64_t whole_x100, shared_x100[kSkMaxPieces], half_x100;   // of `sk_times`, which wants the splits
  bool timed;
  bool halves;           // if it is not shared, it runs in tiles of half height
};

// A tile that k piece ends fall inside of is left in k + 1 slots; one that no end falls inside of needs none.
inline int sk_slots(const Sched& s, const SkRemainder& r, int pieces) {
  int slots = 0, p = problem_of_tile(s, r.begin), problem_end = problem_end_tile(s, p), tile = r.begin;
  int64_t k = tile_cost(s, p), first = 0;   // the tile's steps, and those of the region before it
  bool cut = false;
  const int64_t length = r.cost / pieces;   // the end of piece j is at r.cost * j / pieces, without a division for each
  const int over = (int)(r.cost % pieces);
  int64_t at = 0;
  for (int j = 1, rest = 0; j < pieces; ++j) {
    at += length;
    rest += over;
    if (rest >= pieces) {
      rest -= pieces;
      ++at;
    }
    while (at >= first + k) {
      first += k;
      cut = false;
      if (++tile < problem_end) continue;
      do problem_end = problem_end_tile(s, ++p); while (tile >= problem_end);
      k = tile_cost(s, p);
    }
    if (at > first) {
      slots += cut ? 1 : 2;
      cut = true;
    }
  }
  return slots;
}

// Every tile of XCD s's range contracts over the same number of steps.
inline bool range_has_one_k(const Sched& s) {
  const int last = problem_of_tile(s, s.range_end - 1);
  const int64_t k = tile_cost(s, last);
  for (int p = problem_of_tile(s, s.range_begin); p < last; ++p)
    if (problem_end_tile(s, p) > s.probs[p].tile_begin && tile_cost(s, p) != k) return false;
  return true;
}

// Pieces that end where tiles end (so many per tile) leave one slot each if all tiles have one K; the most pieces that may be
// cut end anywhere.
inline void sk_splits(const Sched& s, SkRemainder& r) {
  const bool one_k = range_has_one_k(s);
  int64_t most = s.wgs;
  if (most > r.cost / kSkMinPairs) most = r.cost / kSkMinPairs;
  if (most > (int64_t)r.tiles * kSkMaxPieces) most = (int64_t)r.tiles * kSkMaxPieces;
  for (int per_tile = 2; r.n_splits < kSkMaxPieces; ++per_tile) {
    const bool per_tile_fits = (int64_t)per_tile * r.tiles <= most;
    const int pieces = per_tile_fits ? per_tile * r.tiles : (int)most;
    if (pieces <= r.tiles) break;   // at most one piece per tile: nothing to gain
    r.split[r.n_splits++] = SkSplit{pieces, one_k && pieces % r.tiles == 0 ? pieces : sk_slots(s, r, pieces)};
    if (!per_tile_fits) break;
  }
}

// Under one K the workgroups come to the remainder together; otherwise one that its whole tiles keep longer than the others
// begins later, and whether it gets a tile, a piece or nothing of the remainder decides when the range is through.
inline void sk_times(const Sched& s, SkRemainder& r) {
  if (r.timed) return;
  r.timed = true;
  const int W = s.wgs, full = (s.range_end - s.range_begin) / W;
  if (range_has_one_k(s)) {
    const int64_t steps = tile_cost(s, problem_of_tile(s, s.range_begin)), round = steps + kTileOverhead;
    r.whole_x100 = (full + (r.tiles > 0 ? 1 : 0)) * round * 100;
    r.half_x100 = full * round * 100 + half_tile_x100(steps);
    for (int i = 0; i < r.n_splits; ++i)
      r.shared_x100[i] = (full * round + kTileOverhead) * 100 + r.cost * 100 / r.split[i].pieces;
    return;
  }
  // steps of each workgroup's whole tiles (without a full round, of those that a remainder tile goes to: none yet)
  const int workgroups = full > 0 ? W : r.tiles;
  std::vector<int64_t> load(workgroups, 0);
  int tile = s.range_begin, p = problem_of_tile(s, tile);
  int64_t steps = tile_cost(s, p) + kTileOverhead, last = 0;
  for (int round = 0; round <= full; ++round) {
    int j = (int)((int64_t)kRoundRotation * round % W);   // position 0 of the round is workgroup -j's
    j = j == 0 ? 0 : W - j;
    const int end = tile + W < s.range_end ? tile + W : s.range_end;
    while (tile < end) {
      while (tile >= problem_end_tile(s, p)) steps = tile_cost(s, ++p) + kTileOverhead;
      int n = problem_end_tile(s, p) < end ? problem_end_tile(s, p) - tile : end - tile;   // tiles of one K side by side
      if (n > W - j) n = W - j;
      for (int i = 0; i < n; ++i) {
        if (round < full) load[j + i] += steps;
        else if (last < load[j + i] + steps) last = load[j + i] + steps;
      }
      tile += n;
      j = j + n == W ? 0 : j + n;
    }
  }
  int64_t longest = 0;
  for (const int64_t l : load) longest = longest < l ? l : longest;
  r.whole_x100 = (longest < last ? last : longest) * 100;
  r.half_x100 = longest * 100;
  for (int j = 0; j < W; ++j) {
    const int at = r.begin + half_position(W, j, full) / 2;
    if (at >= s.range_end) continue;
    const int64_t through = (j < workgroups ? load[j] * 100 : 0) + half_tile_x100(tile_cost(s, problem_of_tile(s, at)));
    if (r.half_x100 < through) r.half_x100 = through;
  }
  int64_t first = 0;   // the longest of the workgroups that get a piece
  for (int i = 0, j = 0; i < r.n_splits; ++i) {
    for (; j < r.split[i].pieces && j < workgroups; ++j) first = first < load[j] ? load[j] : first;
    const int64_t through_x100 = (first + kTileOverhead) * 100 + r.cost * 100 / r.split[i].pieces;
    r.shared_x100[i] = through_x100 < longest * 100 ? longest * 100 : through_x100;
  }
}

// The pieces with which a range is through first while `sharing` XCDs share (0: whole tiles), and when.  Every slot is written
// and read again.
inline int sk_pieces(const Sched& s, const SkRemainder& r, int sharing, int64_t* through_x100) {
  int pieces = 0;
  *through_x100 = r.whole_x100;
  for (int i = 0; i < r.n_splits; ++i) {
    const int64_t price_x100 = (int64_t)r.split[i].slots * kSkPerSlot + (s.gelu ? (int64_t)r.tiles * kSkGeluPerTile : 0);
    const int64_t takes_x100 = r.shared_x100[i] + kSkFixupLaunch * 100 + price_x100 * sharing / kNumXcd;
    if (takes_x100 < *through_x100) {
      *through_x100 = takes_x100;
      pieces = r.split[i].pieces;
    }
  }
  return pieces;
}

// Which remainders of a launch are shared, and in how many pieces each.  A range shares where that is faster for it, at the
// price of the XCDs that share; the launch does if its last range is through sooner for it, the second launch included, which
// also those wait for that do not share; and a range that with whole tiles is through before that keeps them.  Measured on the
// launches of drawn layers that are planned otherwise, against ranges that decide for themselves by the mean remainder tile,
// one slot a piece and all XCDs that might share: 269 take 6.7 % less time in the mean, 167 gain more than 3 %, 14 lose as much
// (a weight gradient of 7 x 3088 x 416, 37005 rows 154 -> 102 us, of 11 x 1552 x 1632, 51592 272 -> 211; GELU launches of about a
// round 38.7 -> 29.9 and 44.1 -> 34.6).  By the workgroups' times but each range for itself 3.2 %; with the slots and the XCDs
// counted but by the mean tile 105 launches took 1.4 % more.
inline void sk_decide(const Sched (&all)[kNumXcd], SkRemainder (&rem)[kNumXcd], int (&pieces)[kNumXcd]) {
  int sharing = 0;
  int64_t through[kNumXcd];
  for (int x = 0; x < kNumXcd; ++x) {
    pieces[x] = 0;
    if (rem[x].n_splits == 0) continue;
    ++sharing;
    sk_times(all[x], rem[x]);
  }
  if (sharing == 0) return;
  auto decide = [&](int at_once) {
    int count = 0;
    for (int x = 0; x < kNumXcd; ++x) {
      if (rem[x].n_splits == 0) continue;
      pieces[x] = sk_pieces(all[x], rem[x], at_once, &through[x]);
      count += pieces[x] > 0 ? 1 : 0;
    }
    return count;
  };
  // Where fewer share than might, the price of those that do is lower, and with it more may share: the smallest number
  // from there on that no more than that many share at.
  int count = decide(sharing);
  if (count == 0) return;
  if (count < sharing)
    for (sharing = count; (count = decide(sharing)) > sharing; ++sharing) {
    }
  int64_t whole = 0, last = 0;
  for (int x = 0; x < kNumXcd; ++x) {
    if (all[x].range_begin == all[x].range_end) continue;
    if (rem[x].n_splits == 0) sk_times(all[x], rem[x]);
    const int64_t alone = rem[x].halves ? rem[x].half_x100 : rem[x].whole_x100;
    const int64_t own = pieces[x] > 0 ? through[x] : alone + kSkFixupLaunch * 100;
    whole = whole < rem[x].whole_x100 ? rem[x].whole_x100 : whole;
    last = last < own ? own : last;
  }
  for (int x = 0; x < kNumXcd; ++x)
    if (last >= whole || rem[x].whole_x100 + kSkFixupLaunch * 100 <= last) pieces[x] = 0;
}

// Workgroup i runs on XCD i % 8.  The tile list is cut into 8 contiguous ranges of equal WORK, one per XCD,
// so that workgroups that share an L2 work on neighbouring tiles; the workgroups of an XCD stride through the
// range, and share its remainder along K when that pays.  k differs per problem in the wgrad form, and a
// tile costs its K steps plus a fixed part (epilogue, tile switch): balancing
// K steps alone left the XCDs that hold the short-K problems 17 % more work than the others.
inline void sched_init(Sched (&all)[kNumXcd], const fp8gmm_gemm_problem* probs, int nprob, int total_tiles, int wgs_per_xcd,
                       bool sk_enable, int epilogue = 0, bool balanced = false) {
  const int W = wgs_per_xcd;
  SkRemainder rem[kNumXcd] = {};
  for (int x = 0; x < kNumXcd; ++x) {
    Sched& s = all[x];
    s.gelu = (epilogue & (FP8GMM_EPI_GELU | FP8GMM_EPI_DGELU)) != 0;
    s.halves = false;
    s.probs = probs;
    s.nprob = nprob;
    s.total_tiles = total_tiles;
    s.wgs = W;
    s.total_cost = x > 0 ? all[0].total_cost : 0;
    if (x == 0) s.total_cost = cost_before(s, total_tiles);
    s.range_begin = x > 0 ? all[x - 1].range_end : 0;
    s.range_end = range_start(s, x + 1);
    const int n_x = s.range_end - s.range_begin;
    s.dp_rounds = (n_x + W - 1) / W;  // plain striding: the last round may be partial
    s.sk_begin = s.range_end;
    s.sk_wgs = 0;
    s.sk_c0 = 0;
    s.sk_cost = 0;
    SkRemainder& r = rem[x];
    r.tiles = n_x % W;
    r.begin = s.range_end - r.tiles;
    if (sk_enable && remainder_may_share(n_x, W)) {
      r.c0 = cost_before(s, r.begin);
      r.cost = cost_before(s, s.range_end) - r.c0;
      sk_splits(s, r);
    }
    if (balanced && r.tiles > 0 && remainder_may_halve(n_x, W, tile_cost(s, problem_of_tile(s, r.begin)), epilogue)) {
      sk_times(s, r);
      r.halves = r.half_x100 < r.whole_x100;
    }
  }
  int pieces[kNumXcd] = {};
  if (sk_enable) sk_decide(all, rem, pieces);
  for (int x = 0; x < kNumXcd; ++x) {
    Sched& s = all[x];
    if (pieces[x] == 0) {
      if (rem[x].halves) {
        s.halves = true;
        s.dp_rounds = (s.range_end - s.range_begin) / W;
        s.sk_begin = rem[x].begin;
      }
      continue;
    }
    s.dp_rounds = (s.range_end - s.range_begin) / W;
    s.sk_begin = rem[x].begin;
    s.sk_wgs = pieces[x];
    s.sk_c0 = rem[x].c0;
    s.sk_cost = rem[x].cost;
  }
}

// piece boundaries of the stream-K region, relative to sk_c0
FP8GMM_HD int64_t sk_bound(const Sched& s, int j) { return s.sk_cost * j / s.sk_wgs; }

// Tile `local` of a problem with tiles_m x tiles_n tiles -> its row / column block.  The m index runs fastest
// inside groups of kRasterRows m-tiles: 32 consecutive tiles (one round of an XCD's workgroups) then form an
// 8 x 4 block that needs 12 operand slabs, whatever the shape of the problem (a 56 x 16 weight-gradient
// problem walked with m fastest over all 56 rows would need 33).
constexpr int kRasterRows = 8;
FP8GMM_HD void tile_origin(int m, int n, int local, int tile_m, int tile_n, int* m0, int* n0) {
  const int tiles_m = (m + tile_m - 1) / tile_m, tiles_n = (n + tile_n - 1) / tile_n;
  const int group = local / (kRasterRows * tiles_n);
  const int within = local - group * (kRasterRows * tiles_n);
  const int rows = tiles_m - group * kRasterRows < kRasterRows ? tiles_m - group * kRasterRows : kRasterRows;
  *m0 = (group * kRasterRows + within % rows) * tile_m;
  *n0 = (within / rows) * tile_n;
}
FP8GMM_HD void tile_origin(int m, int n, int local, int* m0, int* n0) { tile_origin(m, n, local, BM, BN, m0, n0); }

struct Item {
  int tile, prob, m0, n0;
  int k_begin, nk;  // K = 128 steps: first one, how many (0 for a problem without K)
  int slot;         // workspace slot of a partial piece, -1: the piece is the whole tile
};
struct Cursor {
  int dp_i;     // strided tiles already taken
  int sk_tile;  // next tile of this workgroup's stream-K piece, -1: none left
};

FP8GMM_HD void cursor_init(const Sched& s, int j, Cursor& c) {
  c.dp_i = 0;
  c.sk_tile = -1;
  if (j < s.sk_wgs && sk_bound(s, j) < sk_bound(s, j + 1)) c.sk_tile = tile_holding_cost(s, s.sk_c0 + sk_bound(s, j));
}
FP8GMM_HD bool cursor_valid(const Sched& s, int j, const Cursor& c) {
  return (c.dp_i < s.dp_rounds && dp_tile(s, j, c.dp_i) < s.sk_begin) || c.sk_tile >= 0;
}
// `prob_hint`: a problem at or before the one that holds the cursor's tile (a workgroup's tiles come in
// increasing order, so the previous item's problem will do); negative: search the whole table.
FP8GMM_HD Item cursor_item(const Sched& s, int xcd, int j, const Cursor& c, int prob_hint = -1) {
  const bool dp = c.dp_i < s.dp_rounds && dp_tile(s, j, c.dp_i) < s.sk_begin;
  Item it;
  it.tile = dp ? dp_tile(s, j, c.dp_i) : c.sk_tile;
  if (prob_hint < 0) {
    it.prob = problem_of_tile(s, it.tile);
  } else {
    it.prob = prob_hint;
    while (it.prob + 1 < s.nprob && s.probs[it.prob + 1].tile_begin <= it.tile) ++it.prob;
  }
  tile_origin(s.probs[it.prob].m, s.probs[it.prob].n, it.tile - s.probs[it.prob].tile_begin, &it.m0, &it.n0);
  const int real_nk = (s.probs[it.prob].k + 127) / 128;  // a K tail is zero-filled
  it.k_begin = 0;
  it.nk = real_nk;
  it.slot = -1;
  if (!dp) {
    const int64_t c_t = cost_before(s, it.tile) - s.sk_c0, k_t = tile_cost(s, it.prob);
    const int64_t lo = sk_bound(s, j), hi = sk_bound(s, j + 1);
    const int64_t p_lo = (lo > c_t ? lo : c_t) - c_t;
    const int64_t p_hi = (hi < c_t + k_t ? hi : c_t + k_t) - c_t;
    if (p_hi - p_lo < k_t) {  // only tiles with real K work are ever cut (k_t > 1)
      it.k_begin = (int)p_lo;
      it.nk = (int)(p_hi - p_lo);
      it.slot = kSlotsPerWg * (xcd * s.wgs + j) + (p_lo == 0 ? 1 : 0);
    }
  }
  return it;
}
FP8GMM_HD void cursor_advance(const Sched& s, int j, Cursor& c) {
  if (c.dp_i < s.dp_rounds && dp_tile(s, j, c.dp_i) < s.sk_begin) {
    ++c.dp_i;
    return;
  }
  if (c.sk_tile < 0) return;
  const int p = problem_of_tile(s, c.sk_tile);
  const int64_t t_end_cost = cost_before(s, c.sk_tile) - s.sk_c0 + tile_cost(s, p);
  c.sk_tile = (t_end_cost < sk_bound(s, j + 1) && c.sk_tile + 1 < s.range_end) ? c.sk_tile + 1 : -1;
}



// The tile that the workgroup of piece boundary j (1 <= j < sk_wgs) completes in the fix-up pass, or -1:
// the FIRST boundary strictly inside a tile owns it.  `first_piece_wg` is the workgroup that holds the piece
// from the tile's first K step (slot kSlotsPerWg * wg + 1); the following pieces come from workgroups
// j, j + 1, ... (slot kSlotsPerWg * wg) while their boundary lies inside the tile.
FP8GMM_HD int fixup_tile(const Sched& s, int j, int* n_following) {
  *n_following = 0;
  if (j < 1 || j >= s.sk_wgs) return -1;
  const int64_t b = sk_bound(s, j);
  const int tile = tile_holding_cost(s, s.sk_c0 + b);
  if (tile >= s.range_end) return -1;
  const int64_t c_t = cost_before(s, tile) - s.sk_c0, k_t = tile_cost(s, problem_of_tile(s, tile));
  if (b == c_t) return -1;                    // the boundary coincides with a tile boundary
  if (sk_bound(s, j - 1) > c_t) return -1;    // an earlier boundary inside the same tile owns it
  int n = 0;
  for (int q = j; q < s.sk_wgs && sk_bound(s, q) < c_t + k_t; ++q) ++n;
  *n_following = n;
  return tile;
}

}  // namespace fp8gmm
