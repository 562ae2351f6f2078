// How many pieces the keys of a padded prefill are cut into: host code, without HIP.
#pragma once

#include <algorithm>
#include <cstdint>

namespace mi_fa2 {

constexpr int kSplitRows = 128, kSplitStep = 128;   // a tile's packed rows, the keys of a step

struct SplitPlan {
  int64_t tiles;   // of packed rows, over all rows and kv heads
  int pieces;      // each tile's keys are cut into (1: none)
  int each;        // units of keys per piece
};

// The plan for a launch on a device of n_cus CUs whose keys are cut between units of `unit` keys (128,
// or a larger block of the paged cache): the number of pieces with the least time by this model (us,
// fitted to 18 shapes of 5 to 700 queries over 900 to 8,000 keys at 1 to 63 pieces, within 10% of the
// best of them everywhere):
//   unsplit, one work-group per CU or fewer:  6.5 + 1.45 per 128-key step of the longest tile;
//   split, one work-group per CU or fewer:    9.5 + 1.45 per step of a piece
//       + 0.033 per tile and piece (its partials written and read) + 0.05 per piece (the merge).
// Measured unsplit -> split: 150 queries over 3,001 keys 42.4 -> 19.6 us, 5 over 8,000 92.6 -> 13.9,
// 700 over 4,000 53.9 -> 35.8; 700 over 1,000 stays unsplit (19.1, split 21.8).
// Larger units never give more pieces than 128 keys do: the workspace is sized without them.
inline SplitPlan split_plan(int64_t n_cus, int64_t batch, int64_t heads_q, int64_t heads_kv,
                            int64_t seqlen_q, int64_t max_kv, int64_t unit = kSplitStep) {
  SplitPlan plan{0, 1, 1};
  const int64_t unsplit = batch * heads_q * ((seqlen_q + kSplitRows - 1) / kSplitRows);
  if (seqlen_q < 1 || unsplit < 1 || unsplit > n_cus) return plan;
  const int64_t packed = seqlen_q * (heads_q / heads_kv);
  plan.tiles = batch * heads_kv * ((packed + kSplitRows - 1) / kSplitRows);
  const int64_t row_groups = batch * heads_kv * ((packed + 31) / 32);   // four to a tile: what is written
  const int64_t steps = (max_kv + kSplitStep - 1) / kSplitStep, unit_steps = unit / kSplitStep;
  const int64_t units = (max_kv + unit - 1) / unit;
  int64_t most = std::min<int64_t>(n_cus / plan.tiles, steps);
  if (unit_steps > 1)
    most = split_plan(n_cus, batch, heads_q, heads_kv, seqlen_q, max_kv).pieces;
  int64_t best = 650 + 145 * steps - 100;   // in 10 ns; a split has to gain 1 us
  for (int64_t s = 2; s <= std::min(most, units); ++s) {
    const int64_t each = (units + s - 1) / s;
    const int64_t cost = 950 + 145 * each * unit_steps + 33 * row_groups * s / 40 + 5 * s;
    if (cost < best) {
      best = cost;
      plan.pieces = (int)s;
      plan.each = (int)each;
    }
  }
  return plan;
}

}  // namespace mi_fa2
