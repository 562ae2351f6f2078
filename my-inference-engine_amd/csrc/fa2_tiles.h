// Which (row, query head, query tile) a work-group of a prefill launch works on.
#pragma once

#include "fa2_common.h"

namespace mi_fa2 {

// Work-groups are dispatched round-robin over the device's X XCDs (work-group w runs on XCD w % X),
// and each XCD has its own L2.  X is read from the device (8 on a whole MI355X, fewer on a
// partitioned one; a power of two, passed as log2; with X = 1 every mapping below reduces to plain
// rank-major order).  The (row, query head, query tile) of work-group w is chosen so that the
// query heads sharing one kv head (one class c = (row, kv head)) and tile run on the same XCD, so
// one L2 holds their K/V, and so that every XCD walks its tiles longest first with the same mix
// of tile lengths.  rank 0 is a row's last (longest) query tile.
//   * classes dividing X (one or a few long rows): each class has X / classes XCDs of its own, and
//     every XCD walks its class's tiles rank by rank;
//   * otherwise (batches of rows, of equal or ragged lengths): the groups (class, rank) are taken
//     rank-major, group j = rank * stride + c with an odd stride >= classes, and dealt to XCD
//     j % X.  The odd stride rotates a class over the XCDs from one rank to the next, so rows of
//     different lengths spread over all XCDs instead of pinning a class -- and its row's whole
//     work -- to XCD c % X (16 ragged rows of U[16, 1024] tokens on 8 XCDs: the busiest XCD
//     carried 1.9x the least busy one's tiles that way).
//   * packed batches of at most 64 rows (the varlen modes) number only the real (class, rank)
//     groups, rank-major, and deal group j to XCD j % X (prefill_item_packed): a row's class moves
//     over the XCDs as shorter rows drop out of the later ranks.
inline int prefill_grid_size(int classes, int group, int n_qt, int xcd_log2) {
  const int X = 1 << xcd_log2;
  if (classes < X && X % classes == 0) {
    const int per_xcd = (classes * group * n_qt + X - 1) / X;
    return X * per_xcd;
  }
  const int stride = classes | 1;
  return X * ((stride * n_qt + X - 1) / X) * group;
}

// The launch's item map: the divisors of prefill_item, log2 of the device's XCD count and, when
// the classes divide the XCDs, log2 of the XCDs per class (else -1).
struct ItemMap {
  FastDiv group, stride, hkv;
  int32_t classes, xcd_shift, xcd_log2;
};
inline ItemMap make_item_map(int classes, int group, int Hkv, int xcd_log2) {
  ItemMap m{make_fastdiv(group), make_fastdiv(classes | 1), make_fastdiv(Hkv), classes, -1,
            xcd_log2};
  const int X = 1 << xcd_log2;
  if (classes < X && X % classes == 0) {
    m.xcd_shift = 0;
    while ((classes << m.xcd_shift) < X) ++m.xcd_shift;
  }
  return m;
}

// Returns false for the padding work-groups of the grid.
__device__ inline bool prefill_item(int w, const ItemMap& map, int n_qt, int& b, int& h,
                                    int& rank) {
  const int x = w & ((1 << map.xcd_log2) - 1), slot = w >> map.xcd_log2;
  const int group = (int)map.group.d;
  int c;
  if (map.xcd_shift >= 0) {
    const int X = 1 << map.xcd_shift;  // XCDs per class
    c = x >> map.xcd_shift;
    const int u = slot * X + (x & (X - 1));
    rank = fdiv(u, map.group);
    h = (c - fdiv(c, map.hkv) * (int)map.hkv.d) * group + (u - rank * group);
  } else {
    const int stride = (int)map.stride.d;
    const int sg = fdiv(slot, map.group);
    const int j = (sg << map.xcd_log2) + x;  // group, rank-major
    rank = fdiv(j, map.stride);
    c = j - rank * stride;
    if (c >= map.classes) return false;
    h = (c - fdiv(c, map.hkv) * (int)map.hkv.d) * group + (slot - sg * group);
  }
  if (rank >= n_qt) return false;
  b = fdiv(c, map.hkv);
  return true;
}

}  // namespace mi_fa2
