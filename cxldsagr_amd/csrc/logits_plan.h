// How a logits call is cut into (key split, query group) work-groups and how
// these are dealt to the XCDs. Plain C++, for the launcher and the kernel.
#pragma once

#include <stdint.h>

namespace dsa {

// Key range per work-group. `splits` is the stride of the per-split output
// (a multiple of 8 from 8 on); `live` of them hold keys and are launched, for
// each query group.
//
// Work-groups go to the eight XCDs round-robin by linear id, so an XCD's slots
// are the ids of one residue. XCD e takes the key splits e, e + 8, ... with all
// their query groups, which share those keys through its L2; the pairs of the
// last live % 8 splits go round. So each XCD gets as many pairs as the others,
// and about as many of any run of keys or rows: the pairs that a causal bound or
// a call's [starts, ends) leave without keys fall on all of them alike. (An
// eighth of the pairs in split order to each XCD leaves those of the last keys
// idle, and gave a causal prompt's early keys to a few: 4,100 rows x 4,200 keys
// 157 us, 6,000 x 6,000 234, 128 x 65,664 of which 30,128 are seen 66; now 120, 176 and 60.)
struct SplitPlan {
  int64_t qgroups, splits, per, live;
  // Slots of an XCD: its whole splits, then its share of the rest.
  constexpr int64_t slots() const { return live / 8 * qgroups + (live % 8 * qgroups + 7) / 8; }
  constexpr unsigned grid() const { return (unsigned)(8 * slots()); }
};

struct SplitPair {
  uint32_t split, group;
};

// The pair of work-group `id`; split >= live: none.
constexpr SplitPair dealt_pair(uint32_t id, uint32_t qgroups, uint32_t live) {
  const uint32_t xcd = id & 7, slot = id >> 3;
  const uint32_t whole = (live >> 3) * qgroups;
  const bool in_whole = slot < whole;
  const uint32_t at = in_whole ? slot : (slot - whole) * 8 + xcd;
  const uint32_t split = at / qgroups, group = at - split * qgroups;
  return {in_whole ? split * 8 + xcd : (live & ~7u) + split, group};
}

// The split with the least time by rounds of one work-group per CU, each
// kStartUs (operands and first keys) plus kStageUs per stage of `stage_keys`
// keys (the stage's MFMAs; both measured). Splitting for at least one
// work-group per CU and padding the splits to a multiple of 8 left a few
// work-groups, or one XCD's, to a second round that took as long as the first:
// 100 rows x 50,001 keys 81.8 -> 48.0 us, 200 rows x 16,584 keys 59.8 -> 34.6 us.
constexpr double kStartUs = 8.0, kStageUs = 3.0;

constexpr SplitPlan split_plan(int64_t rows, int64_t ldo, int64_t group_rows, int64_t stage_keys,
                               int64_t max_keys, int64_t cus) {
  SplitPlan p{};
  p.qgroups = (rows + group_rows - 1) / group_rows;
  const int64_t stages = (ldo + stage_keys - 1) / stage_keys;
  const int64_t most = stages < cus ? stages : cus;
  double best = 0.0;
  p.per = stages * stage_keys;
  // Split counts with splits of the same length cost the same, so each length is
  // looked at once, with its fewest splits: 45 of 256 counts at 64K columns, 0.8
  // instead of 2.8 us of host time, which callers spend ahead of the first launch.
  int64_t s = 1;
  while (s <= most) {
    const int64_t per_stages = (stages + s - 1) / s;
    const int64_t live = (stages + per_stages - 1) / per_stages;
    const int64_t rounds = (live * p.qgroups + cus - 1) / cus;
    const double cost = (double)rounds * (kStartUs + kStageUs * (double)per_stages);
    if (s == 1 || cost < best) {
      best = cost;
      p.per = per_stages * stage_keys;
    }
    if (per_stages == 1) break;
    s = (stages + per_stages - 2) / (per_stages - 1);  // the fewest with shorter ones
  }
  if (max_keys > 0 && p.per > max_keys) p.per = max_keys;
  p.live = (ldo + p.per - 1) / p.per;
  p.splits = p.live >= 8 ? (p.live + 7) / 8 * 8 : p.live;
  return p;
}

}  // namespace dsa
