// Units that belong to one item (query block) each, for launches of the prefill kernel with fewer items than units: how many
// tile steps a unit takes, and which item it works on.  Host and device code, so that a CPU test can walk it
// (tests/native/prefill_steps.cpp); why and when is at place_of_unit in prefill_mfma.hip.
#pragma once

#include <stdint.h>

#include "decode_items.hpp"  // ARENO_HD

namespace areno {

constexpr uint32_t kSegmentSteps = 8;  // what a segment costs besides its steps, in steps
constexpr float kMostLeastSteps = 8.0f;

// Steps a unit: the least share, of `least` steps or more, at which all items together need no more than the launch's units
// (units_at(share)); 0 if that is a segment's cost larger than equal shares, which it then stays with.  0 < items < units.
template <typename UnitsAt>
ARENO_HD uint32_t share_of_items(uint32_t total, uint32_t items, uint32_t units, float least, UnitsAt units_at) {
  const uint32_t spare = units - items, even = (total + units - 1) / units;
  const uint32_t least_steps = static_cast<uint32_t>(least < 1.0f ? 1.0f : least > kMostLeastSteps ? kMostLeastSteps : least);
  uint32_t lo = even > least_steps ? even : least_steps;
  uint32_t hi = (total + spare - 1) / spare;  // (at which a unit more for every item does)
  if (hi < lo) hi = lo;
  if (hi >= lo + kSegmentSteps) {
    hi = lo + kSegmentSteps - 1;
    if (units_at(hi) > units) return 0;
  }
  while (lo < hi) {
    const uint32_t mid = (lo + hi) / 2;
    if (units_at(mid) <= units) {
      hi = mid;
    } else {
      lo = mid + 1;
    }
  }
  return lo;
}

// The item that unit `unit` works on, items taking of(i) units one behind the other, and which of the item's units it is.
// Of an item of several units each leaves a partial, so the merge finds them at the units behind the first.
struct ItemUnit {
  int item;  // -1: a unit without work
  int nth;
};
template <typename Of>
ARENO_HD ItemUnit item_of_unit(int unit, int items, Of of) {
  int first = 0;
  ItemUnit at = {-1, 0};
  for (int i = 0; i < items; ++i) {
    const int n = of(i);
    if (unit >= first && unit < first + n) at.item = i, at.nth = unit - first;
    first += n;
  }
  return at;
}

}  // namespace areno
