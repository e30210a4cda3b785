// The order in which the workgroups of the packed forward (varlen_mfma.hip) take the query blocks of a launch; host
// and device code, so that a CPU test can walk it (tests/native/varlen_blocks.cpp).
#pragma once

#include <stdint.h>

#include "decode_items.hpp"  // ARENO_HD

namespace areno {

// What the i-th workgroup of a head takes: block `j` of the `nth` (in order) of the sequences that have more than j
// blocks.  Blocks are taken by their place in their sequence, the last ones first over all sequences: a block's keys
// grow with its place, and a launch ends soonest when the longest blocks start first.  With nb[s] blocks in sequence s,
// behind(j) = sum over s of max(0, nb[s] - j) blocks lie at place j or behind it; the i-th has the largest j with
// i < behind(j).  `most`: the largest nb.
struct BlockPlace {
  int j, nth;
};
// False: workgroup i is the nth that has no block.
template <typename Behind>
ARENO_HD bool block_place(int i, int most, Behind behind, BlockPlace& at) {
  const int all = behind(0);
  if (i >= all) {
    at.nth = i - all;
    return false;
  }
  int lo = 0, hi = most, behind_hi = 0;  // behind(lo) > i >= behind(hi)
  while (lo + 1 < hi) {
    const int mid = (lo + hi) >> 1, n = behind(mid);
    if (n > i) {
      lo = mid;
    } else {
      hi = mid;
      behind_hi = n;
    }
  }
  at.j = lo;
  at.nth = i - behind_hi;
  return true;
}

// Division of a sequence's tokens by a block's (8 .. 128) as a multiply and a shift, exact below 2^30: with
// s = ceil(log2(block)) and magic = floor(2^(30 + s) / block) + 1, (n * magic) >> (30 + s) == n / block
struct BlockDivision {
  uint32_t magic;
  int32_t shift;  // behind the product's high word
  ARENO_HD int operator()(int n) const {
    return static_cast<int>(static_cast<uint32_t>((static_cast<uint64_t>(static_cast<uint32_t>(n)) * magic) >> 32) >> shift);
  }
};
ARENO_HD BlockDivision block_division(int block) {
  int s = 3;
  while ((1 << s) < block) ++s;
  return {static_cast<uint32_t>((uint64_t{1} << (30 + s)) / static_cast<uint64_t>(block) + 1), s - 2};
}

}  // namespace areno
