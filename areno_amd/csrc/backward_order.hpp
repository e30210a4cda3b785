// The order in which the workgroups of the matrix-core backward kernels (attention_backward_mfma.hip) take the blocks
// of packed rows; host and device code, so that a CPU test can walk it (tests/native/backward_order.cpp, backward_launch_order.cpp).
#pragma once

#include <stdint.h>

#include "decode_items.hpp"  // ARENO_HD

namespace areno {

// The block of packed rows the i-th workgroup (of a head) takes.  Blocks differ in cost by their place in their
// sequence (a query block late in a long sequence sees the most keys, a key block early in it is seen by the most
// queries), and a launch ends soonest when the expensive blocks start first.  The lengths are not known on the host,
// so the order assumes sequences of about equal length: the packed blocks are cut into num_seqs runs and taken run by
// run in turn, the expensive end of every run first (`from_end`: the last block of a run).  Any order is correct.
ARENO_HD int64_t block_in_cost_order(int64_t i, int64_t blocks, int num_seqs, bool from_end) {
  // (32 bits, which a launch's workgroups have: a 64-bit division is 100 instructions in front of a workgroup's first fetch)
  const uint32_t all = static_cast<uint32_t>(blocks), at = static_cast<uint32_t>(i);
  const uint32_t runs = num_seqs > 0 ? static_cast<uint32_t>(num_seqs) : 1, per = all / runs, rest = all - per * runs;
  if (per == 0) return from_end ? all - 1 - at : at;
  if (from_end) {  // the blocks behind the last whole run belong to the end of the last sequence: first
    if (at < rest) return all - 1 - at;
    const uint32_t j = at - rest;
    return (j % runs) * per + (per - 1 - j / runs);
  }
  if (at >= per * runs) return at;
  return (at % runs) * per + at / runs;
}

// The same for `tokens` rows in blocks of `rows`, whose sequences need not end where blocks do: a run is led by the block that
// holds its sequence's first row (`from_end`: its last), which holds rows of the neighbouring sequence as well.  Cut by
// blocks alone that block, the most expensive one of all, was the last of the run before (or the first of the one behind) and
// started when the others were done: the backward of 3 x 3 196 tokens, 16 / 4 heads of 192, took 2 238 us and takes 1 536 (3 x
// 3 200: 1 508); 2 x 1 500, 32 / 8 of 128: 225 -> 190; of 1 700 launches equal lengths take 0.99 of the time, ragged ones 1.00.
// What takes a division by more than the runs is worked out on the host: every workgroup of a launch starts with this.
struct BlockOrder {
  int32_t blocks, runs;
  int32_t per;      // whole blocks of a sequence; 0: not to be used (short sequences, or too many for the fractions' 32 bits)
  int32_t more;     // rows of all runs behind those
  uint32_t step;    // more / (runs * rows), and the part of a run that a last row lies in front of its end by, in 2^-32
  uint32_t before;
};
inline BlockOrder block_order(int64_t tokens, int rows, int num_seqs) {
  const int64_t runs = num_seqs > 0 ? num_seqs : 1, share = runs * rows, blocks = (tokens + rows - 1) / rows;
  BlockOrder o = {static_cast<int32_t>(blocks), static_cast<int32_t>(runs), 0, 0, 0, 0};
  // (step and before are rounded up, by less than 2^-32 each: a run's fraction, of whole parts of `share`, stays below the next)
  if (blocks > INT32_MAX || runs >= (int64_t{1} << 31) / share || tokens < 2 * share) return o;
  o.per = static_cast<int32_t>(tokens / share);
  o.more = static_cast<int32_t>(tokens - o.per * share);
  o.step = static_cast<uint32_t>(((static_cast<uint64_t>(o.more) << 32) + share - 1) / share);
  o.before = static_cast<uint32_t>(((static_cast<uint64_t>(share - runs) << 32) + share - 1) / share);
  return o;
}
ARENO_HD int32_t block_in_launch_order(int32_t i, const BlockOrder& o, int rows, bool from_end) {
  if (o.per == 0) return static_cast<int32_t>(block_in_cost_order(i, o.blocks, o.runs, from_end));
  const uint32_t runs = static_cast<uint32_t>(o.runs), place = static_cast<uint32_t>(i) / runs;
  int32_t run = i - static_cast<int32_t>(place * runs), behind = static_cast<int32_t>(place);
  const int32_t extra = i - o.per * o.runs;
  if (extra >= 0) {  // the runs that hold a block more than `per`: their cheap ends, last
    const int64_t share = static_cast<int64_t>(runs) * rows;
    if (!from_end && extra >= o.more / rows) return o.blocks - 1;  // (the rows behind the last whole block)
    run = static_cast<int32_t>(((from_end ? extra * share + runs : (extra + 1) * share) + o.more - 1) / o.more) - 1;
    behind = o.per;
  }
  if (from_end) return (run + 1) * o.per + static_cast<int32_t>((static_cast<uint64_t>(run + 1) * o.step + o.before) >> 32) - 1 - behind;
  return run * o.per + static_cast<int32_t>(static_cast<uint64_t>(run) * o.step >> 32) + behind;
}

}  // namespace areno
