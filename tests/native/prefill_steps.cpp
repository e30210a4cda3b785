// CPU check of the prefill kernel's step geometry (areno_amd/csrc/prefill_steps.hpp): the closed forms for the tile
// steps in front of a query block and the bisection that finds the block of a step, held against a walk over the
// blocks with block_tiles(), the one definition of which key tiles a block sees.  Built by
// tests/test_prefill_steps_cpu.py with g++; no GPU code.
#include <math.h>
#include <stdint.h>
#include <stdio.h>

#include <vector>

#include "../../areno_amd/csrc/item_units.hpp"
#include "../../areno_amd/csrc/prefill_steps.hpp"

using namespace areno;

// Checks one sequence shape; returns 0 or writes what differs.  `every_step` also places every step of the sequence
// (quadratic in the sequence's size: for small shapes).
extern "C" int prefill_steps_check(int n_new, int ctx, int tq, int window_left, int every_step, long long* steps_out,
                                   char* msg, int msg_len) {
  const int blocks = query_blocks(n_new, tq);
  long long walked = 0;
  for (int j = 0; j <= blocks; ++j) {
    const int closed = steps_before_block(n_new, ctx, j, tq, window_left);
    if (closed != walked) {
      snprintf(msg, msg_len, "steps_before_block(n_new=%d, ctx=%d, j=%d, tq=%d, window=%d) = %d, the walk gives %lld",
               n_new, ctx, j, tq, window_left, closed, walked);
      return 1;
    }
    if (j == blocks) break;
    const BlockTiles b = block_tiles(n_new, ctx, j, tq, window_left);
    if (b.count() < 1 || b.cnt < 1 || b.tile_lo < 0) {
      snprintf(msg, msg_len, "block_tiles(n_new=%d, ctx=%d, j=%d, tq=%d, window=%d): count %d, tokens %d, tile_lo %d",
               n_new, ctx, j, tq, window_left, b.count(), b.cnt, b.tile_lo);
      return 1;
    }
    // the block of a step: the block's first and last step always, every step on request
    for (int k = 0; k < b.count(); k = (every_step || k == b.count() - 1) ? k + 1 : b.count() - 1) {
      const int off = static_cast<int>(walked) + k;
      const int found = block_of_step(n_new, ctx, tq, window_left, off);
      if (found != j) {
        snprintf(msg, msg_len, "block_of_step(n_new=%d, ctx=%d, tq=%d, window=%d, off=%d) = %d, the walk gives %d",
                 n_new, ctx, tq, window_left, off, found, j);
        return 1;
      }
    }
    walked += b.count();
  }
  if (sequence_steps(n_new, ctx, tq, window_left) != walked) {
    snprintf(msg, msg_len, "sequence_steps(n_new=%d, ctx=%d, tq=%d, window=%d) differs from the walk", n_new, ctx, tq,
             window_left);
    return 1;
  }
  *steps_out = walked;
  return 0;
}

// The same over a grid: n_new in [0, n_hi], ctx in [0, ctx_hi], every tq and window given.
extern "C" int prefill_steps_check_grid(int n_hi, int ctx_hi, const int* tqs, int num_tq, const int* windows,
                                        int num_windows, long long* shapes_out, char* msg, int msg_len) {
  long long shapes = 0, steps = 0;
  for (int t = 0; t < num_tq; ++t)
    for (int w = 0; w < num_windows; ++w)
      for (int ctx = 0; ctx <= ctx_hi; ++ctx)
        for (int n = 0; n <= n_hi; ++n) {
          if (prefill_steps_check(n, ctx, tqs[t], windows[w], 1, &steps, msg, msg_len)) return 1;
          ++shapes;
        }
  *shapes_out = shapes;
  return 0;
}

// Every unit of a launch of few items (areno_amd/csrc/item_units.hpp): the least share that does is taken, and the units walk
// over every item's steps once, in order, an item's units one behind the other as the merge takes them.  *share_out: steps a
// unit, 0: equal shares; -1: not such a launch.
extern "C" int item_units_check(const int* n_new, const int* ctx, int seqs, int tq, int window_left, int units, float cut_cost,
                                int* share_out, char* msg, int msg_len) {
  std::vector<uint32_t> steps;
  uint32_t total = 0;
  for (int s = 0; s < seqs; ++s) {
    for (int j = 0; j < query_blocks(n_new[s], tq); ++j) {
      steps.push_back(static_cast<uint32_t>(block_tiles(n_new[s], ctx[s], j, tq, window_left).count()));
      total += steps.back();
    }
  }
  const int items = static_cast<int>(steps.size());
  *share_out = -1;
  if (items == 0 || items >= units) return 0;
  auto units_at = [&](uint32_t share) {
    uint32_t n = 0;
    for (uint32_t x : steps) n += (x + share - 1) / share;
    return n;
  };
  const float least = sqrtf(cut_cost * static_cast<float>(total) / static_cast<float>(items));
  const uint32_t share = share_of_items(total, static_cast<uint32_t>(items), static_cast<uint32_t>(units), least, units_at);
  uint32_t lo = (total + static_cast<uint32_t>(units) - 1) / static_cast<uint32_t>(units);
  while (lo < kMostLeastSteps && static_cast<float>(lo + 1) <= least) ++lo;
  *share_out = static_cast<int>(share);
  for (uint32_t x = lo; x < lo + kSegmentSteps; ++x) {  // the first of these that does, or none
    if (units_at(x) > static_cast<uint32_t>(units)) continue;
    if (share != x) {
      snprintf(msg, msg_len, "share %u, the least that does is %u", share, x);
      return 1;
    }
    break;
  }
  if (share == 0) {
    if (units_at(lo + kSegmentSteps - 1) > static_cast<uint32_t>(units)) return 0;
    snprintf(msg, msg_len, "equal shares, but %u steps a unit do", lo + kSegmentSteps - 1);
    return 1;
  }
  int item = 0, nth = 0;
  for (int u = 0; u < units; ++u) {
    const ItemUnit at = item_of_unit(u, items, [&](int i) { return static_cast<int>((steps[i] + share - 1) / share); });
    if (at.item != (item < items ? item : -1) || (item < items && at.nth != nth)) {
      snprintf(msg, msg_len, "unit %d: item %d, its unit %d, the walk is at item %d, unit %d", u, at.item, at.nth, item, nth);
      return 1;
    }
    if (item < items && ++nth * share >= steps[item]) ++item, nth = 0;
  }
  if (item < items) {
    snprintf(msg, msg_len, "item %d of %d has steps that no unit takes", item, items);
    return 1;
  }
  return 0;
}
