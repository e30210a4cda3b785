// CPU walk of block_in_launch_order (areno_amd/csrc/backward_order.hpp) over sequences of equal length that end anywhere in
// a block: every order is a permutation of the blocks; the first workgroups take the blocks with the sequences' most expensive
// rows, and none starts more than a block's rows of cost ahead of a later one.  Built by tests/test_backward_order_cpu.py.
#include <stdio.h>

#include <algorithm>
#include <vector>

#include "../../areno_amd/csrc/backward_order.hpp"

extern "C" int backward_launch_order_check(int rows, int max_length, int max_seqs, char* msg, int msg_len) {
  for (int length = 1; length <= max_length; ++length) {
    for (int seqs = 1; seqs <= max_seqs; ++seqs) {
      const int tokens = length * seqs, blocks = (tokens + rows - 1) / rows;
      for (int from_end = 0; from_end < 2; ++from_end) {
        std::vector<int> seen(blocks, 0), cost(blocks, 0);
        const areno::BlockOrder order = areno::block_order(tokens, rows, seqs);
        for (int i = 0; i < blocks; ++i) {
          const long long b = areno::block_in_launch_order(i, order, rows, from_end != 0);
          if (b < 0 || b >= blocks || seen[b]++) {
            snprintf(msg, msg_len, "%d x %d, rows %d, from_end %d: workgroup %d takes block %lld (outside or twice)", seqs, length, rows, from_end, i, b);
            return 1;
          }
          for (int row = b * rows; row < std::min<int>((b + 1) * rows, tokens); ++row)
            cost[i] = std::max(cost[i], from_end ? row % length + 1 : length - row % length);
        }
        if (length < 2 * rows) continue;  // (two blocks and fewer: no order)
        int most = 0;
        for (int i = blocks - 1; i >= 0; --i) {
          if (cost[i] + rows <= most) {
            snprintf(msg, msg_len, "%d x %d, rows %d, from_end %d: workgroup %d has cost %d, one behind it %d", seqs, length, rows, from_end, i, cost[i], most);
            return 1;
          }
          most = std::max(most, cost[i]);
          if (i < seqs && cost[i] != length) {
            snprintf(msg, msg_len, "%d x %d, rows %d, from_end %d: workgroup %d has cost %d", seqs, length, rows, from_end, i, cost[i]);
            return 1;
          }
        }
      }
    }
  }
  return 0;
}

// any tokens (of sequences of any lengths): a permutation
extern "C" int backward_launch_order_permutes(int rows, int max_tokens, int max_seqs, char* msg, int msg_len) {
  for (int tokens = 1; tokens <= max_tokens; ++tokens) {
    const int blocks = (tokens + rows - 1) / rows;
    for (int seqs = 0; seqs <= max_seqs; ++seqs) {
      for (int from_end = 0; from_end < 2; ++from_end) {
        std::vector<int> seen(blocks, 0);
        const areno::BlockOrder order = areno::block_order(tokens, rows, seqs);
        for (int i = 0; i < blocks; ++i) {
          const long long b = areno::block_in_launch_order(i, order, rows, from_end != 0);
          if (b < 0 || b >= blocks || seen[b]++) {
            snprintf(msg, msg_len, "%d tokens, %d sequences, rows %d, from_end %d: workgroup %d takes block %lld (outside or twice)", tokens, seqs, rows, from_end, i, b);
            return 1;
          }
        }
      }
    }
  }
  return 0;
}

// many sequences, whose fractions come near the limit of their 32 bits: a permutation as well
extern "C" int backward_launch_order_of_many(int rows, int seqs, int length, int last, char* msg, int msg_len) {
  const int tokens = length * (seqs - 1) + last, blocks = (tokens + rows - 1) / rows;
  const areno::BlockOrder order = areno::block_order(tokens, rows, seqs);
  for (int from_end = 0; from_end < 2; ++from_end) {
    std::vector<int> seen(blocks, 0);
    for (int i = 0; i < blocks; ++i) {
      const long long b = areno::block_in_launch_order(i, order, rows, from_end != 0);
      if (b < 0 || b >= blocks || seen[b]++) {
        snprintf(msg, msg_len, "%d x %d, rows %d, from_end %d: workgroup %d takes block %lld (outside or twice)", seqs, length, rows, from_end, i, b);
        return 1;
      }
    }
  }
  return 0;
}
