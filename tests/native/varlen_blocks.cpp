// CPU walk of the block order of the packed forward (areno_amd/csrc/varlen_blocks.hpp): for packs of sequences the
// workgroups take every query block once, longest place first, and those behind the last block take none.  Built by
// tests/test_varlen_blocks_cpu.py with g++.
#include <stdio.h>

#include <vector>

#include "../../areno_amd/csrc/varlen_blocks.hpp"

extern "C" int varlen_blocks_check(const int* lens, int num_seqs, int block, char* msg, int msg_len) {
  const areno::BlockDivision div = areno::block_division(block);
  std::vector<int> nb(num_seqs);
  int most = 0, all = 0, tokens = 0;
  for (int s = 0; s < num_seqs; ++s) {
    nb[s] = div(lens[s] + block - 1);
    if (nb[s] != (lens[s] + block - 1) / block) {
      snprintf(msg, msg_len, "%d tokens in blocks of %d: %d", lens[s], block, nb[s]);
      return 1;
    }
    most = nb[s] > most ? nb[s] : most;
    all += nb[s];
    tokens += lens[s];
  }
  auto behind = [&](int j) {
    int n = 0;
    for (int x : nb) n += x > j ? x - j : 0;
    return n;
  };
  std::vector<std::vector<int>> seen(num_seqs);
  for (int s = 0; s < num_seqs; ++s) seen[s].assign(nb[s], 0);
  int last = most;
  const int grid = tokens / block + num_seqs + 1;
  if (grid <= all) {
    snprintf(msg, msg_len, "grid of %d for %d blocks", grid, all);
    return 1;
  }
  for (int i = 0; i < grid; ++i) {
    areno::BlockPlace at;
    const bool found = areno::block_place(i, most, behind, at);
    if (found != (i < all) || (!found && at.nth != i - all)) {
      snprintf(msg, msg_len, "workgroup %d of %d blocks: found %d", i, all, found);
      return 1;
    }
    if (!found) continue;
    int seq = -1, nth = at.nth;
    for (int s = 0; s < num_seqs && seq < 0; ++s) {
      if (nb[s] > at.j && nth-- == 0) seq = s;
    }
    if (seq < 0 || at.j > last || seen[seq][at.j]++) {
      snprintf(msg, msg_len, "workgroup %d takes block %d of sequence %d (outside, twice or out of order)", i, at.j, seq);
      return 1;
    }
    last = at.j;
  }
  return 0;
}

extern "C" int varlen_block_division_check(int block, int n) { return areno::block_division(block)(n) == n / block ? 0 : 1; }
