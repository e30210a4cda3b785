// The pages that a packed prefill launch also stores its tokens' K and V in (varlen_mfma.hip): the arguments of
// areno_hip_cache_write beside K and V themselves, and on the host whether one launch may do both.
#pragma once

#include <stdint.h>

#include "../../include/areno_hip.h"

namespace areno {

struct PageWrite {
  void* k;
  void* v;
  void* k_scale;  // (of an 8-bit cache)
  void* v_scale;
  const int64_t* block_ids;
  const int64_t* block_offsets;
  int64_t num_blocks;
  int32_t block_size;
  int32_t cache_dtype;
  int32_t scale_dtype;
};

struct MemoryRange {
  const void* at;
  int64_t bytes;  // (none: 0 or less)
};
inline bool ranges_meet(const MemoryRange& x, const MemoryRange& y) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(x.at), b = reinterpret_cast<uintptr_t>(y.at);
  return x.bytes > 0 && y.bytes > 0 && a < b + static_cast<uintptr_t>(y.bytes) && b < a + static_cast<uintptr_t>(x.bytes);
}

// Whether an attention launch over packed K / V can store them in the pages as areno_hip_cache_write would: that kernel's 16-byte
// rows, and memory that shows no order between the two.  Workgroups store pages while others still read the launch's inputs,
// and store the output, so neither the pages nor the output may lie where the launch reads, nor the one in the other.  (The output
// in q, k or v is for the attention alone to bear.)
inline bool pages_fit(const areno_paged_cache& c, const void* q, const void* k, const void* v, const void* out, int32_t dtype, int64_t tokens,
                      int32_t q_heads, const int32_t* cu_seqlens, int32_t num_seqs, const int64_t* block_ids, const int64_t* block_offsets) {
  const bool quantized = c.cache_dtype == ARENO_DT_I8 || c.cache_dtype == ARENO_DT_FP8_E4M3;
  if (dtype != ARENO_DT_F16 && dtype != ARENO_DT_BF16) return false;
  if (c.head_dim != 64 && c.head_dim != 128 && c.head_dim != 256 && (quantized || c.head_dim != 192)) return false;
  if (!quantized && c.cache_dtype != dtype) return false;
  if ((reinterpret_cast<uintptr_t>(c.k) | reinterpret_cast<uintptr_t>(c.v)) % 16 != 0) return false;
  const int64_t rows = c.num_blocks * c.block_size * c.kv_heads;
  const int64_t pool = rows * c.head_dim * (quantized ? 1 : 2), scales = quantized ? rows * (c.scale_dtype == ARENO_DT_F16 ? 2 : 4) : 0;
  const int64_t q_bytes = tokens * q_heads * c.head_dim * 2, kv_bytes = tokens * c.kv_heads * c.head_dim * 2;
  const MemoryRange output = {out, q_bytes};
  const MemoryRange written[] = {{c.k, pool}, {c.v, pool}, {c.k_scale, scales}, {c.v_scale, scales}};
  const MemoryRange tensors[] = {{q, q_bytes}, {k, kv_bytes}, {v, kv_bytes}, output};
  const MemoryRange indices[] = {{cu_seqlens, (int64_t{num_seqs} + 1) * 4}, {block_ids, tokens * 8}, {block_offsets, tokens * 8}};
  for (const MemoryRange& w : written) {
    for (const MemoryRange& r : tensors) {
      if (ranges_meet(w, r)) return false;
    }
    for (const MemoryRange& r : indices) {
      if (ranges_meet(w, r)) return false;
    }
  }
  return !ranges_meet(output, indices[1]) && !ranges_meet(output, indices[2]);
}

}  // namespace areno
