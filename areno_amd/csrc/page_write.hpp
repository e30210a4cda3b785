// The pages that a packed prefill launch also stores its tokens' K and V in (varlen_mfma.hip): the arguments of
// areno_hip_cache_write beside K and V themselves.
#pragma once

#include <stdint.h>

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

}  // namespace areno
