// CPU check of when a packed prefill launch may store the pages as well (areno_amd/csrc/page_write.hpp).  The
// tensors of a call lie one behind the other in an address range that nothing reads; then one of them after the other is
// moved so that it shares its last or its first byte with another.  Built by tests/test_page_write_cpu.py with g++.
#include <stdio.h>

#include <initializer_list>

#include "../../areno_amd/csrc/page_write.hpp"

namespace {
enum { CACHE_K, CACHE_V, SCALE_K, SCALE_V, Q, K, V, OUT, CU, IDS, OFFSETS, COUNT };
struct Call {
  int64_t at[COUNT], bytes[COUNT];
};
bool fits(const Call& c, int cache_dtype, int scale_dtype, int act, int head_dim) {
  auto p = [&](int i) { return reinterpret_cast<void*>(static_cast<uintptr_t>(c.at[i])); };
  areno_paged_cache cache = {};
  cache.k = p(CACHE_K), cache.v = p(CACHE_V);
  if (c.bytes[SCALE_K] > 0) cache.k_scale = p(SCALE_K), cache.v_scale = p(SCALE_V);
  cache.num_blocks = 6, cache.block_size = 16, cache.kv_heads = 2, cache.head_dim = head_dim;
  cache.cache_dtype = cache_dtype, cache.scale_dtype = scale_dtype;
  return areno::pages_fit(cache, p(Q), p(K), p(V), p(OUT), act, 80, 8, static_cast<int32_t*>(p(CU)), 3, static_cast<int64_t*>(p(IDS)),
                          static_cast<int64_t*>(p(OFFSETS)));
}
}  // namespace

extern "C" int page_write_check(int cache_dtype, int scale_dtype, int act, int head_dim, int element, int scale_element, char* msg, int msg_len) {
  const int64_t rows = 6 * 16 * 2, pool = rows * head_dim * element, scales = rows * scale_element, q = 80 * 8 * head_dim * 2,
                kv = 80 * 2 * head_dim * 2;
  Call c = {{}, {pool, pool, scales, scales, q, kv, kv, q, 16, 640, 640}};
  int64_t next = 1 << 20;
  for (int i = 0; i < COUNT; ++i) c.at[i] = next, next += c.bytes[i];  // (each ends where the next begins)
  if (!fits(c, cache_dtype, scale_dtype, act, head_dim)) {
    snprintf(msg, msg_len, "tensors side by side are refused");
    return 1;
  }
  for (int w = CACHE_K; w <= OUT; ++w) {
    if (w >= Q && w < OUT) continue;
    for (int r = Q; r < COUNT; ++r) {
      if (c.bytes[w] == 0 || r == w) continue;
      if (w == OUT && r != IDS && r != OFFSETS) continue;
      for (const int64_t at : {c.at[w] - c.bytes[r] + 1, c.at[w] + c.bytes[w] - 1, c.at[w] + c.bytes[w] / 2}) {
        Call moved = c;
        moved.at[r] = at;
        if (fits(moved, cache_dtype, scale_dtype, act, head_dim)) {
          snprintf(msg, msg_len, "tensor %d shares bytes with tensor %d", r, w);
          return 1;
        }
      }
    }
  }
  return 0;
}
