// Arguments shared by the backward kernels of the causal varlen / dense attention ops (attention_backward.hip: the
// vector-ALU kernels for every head dim and dtype; attention_backward_mfma.hip: matrix-core kernels for 16-bit
// inputs at head dims 64, 128, 192 and 256).
#pragma once

#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>

#include "areno_hip.h"
#include "backward_order.hpp"
#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#endif

namespace areno {

struct BwdParams {
  const void* grad_out;
  const void* q;
  const void* k;
  const void* v;
  const void* out;
  void* grad_q;  // gradients in fp32, or in the inputs' 16-bit type (grad_dtype)
  void* grad_k;
  void* grad_v;
  float* row_stats;  // [q_tokens * q_heads][2] (matrix cores: by head, then row): log2-domain log-sum-exp of the scaled scores, dO . O (matrix cores: -(dO . O))
  const int32_t* cu_q;
  const int32_t* cu_k;
  const int32_t* ctx;  // may be nullptr: 0
  BlockOrder q_order, k_order;  // matrix cores: of the dq kernel's blocks and of the dkv kernel's
  int64_t q_tokens;
  int64_t k_tokens;
  int32_t num_seqs;
  int32_t q_heads;
  int32_t kv_heads;
  int32_t window_left;
  int32_t head_dim;
  int32_t dtype;
  int32_t grad_dtype;  // ARENO_DT_F32, or `dtype` when that is a 16-bit type: the fp32 sums rounded once, at the store
  float scale;
  float scale_log2e;
};

#if defined(__HIPCC__)
// one gradient element in the type `grad_dtype` names
__device__ inline __attribute__((always_inline)) void store_grad(void* base, int64_t i, float x, int32_t grad_dtype) {
  if (grad_dtype == ARENO_DT_F32) {
    static_cast<float*>(base)[i] = x;
  } else if (grad_dtype == ARENO_DT_BF16) {
    static_cast<__bf16*>(base)[i] = static_cast<__bf16>(x);
  } else {
    static_cast<_Float16*>(base)[i] = static_cast<_Float16>(x);
  }
}
// Many of them: `body` gets a function that stores four consecutive elements (from a multiple of 4) in the type that
// `grad_dtype` names, fp32 or the inputs' T.  The type is asked for once.  Asked for at each store, 32 of a wave with 32 rows,
// it was a hundred jumps through code that a short block meets for the first time, and enough live values to spill up to 94
// registers.  Backward, us: 1 x 4 tokens, 6 / 6 heads of 128: 13.0 -> 10.7; 5 x 22, window 16: 23.9 -> 22.9; 4 x 600, 8 / 2 of 64:
// 44.0 -> 43.2; with the forward, 2 717 tokens in four sequences, 16 / 8 heads of 256, window 512: 255 -> 231.
template <typename T>
struct GradStore {
  __device__ inline __attribute__((always_inline)) void operator()(void* base, int64_t i, float a, float b, float c, float d) const {
    typedef __attribute__((ext_vector_type(4))) float f32x4;
    typedef __attribute__((ext_vector_type(4))) T t4;
    *reinterpret_cast<t4*>(static_cast<T*>(base) + i) = __builtin_convertvector((f32x4{a, b, c, d}), t4);
  }
};
template <typename T, typename Body>
__device__ inline __attribute__((always_inline)) void store_grads(int32_t grad_dtype, const Body& body) {
  if (grad_dtype == ARENO_DT_F32) {
    body(GradStore<float>{});
  } else {
    body(GradStore<T>{});
  }
}
// What a workgroup's start needs of the arguments, asked for at once: left alone the compiler asks for each part in front of its
// use, three round trips in a row (2.8 % of launches of 1 .. 3 sequences of up to 100 tokens).
__device__ inline __attribute__((always_inline)) void ask_for_arguments(const BwdParams& p, const BlockOrder& order) {
  asm volatile("" : : "s"(order.blocks), "s"(order.runs), "s"(order.per), "s"(order.step), "s"(order.before), "s"(p.q_heads), "s"(p.kv_heads),
               "s"(p.num_seqs), "s"(p.q_tokens), "s"(p.k_tokens), "s"(p.q), "s"(p.k), "s"(p.v), "s"(p.grad_out), "s"(p.out), "s"(p.cu_q), "s"(p.cu_k), "s"(p.ctx));
  __builtin_amdgcn_sched_barrier(0);
}
// The last sequence that starts at or in front of `row` (the one that holds it, when the row exists).  Every lane looks at one
// of 64 places, so up to 64 sequences take one round trip to memory where halving took one per bit of their number, with
// nothing else under way.  (All lanes of the wave take part; `row` is the same for them.)
__device__ inline __attribute__((always_inline)) int seq_of_row(const int32_t* cu, int num_seqs, int64_t row) {
  const int lane = static_cast<int>(threadIdx.x) & 63;
  int first = 0;
  for (int left = num_seqs; left > 1;) {  // among [first, first + left)
    const int apart = (left + 63) >> 6, at = lane * apart;
    const bool starts = at < left && static_cast<int64_t>(cu[first + at]) <= row;
    const int behind = (__builtin_popcountll(__builtin_amdgcn_ballot_w64(starts)) - 1) * apart;
    if (behind > 0) first += behind, left -= behind;
    left = left < apart ? left : apart;
  }
  return first;
}

// whether a switch has this value (read at every launch)
inline bool fixed_by(const char* name, const char* value) {
  const char* const e = getenv(name);
  return e != nullptr && strcmp(e, value) == 0;
}

// a kernel with its launch shape
typedef void (*bwd_fn)(BwdParams);
struct BwdLaunch {
  bwd_fn fn;  // nullptr: its LDS size was refused
  int lds_bytes, threads, rows;  // (rows of a block)
};
// the kernels on 32 x 32 x 16 products (attention_backward_dkv.hip), head dims 64 and 128, 16-bit types; `groups`: workgroups
// of a kv head
BwdLaunch dkv32_launch(const BwdParams& p, int64_t* groups);
// head dims 192 and 256 (attention_backward_wide.hip): the dkv kernel over blocks of 64 keys, or of 32 with its stream in two
// parts, by the blocks of 32 and the steps of their streams
int dkv32_wide_parts(const BwdParams& p);
BwdLaunch dq32_wide_launch(const BwdParams& p);
BwdLaunch dkv32_wide_launch(const BwdParams& p, int64_t* groups);
#endif

// Matrix-core backward (attention_backward_mfma.hip): launches both kernels on `stream` and returns ARENO_OK, or
// ARENO_ERR_UNSUPPORTED when the shape is not one it serves (the caller then takes the vector-ALU kernels).
int launch_attention_backward_mfma(const BwdParams& p, void* stream);

}  // namespace areno
