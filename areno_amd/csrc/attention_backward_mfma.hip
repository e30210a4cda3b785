// Backward of the causal varlen / dense attention ops on the matrix cores (gfx950): 16-bit inputs, head dims 64,
// 128, 192 and 256.  Same contract as the vector-ALU kernels of attention_backward.hip (fp32 dQ, dK, dV from dO, Q, K, V and the
// saved output; areno/accel/csrc/attention.cu:244-524 in the reference), same two launches, no atomics:
//
//   dq kernel    (head dims 64 and 128 here) a workgroup owns 64 or 128 packed query rows of one q head (four waves of 16 or
//                32 rows) and streams the keys its rows may see in tiles of 32 through LDS.  Per tile, with the keys as the
//                rows of the products (the layout of the forward kernel):  S^T = K . Q^T  and  dP^T = V . dO^T,
//                the online softmax of the forward on S^T, dS^T = P^T * (dP^T - dO . O), and
//                dQ^T += K^T . dS^T  with the lane's own dS^T values as the B operand (rounded to the inputs' type) and K^T
//                read transposed from the same LDS tile.  A row's softmax reference moves as in the forward (the
//                accumulator is rescaled), so one pass over the keys gives dQ, the row's log-sum-exp and dO . O (left in
//                the workspace).
//   dkv kernel   (attention_backward_dkv.hip) a workgroup owns packed key rows of one kv head and streams, for every q head
//                of the group, the query rows that may see them:  S = Q . K^T,  dP = dO . V^T,  P = exp2(S - lse),
//                dS = P * (dP - dO . O),  dV^T += dO^T . P  and  dK^T += Q^T . dS.  Every gradient element has one owner.
// Head dims 192 and 256 have both kernels in attention_backward_wide.hip.
// Both launches take their blocks in an order that lets their workgroups end together: see block_in_launch_order.
//
// The streamed index of a tile (keys in the dq kernel, queries in the dkv kernel) is the contraction index of the
// second pair of products; a 16 x 16 product leaves element 4 g + j of that index in lane group g, which is exactly
// how the next product wants its B operand, and the A operand comes from the LDS tile through transposing reads
// (ds_read_b64_tr_b16), so nothing is shuffled between the products.
// Geometry as in attention_backward.hip: sequence s has queries [cu_q[s], cu_q[s+1]) at positions ctx[s] + i and keys
// [cu_k[s], cu_k[s+1]) at positions 0 ..; a query at position t sees keys max(0, t - window) .. t.  A block of
// packed rows may hold rows of several sequences; it goes through them one after the other, the rows of the others
// masked.

#include <algorithm>

#include "attention_backward.hpp"
#include "decode_mfma_kernels.hpp"
#include "mfma32_tiles.hpp"

namespace areno {
namespace {

constexpr int kBmWaves = 4;
constexpr int kBmThreads = kBmWaves * kWave;
constexpr int kBmRows = 16 * kBmWaves;  // packed rows a workgroup owns
constexpr int kBmTile = 32;             // streamed rows per step
constexpr float kBmNegInf = -__builtin_huge_valf();

// A tile of 32 rows x D 16-bit elements in LDS, row stride D * 2 + 16 bytes: the row operands (16 lanes read the same
// 16-byte chunk of 16 rows) meet every bank once, the transposed ones (32 lanes read 32 bytes of 8 consecutive rows)
// meet every bank twice.  (A layout without any bank conflict -- rows back to back, the chunks of a row permuted by
// a function of the row -- was measured, with four and with eight waves on a compute unit's LDS: LDS is busy 40 %
// less with it and no launch got faster, small ones 3-8 % slower from the address registers it takes.)  Staging: every thread moves kChunks 16-byte chunks of a tensor
// through registers.
template <int D>
struct BmTile {
  static constexpr int RS = D * 2 + 16;
  static constexpr int kChunksPerRow = D * 2 / 16;
  static constexpr int kChunks = kBmTile * kChunksPerRow / kBmThreads;  // per thread: 1 (D = 64) or 2 (D = 128)
  static_assert(kBmTile * kChunksPerRow % kBmThreads == 0, "tile chunks");
  static __device__ __forceinline__ int chunk_pos(int r, int c) { return r * RS + (c << 4); }
};

// Operand reads.  Row operand (A of the first pair of products): row 16 tg + lr of the tile, elements
// (D / 4) lk + 8 sl .. + 8 -- the same split of the head over the four lane groups as the register operands.
template <int KIND, typename T, int D>
__device__ __forceinline__ typename MfmaOps<KIND>::vec8 tile_row_operand(const char* tile, int tg, int sl, int lr, int lk) {
  using V8 = typename MfmaOps<KIND>::vec8;
  return *reinterpret_cast<const V8*>(tile + T::chunk_pos(16 * tg + lr, (D / 32) * lk + sl));
}
// Transposed operand (A of the second pair): head elements 16 nb + lr as rows, the tile's 32 rows as the contraction
// index in the order lane group lk holds them after the first pair (rows 4 lk .. 4 lk + 3, then 16 + 4 lk .. + 3).
template <int KIND, typename T>
__device__ __forceinline__ typename MfmaOps<KIND>::vec8 tile_transposed_operand(char* tile, int nb, int lr, int lk) {
  using V8 = typename MfmaOps<KIND>::vec8;
  uint32_t w[4];
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    const int row = 16 * half + 4 * lk + (lr >> 2);
    char* a = tile + T::chunk_pos(row, 2 * nb + ((lr & 3) >> 1)) + 8 * (lr & 1);
    const short4_t r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)a);
    const uint2_t u = __builtin_bit_cast(uint2_t, r);
    w[2 * half] = u[0];
    w[2 * half + 1] = u[1];
  }
  return __builtin_bit_cast(V8, uint4_t{w[0], w[1], w[2], w[3]});
}
// eight values of the streamed index, as a lane holds them after the first pair of products ([tg][j]), as B operand
template <int KIND>
__device__ __forceinline__ typename MfmaOps<KIND>::vec8 streamed_operand(const float (&x)[2][4]) {
  using V8 = typename MfmaOps<KIND>::vec8;
  return __builtin_bit_cast(V8, uint4_t{pack_pair<KIND>(x[0][0], x[0][1]), pack_pair<KIND>(x[0][2], x[0][3]),
                                        pack_pair<KIND>(x[1][0], x[1][1]), pack_pair<KIND>(x[1][2], x[1][3])});
}

// ---- dQ (and the rows' statistics) ------------------------------------------------------------------------------------
// Bound by what a wave issues and waits for between its products, so a tile has one barrier (two LDS buffers), a
// row's softmax reference mostly stays where it is (no lane swaps, no rescaling), and dP - dO . O comes out of the
// product, which starts at -(dO . O); the dkv kernel's does too (forward and backward of 2 x 2 048 tokens, 28 / 4 heads of
// 128, bf16: 435 -> 427 us).  Short sequences are mostly a block's start: its sequence is found in one round trip, the first
// tile is on its way together with Q.  In a step the operands are read ahead of their products and the exponentials go
// between the products of dP.  Forward and backward, us, before and with these: 16 x 20 .. 600 tokens, 16 heads of 64, fp16: 83.6,
// 80.8; 12 x 100 .. 900, 32 / 8 heads of 64, bf16: 134.7, 131.1 (137 with three waves per SIMD, hence the bound of four); 6 x 60 ..
// 450, 28 / 4 heads of 128, fp16: 90.0, 86.9.
template <int KIND, int D>
__global__ __launch_bounds__(kBmThreads, D == 64 ? 4 : 2) void bwd_mfma_dq_kernel(BwdParams p) {
  using Ops = MfmaOps<KIND>;
  using V8 = typename Ops::vec8;
  using T = BmTile<D>;
  constexpr int NS = D / 32, NB = D / 16;
  constexpr int kRows = kBmRows;  // packed rows of the workgroup
  constexpr int kWaveRows = 16;
  __shared__ __attribute__((aligned(16))) char k_lds[2 * kBmTile * T::RS];
  __shared__ __attribute__((aligned(16))) char v_lds[2 * kBmTile * T::RS];

  ask_for_arguments(p, p.q_order);
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = uniform(tid >> 6);  // (in a scalar register: what follows from it is scalar work and scalar branches)
  const int lr = lane & 15, lk = lane >> 4;
  // workgroups in launch order: the heads of a block next to each other, the blocks by cost
  const int h = static_cast<int>(blockIdx.x % static_cast<unsigned>(p.q_heads));
  const int kvh = h / (p.q_heads / p.kv_heads);
  const int64_t r0 = int64_t{block_in_launch_order(static_cast<int>(blockIdx.x / static_cast<unsigned>(p.q_heads)), p.q_order, kRows, true)} * kRows;
  const int64_t block_end = r0 + kRows < p.q_tokens ? r0 + kRows : p.q_tokens;
  const int64_t wave_row0 = r0 + kWaveRows * wave;
  int64_t row;  // this lane's query rows (columns of the products)
  row = wave_row0 + lr;

  int covered = 0;  // (where the sequences seen so far end)
  int s = uniform(seq_of_row(p.cu_q, p.num_seqs, r0));
  for (int64_t sq0 = uniform(p.cu_q[s]), sq1; s < p.num_seqs && sq0 < block_end; ++s, sq0 = sq1) {
    // (asked for together)
    const int q_end = p.cu_q[s + 1], k_begin = p.cu_k[s], k_end = p.cu_k[s + 1], before = p.ctx != nullptr ? p.ctx[s] : 0;
    sq1 = covered = uniform(q_end);
    const int64_t q_lo = sq0 > r0 ? sq0 : r0, q_hi = sq1 < block_end ? sq1 : block_end;
    if (q_lo >= q_hi) continue;
    const int ctx = uniform(before);
    const int64_t k_base = uniform(k_begin);
    const int n_k = uniform(k_end) - static_cast<int>(k_base);
    const bool live = row >= q_lo && row < q_hi;
    const int pos = live ? ctx + static_cast<int>(row - sq0) : -1;
    const uint64_t live_lanes = __builtin_amdgcn_ballot_w64(live);
    const bool wave_live = live_lanes != 0, wave_full = live_lanes == ~0ull;
    // (the positions of the wave's query rows, when all of them belong to this sequence)
    const int wave_pos_lo = ctx + static_cast<int>(wave_row0 - sq0), wave_pos_hi = wave_pos_lo + kWaveRows - 1;
    const int pos_min = ctx + static_cast<int>(q_lo - sq0), pos_max = ctx + static_cast<int>(q_hi - 1 - sq0);
    const int key_lo = p.window_left >= 0 ? (pos_min - p.window_left > 0 ? pos_min - p.window_left : 0) : 0;
    const int key_hi = pos_max < n_k - 1 ? pos_max : n_k - 1;

    const int t0 = key_lo / kBmTile, t1 = key_hi / kBmTile;
    uint4_t kreg[T::kChunks], vreg[T::kChunks];
    auto fetch = [&](int t) {
#pragma unroll
      for (int i = 0; i < T::kChunks; ++i) {
        const int c = tid + kBmThreads * i;
        const int r = c / T::kChunksPerRow, col = c % T::kChunksPerRow;
        const int key = kBmTile * t + r < n_k ? kBmTile * t + r : n_k - 1;  // rows past the end repeat the last key
        const int64_t off = ((k_base + key) * p.kv_heads + kvh) * (D * 2) + col * 16;
        kreg[i] = load16(p.k, off);
        vreg[i] = load16(p.v, off);
      }
    };
    // this lane's parts of its rows of Q and dO (B operands), and dO . O; the first tile is asked for behind them, so that
    // both are on their way together
    const int64_t row_elem = (row * p.q_heads + h) * D;
    V8 qop[NS], gop[NS];
    float4_t acc[NB];
    float m_run = kBmNegInf, l_lane = 0.0f, d = 0.0f;
    {
      uint4_t qw[NS], gw[NS], ow[NS];
#pragma unroll
      for (int sl = 0; sl < NS; ++sl) qw[sl] = gw[sl] = ow[sl] = uint4_t{0u, 0u, 0u, 0u};
      if (live) {
#pragma unroll
        for (int sl = 0; sl < NS; ++sl) {
          const int64_t off = (row_elem + (D / 4) * lk + 8 * sl) * 2;
          qw[sl] = load16(p.q, off);
          gw[sl] = load16(p.grad_out, off);
          ow[sl] = load16(p.out, off);
        }
      }
      if (key_hi >= key_lo) fetch(t0);
#pragma unroll
      for (int sl = 0; sl < NS; ++sl) {
        qop[sl] = __builtin_bit_cast(V8, qw[sl]);
        gop[sl] = __builtin_bit_cast(V8, gw[sl]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          d += operand_element<KIND>(gw[sl][j], 0) * operand_element<KIND>(ow[sl][j], 0) +
               operand_element<KIND>(gw[sl][j], 1) * operand_element<KIND>(ow[sl][j], 1);
        }
      }
    }
    const float delta = rows_sum(d);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

    if (key_hi >= key_lo) {  // (the same for the whole workgroup)
      auto publish = [&](int buf) {
#pragma unroll
        for (int i = 0; i < T::kChunks; ++i) {
          const int c = tid + kBmThreads * i;
          const int r = c / T::kChunksPerRow, col = c % T::kChunksPerRow;
          *reinterpret_cast<uint4_t*>(k_lds + buf * (kBmTile * T::RS) + T::chunk_pos(r, col)) = kreg[i];
          *reinterpret_cast<uint4_t*>(v_lds + buf * (kBmTile * T::RS) + T::chunk_pos(r, col)) = vreg[i];
        }
      };
      auto step = [&](int t, int buf) {
        char* const s_k = k_lds + buf * (kBmTile * T::RS);
        char* const s_v = v_lds + buf * (kBmTile * T::RS);
        if (t < t1) fetch(t + 1);
        if (wave_live) {
          // the products' operands in one stream, each read kAhead products in front of its own: rows of K and of V (the
          // two groups of 16 in turn, so that a product does not wait for the one before), columns of K
          constexpr int kAhead = 4, kRowReads = 2 * NS, kReads = 2 * kRowReads + NB;
          auto read = [&](int x) {
            if (x < kRowReads) return tile_row_operand<KIND, T, D>(s_k, x & 1, x >> 1, lr, lk);
            if (x < 2 * kRowReads) return tile_row_operand<KIND, T, D>(s_v, x & 1, (x - kRowReads) >> 1, lr, lk);
            return tile_transposed_operand<KIND, T>(s_k, x - 2 * kRowReads, lr, lk);
          };
          V8 operand[kAhead];
#pragma unroll
          for (int x = 0; x < kAhead; ++x) operand[x] = read(x);
          float4_t sc[2] = {}, dp[2];
#pragma unroll
          for (int x = 0; x < kRowReads; ++x) {
            __builtin_amdgcn_sched_barrier(0);
            sc[x & 1] = Ops::mfma(operand[x % kAhead], qop[x >> 1], sc[x & 1]);
            operand[x % kAhead] = read(x + kAhead);
          }
          // most tiles lie below the diagonal and inside the window as a whole: every query row of this wave sees
          // every key of the tile, and nothing needs a mask
          const int key_first = kBmTile * t, key_last = key_first + kBmTile - 1;
          const bool plain = wave_full && key_last < n_k && key_last <= wave_pos_lo &&
                             (p.window_left < 0 || key_first >= wave_pos_hi - p.window_left);
          if (!plain) {
            const int base = key_first + 4 * lk;  // keys base + 16 tg + j
            const int last = min(pos, n_k - 1) - base, first = p.window_left < 0 ? -base : pos - p.window_left - base;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const int key = 16 * (e >> 2) + (e & 3);
              sc[e >> 2][e & 3] = key >= first && key <= last ? sc[e >> 2][e & 3] : kBmNegInf;
            }
          }
          // The reference of a row is raised only when a score of the wave exceeds its row's by more than 2^kLazy: most
          // tiles then take no lane swaps and no rescaling.  bf16 has room for probabilities up to 2^8 in dS; fp16 may
          // not (dS is packed with them), so there the reference follows every new maximum as it is.
          constexpr float kLazy = KIND == KV_BF16 ? 8.0f : 0.0f;
          float mt = max3_f32(sc[0][0], sc[0][1], sc[0][2]);
          mt = max3_f32(mt, sc[0][3], sc[1][0]);
          mt = max3_f32(mt, sc[1][1], sc[1][2]);
          mt = max_f32(mt, sc[1][3]);
          if (__builtin_amdgcn_ballot_w64(mt * p.scale_log2e > m_run + kLazy) != 0) {
            const float m_new = max_f32(m_run, rows_max(mt) * p.scale_log2e);  // (the scale is positive)
            const float m_ref = m_new == kBmNegInf ? 0.0f : m_new;
            const float alpha = settled(fast_exp2(m_run - m_ref));  // 0 while the row has seen no key
            m_run = m_new;
            scale_in_place(l_lane, alpha);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                float x = acc[nb][j];
                scale_in_place(x, alpha);
                acc[nb][j] = x;
              }
            }
          }
          const float m_ref = m_run == kBmNegInf ? 0.0f : m_run;
          dp[0] = dp[1] = float4_t{-delta, -delta, -delta, -delta};  // dP comes out less dO . O
#pragma unroll
          for (int x = 0; x < kRowReads; ++x) {
            __builtin_amdgcn_sched_barrier(0);
            dp[x & 1] = Ops::mfma(operand[(kRowReads + x) % kAhead], gop[x >> 1], dp[x & 1]);
            operand[(kRowReads + x) % kAhead] = read(kRowReads + x + kAhead);
            // the exponentials between the products of dP (exp2(-inf) = 0: masked keys)
#pragma unroll
            for (int e = 8 / kRowReads * x; e < 8 / kRowReads * (x + 1); ++e) {
              const float pe = fast_exp2(__builtin_fmaf(sc[e >> 2][e & 3], p.scale_log2e, -m_ref));
              sc[e >> 2][e & 3] = pe;
              l_lane += pe;
            }
          }
          __builtin_amdgcn_sched_barrier(0);
          float ds[2][4];
#pragma unroll
          for (int e = 0; e < 8; ++e) ds[e >> 2][e & 3] = sc[e >> 2][e & 3] * dp[e >> 2][e & 3];
          const V8 dsop = streamed_operand<KIND>(ds);
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            const int x = 2 * kRowReads + nb;
            __builtin_amdgcn_sched_barrier(0);
            acc[nb] = Ops::mfma(operand[x % kAhead], dsop, acc[nb]);
            if (x + kAhead < kReads) operand[x % kAhead] = read(x + kAhead);
          }
        }
        // (tile t - 1, which lay where t + 1 goes, was read in front of the last barrier)
        if (t < t1) publish(buf ^ 1);
        __syncthreads();
      };
      __syncthreads();  // the tiles' previous readers (an earlier sequence of this block) are done
      publish(0);
      __syncthreads();
      for (int t = t0; t <= t1; t += 2) {
        step(t, 0);
        if (t + 1 <= t1) step(t + 1, 1);
      }
    }

    // dQ = scale / l * sum_k p_k (dP_k - dO . O) K_k; the row's log-sum-exp (log2 domain) and -(dO . O) for the dkv kernel
    const float l_tot = rows_sum(l_lane);
    const float f = l_tot > 0.0f ? p.scale / l_tot : 0.0f;
    const int l = lane_now(), lr_ = l & 15, lk_ = l >> 4;  // (worked out anew: kept, they would cost the loop registers)
    const int64_t at = wave_row0 + lr_;
    if (p.grad_dtype != ARENO_DT_F32) {  // as whole rows, through the tiles' LDS: they are read
      using Stage = RowStage<2 * NB>;
      char* const stage = k_lds + wave * (kWaveRows * Stage::kRowBytes);
      static_assert(kBmWaves * kWaveRows * Stage::kRowBytes <= sizeof(k_lds), "the rows' place");
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        Stage::put(stage, lr_, 2 * nb + (lk_ >> 1), lk_ & 1, pack_pair<KIND>(acc[nb][0] * f, acc[nb][1] * f), pack_pair<KIND>(acc[nb][2] * f, acc[nb][3] * f));
      Stage::template take<kWaveRows>(stage, l, [&](int r, int chunk, uint4_t w) {
        const int64_t to = wave_row0 + r;
        if (to >= q_lo && to < q_hi) *reinterpret_cast<uint4_t*>(static_cast<char*>(p.grad_q) + ((to * p.q_heads + h) * D + 8 * chunk) * 2) = w;
      });
    }
    if (at >= q_lo && at < q_hi) {
      if (p.grad_dtype == ARENO_DT_F32) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          GradStore<float>{}(p.grad_q, (at * p.q_heads + h) * D + 4 * lk_ + 16 * nb, acc[nb][0] * f, acc[nb][1] * f, acc[nb][2] * f, acc[nb][3] * f);
      }
      if (lk_ == 0) {
        float* st = p.row_stats + (h * p.q_tokens + at) * 2;
        // a row without visible keys gets a reference no score reaches: its probabilities come out as zeros
        st[0] = l_tot > 0.0f ? m_run + __builtin_log2f(l_tot) : __builtin_huge_valf();
        st[1] = -delta;
      }
    }
  }
  row = wave_row0 + (lane_now() & 15);
  if (row >= covered && row < p.q_tokens) {  // behind the last sequence, the end of a padded pack
    const int64_t row_elem = (row * p.q_heads + h) * D + 4 * (lane_now() >> 4);
    store_grads<typename Mfma32<KIND>::elem>(p.grad_dtype, [&](auto store) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) store(p.grad_q, row_elem + 16 * nb, 0.0f, 0.0f, 0.0f, 0.0f);
    });
  }
}

// The same with 32 query rows per wave, 128 per workgroup, on 32 x 32 x 16 products, for long sequences: an operand read
// from LDS serves a product of twice the size, the K and V tiles are fetched straight into LDS (mfma32_tiles.hpp), an
// operand is read four products in front of its own and the exponentials go between the products of dP.  Bound by the
// matrix cores (busy 53 % of the cycles, at the clock that they then leave, 1.7 GHz) and the vector ALU.  Forward and
// backward of 4 x 4 096 tokens, 32 / 8 heads of 128, bf16: 2 429 -> 2 375 us with the operands read ahead.  (Registers spill
// at head dim 128 once per sequence of a block, not in the tile loop.)
template <int KIND, int D>
__global__ __launch_bounds__(kBmThreads, 2) void bwd_mfma32_dq_kernel(BwdParams p) {
  using M = Mfma32<KIND>;
  using V8 = typename M::vec8;
  using T = LdsTile<D, kBmTile, kBmWaves>;
  constexpr int NKS = D / 16, NB = D / 32, NF = T::kFetches;
  constexpr int kRows = 32 * kBmWaves;
  constexpr int kBuffer = 2 * T::kBytes;  // K, V
  __shared__ __attribute__((aligned(1024))) char lds[2 * kBuffer];

  ask_for_arguments(p, p.q_order);
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = uniform(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int h = static_cast<int>(blockIdx.x % static_cast<unsigned>(p.q_heads));
  const int kvh = h / (p.q_heads / p.kv_heads);
  const int block = uniform(block_in_launch_order(static_cast<int>(blockIdx.x / static_cast<unsigned>(p.q_heads)), p.q_order, kRows, true));
  const int64_t r0 = static_cast<int64_t>(block) * kRows;
  const int64_t block_end = r0 + kRows < p.q_tokens ? r0 + kRows : p.q_tokens;
  const int64_t wave_row0 = r0 + 32 * wave;
  const int64_t row = wave_row0 + l32;  // this lane's query row (a column of the products)
  const uint32_t at_rows = T::rows_base(l32, half), at_columns = T::columns_base(lane);
  const uint32_t lds0 = lds_address(lds);
  const uint32_t stride = static_cast<uint32_t>(p.kv_heads) * (D * 2);
  int fetch_row[NF];
  uint32_t fetch_chunk[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int slot = (wave * NF + f) * 64 + lane;
    fetch_row[f] = slot / T::kChunksPerRow;
    fetch_chunk[f] = static_cast<uint32_t>((slot % T::kChunksPerRow) ^ T::twist(fetch_row[f])) * 16u;
  }

  int covered = 0;  // (where the sequences seen so far end)
  for (int s = uniform(seq_of_row(p.cu_q, p.num_seqs, r0)); s < p.num_seqs; ++s) {
    const int64_t sq0 = uniform(p.cu_q[s]), sq1 = covered = uniform(p.cu_q[s + 1]);
    if (sq0 >= block_end) break;
    const int64_t q_lo = sq0 > r0 ? sq0 : r0, q_hi = sq1 < block_end ? sq1 : block_end;
    if (q_lo >= q_hi) continue;
    const int ctx = p.ctx != nullptr ? uniform(p.ctx[s]) : 0;
    const int64_t k_first = uniform(p.cu_k[s]);
    const int n_k = uniform(p.cu_k[s + 1]) - static_cast<int>(k_first);
    const bool live = row >= q_lo && row < q_hi;
    const int pos = live ? ctx + static_cast<int>(row - sq0) : -1;
    const uint64_t live_lanes = __builtin_amdgcn_ballot_w64(live);
    const bool wave_live = live_lanes != 0, wave_full = live_lanes == ~0ull;
    const int wave_pos_lo = ctx + static_cast<int>(wave_row0 - sq0), wave_pos_hi = wave_pos_lo + 31;
    const int pos_min = ctx + static_cast<int>(q_lo - sq0), pos_max = ctx + static_cast<int>(q_hi - 1 - sq0);
    const int key_lo = p.window_left >= 0 ? (pos_min - p.window_left > 0 ? pos_min - p.window_left : 0) : 0;
    const int key_hi = pos_max < n_k - 1 ? pos_max : n_k - 1;

    // this lane's parts of its row of Q and dO (B operands), and dO . O
    const int64_t row_elem = (row * p.q_heads + h) * D;
    V8 qop[NKS], gop[NKS];
    float delta = 0.0f;
    uint4_t qw[NKS], gw[NKS], ow[NKS];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qw[ks] = gw[ks] = ow[ks] = uint4_t{0u, 0u, 0u, 0u};
    if (live) {
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const int64_t off = (row_elem + 16 * ks + 8 * half) * 2;
        qw[ks] = load16(p.q, off);
        gw[ks] = load16(p.grad_out, off);
        ow[ks] = load16(p.out, off);
      }
    }
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      // (waited for here: left to their first use inside the loop, that wait would cover every tile's fetches as well)
      asm volatile("" : "+v"(qw[ks]), "+v"(gw[ks]));
      qop[ks] = __builtin_bit_cast(V8, qw[ks]);
      gop[ks] = __builtin_bit_cast(V8, gw[ks]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        delta += operand_element<KIND>(gw[ks][j], 0) * operand_element<KIND>(ow[ks][j], 0) +
                 operand_element<KIND>(gw[ks][j], 1) * operand_element<KIND>(ow[ks][j], 1);
      }
    }
    auto both_halves = [](float x, auto op) {
      uint32_t a = __builtin_bit_cast(uint32_t, x), b = a;
      swap_rows32(a, b);
      return op(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
    };
    auto sum = [](float a, float b) { return a + b; };
    delta = both_halves(delta, sum);
    float16_t acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = zero16();
    float m_run = kBmNegInf, l_lane = 0.0f;

    if (key_hi >= key_lo) {  // (the same for the whole workgroup)
      const int t0 = key_lo / kBmTile, t1 = key_hi / kBmTile;
      const int64_t head_base = (k_first * p.kv_heads + kvh) * (D * 2);
      auto fetch = [&](int t, int buf) {
        const int rows = n_k - t * kBmTile;  // rows of the tile that exist; the ones behind repeat the last
        const int64_t tile_base = head_base + static_cast<int64_t>(t) * kBmTile * stride;
        const char* kb = static_cast<const char*>(p.k) + tile_base;
        const char* vb = static_cast<const char*>(p.v) + tile_base;
        const uint32_t dst = lds0 + static_cast<uint32_t>(buf * kBuffer + wave * (NF * 1024));
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          const uint32_t off = static_cast<uint32_t>(min(fetch_row[f], rows - 1)) * stride + fetch_chunk[f];
          fetch_to_lds(kb, off, dst + f * 1024);
          fetch_to_lds(vb, off, dst + T::kBytes + f * 1024);
        }
      };
      auto step = [&](int t, int buf) {
        fetched_barrier();  // tile t (asked for a step ago) is there, and every wave has left tile t - 1
        if (t < t1) fetch(t + 1, buf ^ 1);
        if (!wave_live) return;
        const int key_first = kBmTile * t, key_last = key_first + kBmTile - 1;
        if (wave_full && key_first > wave_pos_hi) return;
        char* const k_lds = lds + buf * kBuffer;
        char* const v_lds = k_lds + T::kBytes;
        // the products' operands in one stream, each read kAhead products in front of its own (as in the dkv kernel):
        // rows of K and of V, columns of K
        auto read = [&](int x) {
          if (x < NKS) return tile_rows<KIND, T>(k_lds, at_rows, 0, x);
          if (x < 2 * NKS) return tile_rows<KIND, T>(v_lds, at_rows, 0, x - NKS);
          return tile_columns<KIND, T>(k_lds, at_columns, 16 * ((x - 2 * NKS) / NB), (x - 2 * NKS) % NB);
        };
        constexpr int kAhead = 4, kReads = 2 * NKS + 2 * NB;
        V8 operand[kAhead];
#pragma unroll
        for (int x = 0; x < kAhead; ++x) operand[x] = read(x);
        float16_t sc = zero16(), dp;
#pragma unroll
        for (int x = 0; x < NKS; ++x) {
          __builtin_amdgcn_sched_barrier(0);
          sc = M::mfma(operand[x % kAhead], qop[x], sc);
          operand[x % kAhead] = read(x + kAhead);
        }
        const bool plain = wave_full && key_last < n_k && key_last <= wave_pos_lo &&
                           (p.window_left < 0 || key_first >= wave_pos_hi - p.window_left);
        if (!plain) {
          const int base = key_first + 4 * half;  // keys base + 8 c + j
          const int last = min(pos, n_k - 1) - base, first = p.window_left < 0 ? -base : pos - p.window_left - base;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int key = 8 * (i >> 2) + (i & 3);
            sc[i] = key >= first && key <= last ? sc[i] : kBmNegInf;
          }
        }
        constexpr float kLazy = KIND == KV_BF16 ? 8.0f : 0.0f;  // (as above)
        float mt = sc[0];
#pragma unroll
        for (int i = 1; i < 15; i += 2) mt = max3_f32(mt, sc[i], sc[i + 1]);
        mt = max_f32(mt, sc[15]);
        if (__builtin_amdgcn_ballot_w64(mt * p.scale_log2e > m_run + kLazy) != 0) {
          mt = both_halves(mt, [](float a, float b) { return max_f32(a, b); });
          const float m_new = max_f32(m_run, mt * p.scale_log2e);  // (the scale is positive)
          const float m_ref = m_new == kBmNegInf ? 0.0f : m_new;
          const float alpha = settled(fast_exp2(m_run - m_ref));  // 0 while the row has seen no key
          m_run = m_new;
          scale_in_place(l_lane, alpha);
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              float x = acc[nb][i];
              scale_in_place(x, alpha);
              acc[nb][i] = x;
            }
          }
        }
        const float m_ref = m_run == kBmNegInf ? 0.0f : m_run;
#pragma unroll
        for (int i = 0; i < 16; ++i) dp[i] = -delta;
#pragma unroll
        for (int x = 0; x < NKS; ++x) {
          __builtin_amdgcn_sched_barrier(0);
          dp = M::mfma(operand[(NKS + x) % kAhead], gop[x], dp);
          operand[(NKS + x) % kAhead] = read(NKS + x + kAhead);
          // the exponentials between the products of dP
#pragma unroll
          for (int i = 16 / NKS * x; i < 16 / NKS * (x + 1); ++i) {
            sc[i] = fast_exp2(__builtin_fmaf(sc[i], p.scale_log2e, -m_ref));
            l_lane += sc[i];
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        V8 dsop[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          uint32_t w[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int i = 8 * b + 2 * j;
            w[j] = pack_pair<KIND>(sc[i] * dp[i], sc[i + 1] * dp[i + 1]);
          }
          dsop[b] = __builtin_bit_cast(V8, uint4_t{w[0], w[1], w[2], w[3]});
        }
#pragma unroll
        for (int x = 0; x < 2 * NB; ++x) {
          acc[x % NB] = M::mfma(operand[(2 * NKS + x) % kAhead], dsop[x / NB], acc[x % NB]);
          if (2 * NKS + x + kAhead < kReads) operand[(2 * NKS + x) % kAhead] = read(2 * NKS + x + kAhead);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      fetched_barrier();  // the tiles' previous readers (an earlier sequence of this block) are done
      fetch(t0, 0);
      for (int t = t0; t <= t1; t += 2) {
        step(t, 0);
        if (t + 1 <= t1) step(t + 1, 1);
      }
    }

    const float l_tot = both_halves(l_lane, sum);
    const float f = l_tot > 0.0f ? p.scale / l_tot : 0.0f;
    handed_barrier();  // (every wave has read its last tile)
    const int l = lane_now();
    const int64_t at = wave_row0 + (l & 31);
    // (as whole rows, the kernel in us: 2 x 2 048 tokens, 28 / 4 heads of 128: 131 -> 123; 4 x 4 096, 32 / 8: 814 -> 790)
    if (p.grad_dtype != ARENO_DT_F32) {
      using Stage = RowStage<4 * NB>;
      char* const stage = lds + wave * (32 * Stage::kRowBytes);
      static_assert(kRows * Stage::kRowBytes <= sizeof(lds), "the rows' place");
#pragma unroll
      for (int x = 0; x < 4 * NB; ++x) {
        const int nb = x >> 2, c = 4 * (x & 3);
        Stage::put(stage, l & 31, x, l >> 5, pack_pair<KIND>(acc[nb][c] * f, acc[nb][c + 1] * f), pack_pair<KIND>(acc[nb][c + 2] * f, acc[nb][c + 3] * f));
      }
      Stage::template take<32>(stage, l, [&](int r, int chunk, uint4_t w) {
        const int64_t to = wave_row0 + r;
        if (to >= q_lo && to < q_hi) *reinterpret_cast<uint4_t*>(static_cast<char*>(p.grad_q) + ((to * p.q_heads + h) * D + 8 * chunk) * 2) = w;
      });
    }
    if (at >= q_lo && at < q_hi) {
      if (p.grad_dtype == ARENO_DT_F32) {
#pragma unroll
        for (int x = 0; x < 4 * NB; ++x) {
          const int nb = x >> 2, c = 4 * (x & 3);
          GradStore<float>{}(p.grad_q, (at * p.q_heads + h) * D + 8 * x + 4 * (l >> 5), acc[nb][c] * f, acc[nb][c + 1] * f, acc[nb][c + 2] * f, acc[nb][c + 3] * f);
        }
      }
      if (l < 32) {
        float* st = p.row_stats + (h * p.q_tokens + at) * 2;
        st[0] = l_tot > 0.0f ? m_run + __builtin_log2f(l_tot) : __builtin_huge_valf();
        st[1] = -delta;
      }
    }
  }
  const int l = lane_now();
  const int64_t at = wave_row0 + (l & 31);
  if (at >= covered && at < p.q_tokens) {  // behind the last sequence, the end of a padded pack
    const int64_t elem = (at * p.q_heads + h) * D + 4 * (l >> 5);
    store_grads<typename M::elem>(p.grad_dtype, [&](auto store) {
#pragma unroll
      for (int c = 0; c < D / 8; ++c) store(p.grad_q, elem + 8 * c, 0.0f, 0.0f, 0.0f, 0.0f);
    });
  }
}

constexpr int64_t kBmComputeUnits = 256;

// Whether the vector-ALU kernels take a launch of wide heads in less time.  A matrix-core workgroup goes through the
// sequences of its block one after the other, at least one tile each (the dkv kernel for every q head of the group);
// the vector-ALU kernels have a wave per row and do not care.  For sequences of 64 tokens and more the matrix cores
// win by up to 30 times, for many single tokens they lose by as much; in between both are estimated, in us, from what 1 494
// launches of 1 .. 400 sequences took, most of 1 .. 64 tokens (head dims 192 and 256, ten head ratios, equal and ragged lengths,
// windows).  The choice takes 0.1 % longer than the better of both (more than a tenth in 6, 44 % at most, of ragged lengths).
// vector ALU, matrix cores, in us, heads of 256: 12 / 4, 4 x 21 tokens 70, 46; 5 x 5 53, 58; 8 / 2, 31 x 7 80, 87; 44 x 8 104, 67; 16 / 8,
// 77 x 2 124, 180; of 192: 8 / 1, 2 x 12 54, 37; 24 / 8, 6 x 12 63, 52; 12 / 4, 18 x 7 58, 73.
bool vector_alu_is_faster(const BwdParams& p) {
  const bool d256 = p.head_dim == 256;
  auto ceil_div = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  // (lengths are taken to be about equal; a window of w shows w + 1 keys to a query)
  const int64_t seqs = p.num_seqs, group = p.q_heads / p.kv_heads;
  const int64_t queries = std::max<int64_t>(p.q_tokens / seqs, 1), keys = std::max<int64_t>(p.k_tokens / seqs, 1);
  const int64_t reach = p.window_left >= 0 ? p.window_left + int64_t{1} : INT32_MAX;
  // matrix cores: sequences in a block (which ends inside one as often as not), steps of each, rounds of workgroups
  auto in_block = [&](int64_t rows, int64_t length) { return std::min(static_cast<double>(seqs), ceil_div(rows, length) + 0.5); };
  const int parts = dkv32_wide_parts(p);
  const int64_t dkv_rows = 64 / parts, dkv_rounds = ceil_div(ceil_div(p.k_tokens, dkv_rows) * p.kv_heads, kBmComputeUnits);
  const double dkv_steps = in_block(dkv_rows, keys) *
                           ceil_div(ceil_div(std::min(queries, reach + dkv_rows), kBmTile) * group, parts) * dkv_rounds;
  const double dq_steps = in_block(kBmRows, queries) * ceil_div(std::min(keys, reach + kBmRows), kBmTile) *
                          ceil_div(ceil_div(p.q_tokens, kBmRows) * p.q_heads, 2 * kBmComputeUnits);
  const double matrix_cores = d256 ? 11.5 * dkv_rounds + 2.85 * dkv_steps + 4.2 * dq_steps : 10.5 * dkv_rounds + 2.5 * dkv_steps + 3.4 * dq_steps;
  // vector ALU: a wave per row, one of them per SIMD; a row's start and its keys or pairs, 16 at a time
  const int64_t seen = std::min(keys, reach), pairs = std::min(queries, reach) * group, waves = 4 * kBmComputeUnits;
  const int64_t q_rounds = ceil_div(p.q_tokens * p.q_heads, waves), k_rounds = ceil_div(p.k_tokens * p.kv_heads, waves);
  const double vector_alu = d256 ? q_rounds * (21.2 + 2.29 * ceil_div(seen, 16)) + k_rounds * (24.1 + 4.25 * ceil_div(pairs, 16))
                                 : q_rounds * (16 + 1.41 * ceil_div(seen, 16)) + k_rounds * (18.1 + 2.74 * ceil_div(pairs, 16));
  return vector_alu < matrix_cores;
}

}  // namespace

int launch_attention_backward_mfma(const BwdParams& p, void* stream) {
  if (p.dtype != ARENO_DT_BF16 && p.dtype != ARENO_DT_F16) return ARENO_ERR_UNSUPPORTED;
  if (p.head_dim != 64 && p.head_dim != 128 && p.head_dim != 192 && p.head_dim != 256) return ARENO_ERR_UNSUPPORTED;
  // the kernels mask raw scores and take row maxima before scaling: any other scale is for the vector-ALU kernels, as in
  // the forward (launch_prefill_mfma)
  if (!(p.scale_log2e > 0.0f)) return ARENO_ERR_UNSUPPORTED;
  if (p.q_heads > 65535 || p.kv_heads > 65535) return ARENO_ERR_UNSUPPORTED;
  const int64_t q_blocks = (p.q_tokens + kBmRows - 1) / kBmRows, k_blocks = (p.k_tokens + kBmRows - 1) / kBmRows;
  if (q_blocks * p.q_heads > 0x7fffffffLL || k_blocks * p.kv_heads > 0x7fffffffLL) return ARENO_ERR_UNSUPPORTED;
  const bool bf16 = p.dtype == ARENO_DT_BF16;
  // The dq kernel with 32 rows per wave where a row sees many keys and the launch has several workgroups per compute unit:
  // small launches are their longest block, whose start and end take longer with twice the rows, and so are blocks of
  // many short sequences, which it takes one after the other.  The backward with 16 and 32 rows, us (in brackets workgroups of 64
  // rows per unit), D = 128: 4 x 4 096 tokens, 32 / 8 heads (32) 2 194, 1 802; 2 x 2 048, 28 / 4 (7) 286, 255; 1 x 4 096, 16 / 16 (4) 302, 263; 6 / 6
  // (1.5) 187, 179; 1 x 2 048, 16 / 16 (2) 109, 106; 6 / 6 (0.8) 95.2, 97.1; 4 x 1 024, 16 / 16 (4) 108, 101; 2 x 1 024 (2) 65.3, 66.9; 1 x 1 024 (1) 55.2,
  // 58.4; 1 x 600 (0.6) 39.0, 44.3; 28 / 4 heads, 4 x 600 (4.2) 161, 155; 64 x 512 (56) 769, 755; 16 x 256 (7) 85.9, 89.9; 256 x 128 (56) 465, 537;
  // 512 x 8 (7) 158, 229; windows over 4 x 2 048 (14): 1 024 440, 382; 512 296, 271; 256 195, 198; 128 149, 163.  D = 64: 4 x 4 096, 32 / 8 (32)
  // 1 178, 1 044; 4 x 1 024, 16 / 16 (4) 60.6, 59.4; 2 x 1 024 (2) 40.7, 42.1; 12 x 512 (6) 60.1, 62.3; 28 / 4 heads, 64 x 512 (56) 402, 406; 256 x 128
  // (56) 243, 272; windows over 4 x 2 048: 512 155, 151; 256 105, 107; 128 75.8, 85.5.
  // ARENO_BACKWARD_DQ_ROWS=16|32 (read at every launch) fixes the choice, for tests and timing; at head dims 192 and 256,
  // which have one form, either value asks for it whatever the estimate says, as ARENO_BACKWARD_PARTS does.
  const int64_t mean_length = p.q_tokens / (p.num_seqs > 0 ? p.num_seqs : 1);
  const int64_t seen = p.window_left >= 0 ? std::min<int64_t>(mean_length, p.window_left + int64_t{1}) : mean_length;
  const int64_t workgroups = q_blocks * p.q_heads;  // (of 64 rows)
  int dq_rows = p.head_dim == 128 ? ((seen >= 512 && workgroups >= 3 * kBmComputeUnits) || (seen > 1024 && workgroups >= kBmComputeUnits * 3 / 2) ? 32 : 16)
                                  : (seen >= 512 && mean_length >= 1024 && workgroups >= 4 * kBmComputeUnits ? 32 : 16);
  if (fixed_by("ARENO_BACKWARD_DQ_ROWS", "32")) dq_rows = 32;
  if (fixed_by("ARENO_BACKWARD_DQ_ROWS", "16")) dq_rows = 16;
  // (head dims 192 and 256: not for many very short sequences, unless a switch asks for these kernels)
  if (p.head_dim > 128) {
    const bool asked_for = fixed_by("ARENO_BACKWARD_DQ_ROWS", "16") || fixed_by("ARENO_BACKWARD_DQ_ROWS", "32") ||
                           fixed_by("ARENO_BACKWARD_PARTS", "1") || fixed_by("ARENO_BACKWARD_PARTS", "2");
    if (!asked_for && vector_alu_is_faster(p)) return ARENO_ERR_UNSUPPORTED;
  }
  BwdLaunch dq, dkv;
  int64_t dkv_groups = 0;  // workgroups of a kv head
  if (p.head_dim > 128) {
    dq = dq32_wide_launch(p);
    dkv = dkv32_wide_launch(p, &dkv_groups);
  } else {
    bwd_fn fn;
    if (p.head_dim == 64) {
      fn = dq_rows == 32 ? (bf16 ? bwd_mfma32_dq_kernel<KV_BF16, 64> : bwd_mfma32_dq_kernel<KV_F16, 64>)
                         : (bf16 ? bwd_mfma_dq_kernel<KV_BF16, 64> : bwd_mfma_dq_kernel<KV_F16, 64>);
    } else {
      fn = dq_rows == 32 ? (bf16 ? bwd_mfma32_dq_kernel<KV_BF16, 128> : bwd_mfma32_dq_kernel<KV_F16, 128>)
                         : (bf16 ? bwd_mfma_dq_kernel<KV_BF16, 128> : bwd_mfma_dq_kernel<KV_F16, 128>);
    }
    dq = BwdLaunch{fn, 0, kBmThreads, kBmWaves * dq_rows};
    dkv = dkv32_launch(p, &dkv_groups);
  }
  const char* op = "areno_hip_attention_backward";
  if (dq.fn == nullptr || dkv.fn == nullptr) return fail(ARENO_ERR_LAUNCH, "%s: the kernels' LDS size was refused", op);
  hipStream_t s = static_cast<hipStream_t>(stream);
  BwdParams params = p;
  params.q_order = block_order(p.q_tokens, dq.rows, p.num_seqs);
  params.k_order = block_order(p.k_tokens, dkv.rows, p.num_seqs);
  if (q_blocks > 0) {
    const int64_t dq_blocks = (p.q_tokens + dq.rows - 1) / dq.rows;
    hipLaunchKernelGGL(dq.fn, dim3(static_cast<unsigned>(dq_blocks * p.q_heads)), dim3(dq.threads), dq.lds_bytes, s, params);
    if (int rc = check_launch(op)) return rc;
  }
  if (k_blocks > 0) {
    hipLaunchKernelGGL(dkv.fn, dim3(static_cast<unsigned>(dkv_groups * p.kv_heads)), dim3(dkv.threads), dkv.lds_bytes, s, params);
    if (int rc = check_launch(op)) return rc;
  }
  return ARENO_OK;
}

}  // namespace areno
