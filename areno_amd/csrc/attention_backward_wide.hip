// Backward of the causal varlen / dense attention ops at head dims 192 and 256 on 32 x 32 x 16 matrix products (gfx950),
// 16-bit inputs: the two launches of attention_backward_mfma.hip for them.  The reference: areno/accel/csrc/attention.cu:244-524.
//
// What 32 rows need is more registers than a wave has (operands of two tensors and dK and dV are 384 at head dim 256), so
// two waves work on them together, each on one of the first two products:
//   dq    one holds Q:  S^T = K . Q^T, the online softmax, P;  one holds dO:  dP^T = V . dO^T - dO . O;  they exchange P and dP
//         in LDS, and each takes half the columns of  dQ^T += K^T . dS^T,  dS = P * dP;
//   dkv   one holds K and dV:  S = Q . K^T,  P = exp2(S - lse), which it hands over in LDS,  dV^T += dO^T . P;
//         one holds V and dK:  dP = dO . V^T - dO . O,  dS = P * dP,  dK^T += Q^T . dS.
// The streamed rows come in tiles of 32 that the memory pipe puts into LDS; a C tile of the first products is the B operand
// of the last as it lies (mfma32_tiles.hpp).  P and dS are not rounded to 16 bits on the way (wide_weights), and S is summed
// in the same order in both kernels, so that its roundings do not count between P and the log-sum-exp.
//
// Bound: what one wave issues and waits for (dkv: one wave per SIMD, 500 vector instructions and 64 products of 32
// cycles a step, a third of the time in waits; dq: two).  Against 16 x 16 x 32 products with 16 rows per wave, the backward, us: 2 717
// tokens in four sequences, 16 / 8 heads of 256, window 512, bf16: 354 -> 198 (the profiler's dkv 239 -> 133, dq 109 -> 77);
// 1 x 1 000, 8 / 1 heads: 910 -> 217.  Relative error of dV against 64 bits, before
// and now: 2.74e-7, 2.64e-7 (bf16), 2.83e-7, 2.71e-7 (fp16); queries four times as large: 6.2e-7, 5.7e-7.
#include <algorithm>
#include <atomic>

#include "attention_backward.hpp"
#include "mfma32_tiles.hpp"

namespace areno {
namespace {

constexpr int kWideTile = 32;  // query rows per step
constexpr float kWideNegInf = -__builtin_huge_valf();
extern __shared__ __attribute__((aligned(1024))) char wide_lds[];

// Sixteen values of a column (with the other lane half's, thirty-two) as three 16-bit B operands of either block of 16 rows
// that add up to them, times a power of two in fp16: the 16-bit inputs of wide heads had fp32 kernels until the matrix
// cores took them, and lose nothing by it.
// bf16 holds eight significant bits with fp32's exponents: the upper half of a value's word, that of the rest and what is
// left then are its 24.  fp16 holds eleven in a narrow range: the values of a column are first scaled together, so that the
// largest comes to lie in [2^14, 2^15); what three parts leave, below fp16's smallest step of 2^-24, is less than 2^-38 of it.
template <int KIND>
struct WideWeights {
  typename Mfma32<KIND>::vec8 part[3][2];
  float unscale;
};
template <int KIND>
__device__ __forceinline__ WideWeights<KIND> wide_weights(float16_t x) {
  using V8 = typename Mfma32<KIND>::vec8;
  WideWeights<KIND> s;
  if constexpr (KIND == KV_F16) {
    float most = __builtin_fabsf(x[0]);
#pragma unroll
    for (int i = 1; i < 15; i += 2) most = max3_f32(most, __builtin_fabsf(x[i]), __builtin_fabsf(x[i + 1]));
    most = max_f32(most, __builtin_fabsf(x[15]));
    uint32_t a = __builtin_bit_cast(uint32_t, most), b = a;
    swap_rows32(a, b);
    most = max_f32(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
    // exponent field of the scale: 2^14 over the largest value's power of two (at most 2^126, for its inverse)
    const uint32_t field = min(268u - (__builtin_bit_cast(uint32_t, most) >> 23), 253u);
    const float scale = __builtin_bit_cast(float, field << 23);
    s.unscale = __builtin_bit_cast(float, (254u - field) << 23);
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] *= scale;
  }
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    uint32_t w[3][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float lo = x[8 * b + 2 * j], hi = x[8 * b + 2 * j + 1];
#pragma unroll
      for (int i = 0; i < 3; ++i) {  // (the subtractions are exact)
        if constexpr (KIND == KV_F16) {
          const auto h = __builtin_amdgcn_cvt_pkrtz(lo, hi);
          w[i][j] = __builtin_bit_cast(uint32_t, h);
          lo -= static_cast<float>(h[0]);
          hi -= static_cast<float>(h[1]);
        } else {
          const uint32_t ul = __builtin_bit_cast(uint32_t, lo), uh = __builtin_bit_cast(uint32_t, hi);
          w[i][j] = __builtin_amdgcn_perm(uh, ul, 0x07060302u);  // the upper halves, lo's in the low one
          lo -= __builtin_bit_cast(float, ul & 0xffff0000u);
          hi -= __builtin_bit_cast(float, uh & 0xffff0000u);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) s.part[i][b] = __builtin_bit_cast(V8, uint4_t{w[i][0], w[i][1], w[i][2], w[i][3]});
  }
  return s;
}

// acc += columns . the values that the parts add up to, over NB blocks of 32 columns; operand 2 nb + b holds the columns of
// block nb and 16 rows b, the first kAhead of them are there.  A tile's products are summed by themselves, the small ones
// first, so the running sum rounds once per tile; one block's sum is added up between the next one's products (and a step's
// addresses are not kept: the kernels of 2 368 tokens in four sequences, 16 / 8 heads of 256, window 512: dkv 126 -> 122.5 us, dq 73.2 -> 72).
template <int KIND, int NB, int AHEAD, typename Columns>
__device__ __forceinline__ void add_products(const WideWeights<KIND>& weights, typename Mfma32<KIND>::vec8 (&operand)[AHEAD],
                                             const Columns& columns, float16_t (&acc)[NB]) {
  // (values e0 .. e1 - 1 of a block's)
  auto add = [&](int nb, const float16_t& sum, int e0, int e1) {
#pragma unroll
    for (int e = e0; e < e1; ++e) {
      if constexpr (KIND == KV_BF16) {
        acc[nb][e] += sum[e];
      } else {
        acc[nb][e] = __builtin_fmaf(sum[e], weights.unscale, acc[nb][e]);
      }
    }
  };
  float16_t sums[2];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    __builtin_amdgcn_sched_barrier(0);
    float16_t sum = zero16();
#pragma unroll
    for (int x = 0; x < 6; ++x) {
      sum = Mfma32<KIND>::mfma(operand[(2 * nb + x % 2) % AHEAD], weights.part[2 - x / 2][x % 2], sum);
      if (x >= 4 && 2 * nb + x - 4 + AHEAD < 2 * NB) operand[(2 * nb + x - 4) % AHEAD] = columns(2 * nb + x - 4 + AHEAD);
      if (nb > 0 && x > 0) add(nb - 1, sums[(nb - 1) & 1], (x - 1) * 16 / 5, x * 16 / 5);
      __builtin_amdgcn_sched_barrier(0);
    }
    sums[nb & 1] = sum;
  }
  add(NB - 1, sums[(NB - 1) & 1], 0, 16);
}

__device__ __forceinline__ float both_halves_max(float x) {
  uint32_t a = __builtin_bit_cast(uint32_t, x), b = a;
  swap_rows32(a, b);
  return max_f32(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
}
__device__ __forceinline__ float both_halves_sum(float x) {
  uint32_t a = __builtin_bit_cast(uint32_t, x), b = a;
  swap_rows32(a, b);
  return __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
}

// ---- dQ (and the rows' statistics) ------------------------------------------------------------------------------------
constexpr int kWideDqWaves = 4;  // two pairs
template <int D>
struct WideDqShape {
  using Tile = LdsTile<D, kWideTile, kWideDqWaves>;
  static constexpr int kRows = 16 * kWideDqWaves;
  static constexpr int kV = 2 * Tile::kBytes;  // two tiles of K, one of V
  static constexpr int kHands = kV + Tile::kBytes;
  static constexpr int kHand = 2 * 16 * kWave * 4 + kWave * 4;  // P, dP, the rows' references
  static constexpr int kLdsBytes = kHands + kWideDqWaves / 2 * kHand;
};

template <int KIND, int D>
__global__ __launch_bounds__(kWideDqWaves* kWave) __attribute__((amdgpu_waves_per_eu(2, 2))) void bwd_mfma32_wide_dq_kernel(BwdParams p) {
  using M = Mfma32<KIND>;
  using V8 = typename M::vec8;
  using L = WideDqShape<D>;
  using T = typename L::Tile;
  constexpr int NKS = D / 16, NB = D / 64, NF = T::kFetches;  // NB: a wave's blocks of 32 columns of dQ, every second one

  ask_for_arguments(p, p.q_order);
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave_of_block = uniform(tid >> 6);
  const int wave = wave_of_block >> 1;     // whose 32 query rows
  const bool second = wave_of_block & 1;  // dO and dP
  const int half = lane >> 5;
  const int h = static_cast<int>(blockIdx.x % static_cast<unsigned>(p.q_heads));
  const int kvh = h / (p.q_heads / p.kv_heads);
  const int block = uniform(block_in_launch_order(static_cast<int>(blockIdx.x / static_cast<unsigned>(p.q_heads)), p.q_order, L::kRows, true));
  const int64_t r0 = static_cast<int64_t>(block) * L::kRows;
  const int64_t block_end = r0 + L::kRows < p.q_tokens ? r0 + L::kRows : p.q_tokens;
  const int64_t wave_row0 = r0 + 32 * wave;
  const int64_t row = wave_row0 + (lane & 31);  // this lane's query row (a column of the products)
  const int64_t row_elem = (row * p.q_heads + h) * D;

  uint32_t at_rows = T::rows_base(lane & 31, half) + (second ? L::kV : 0);
  uint32_t at_columns = T::columns_base(lane) ^ (second ? 4u << 4 : 0u);
  const uint32_t lds0 = lds_address(wide_lds);
  const uint32_t stride = static_cast<uint32_t>(p.kv_heads) * (D * 2);
  // where a lane's chunk of fetch f lies in a tile; a fetch is two rows at head dim 256, and then only bits of the twist and
  // the scalar rows differ between fetches
  uint32_t offsets[D == 256 ? 1 : NF];
#pragma unroll
  for (int f = 0; f < (D == 256 ? 1 : NF); ++f) {
    const int slot = (D == 256 ? 0 : (wave_of_block * NF + f) * 64) + lane, r = slot / T::kChunksPerRow;
    offsets[f] = static_cast<uint32_t>(r) * stride + static_cast<uint32_t>((slot % T::kChunksPerRow) ^ T::twist(r)) * 16u;
  }
  auto fetch_offset = [&](int f) {
    if constexpr (D != 256) return offsets[f];
    const int r = 2 * (wave_of_block * NF + f);
    return (offsets[0] ^ static_cast<uint32_t>(T::twist(r) << 4)) + static_cast<uint32_t>(r) * stride;
  };
  float4_t* const hand = reinterpret_cast<float4_t*>(wide_lds + L::kHands + wave * L::kHand) + lane;
  float* const reference = reinterpret_cast<float*>(wide_lds + L::kHands + wave * L::kHand + 2 * 16 * kWave * 4) + lane;

  // (the block's first sequence is looked up while the rows below are on their way)
  int s = uniform(seq_of_row(p.cu_q, p.num_seqs, r0));
  int64_t sq0 = uniform(p.cu_q[s]), sq1;
  V8 own[NKS];  // this lane's parts of its row of Q or dO (B operands)
  float delta = 0.0f;
  {
    uint4_t w[NKS], o[NKS];
    const void* const from = second ? p.grad_out : p.q;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) w[ks] = o[ks] = uint4_t{0u, 0u, 0u, 0u};
    if (row < p.q_tokens) {
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) w[ks] = load16(from, (row_elem + 16 * ks + 8 * half) * 2);
      if (second) {
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) o[ks] = load16(p.out, (row_elem + 16 * ks + 8 * half) * 2);
      }
    }
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      // (waited for here: left to their first use inside the loop, that wait would cover every tile's fetches as well)
      asm volatile("" : "+v"(w[ks]));
      own[ks] = __builtin_bit_cast(V8, w[ks]);
      if (second) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          delta += operand_element<KIND>(w[ks][j], 0) * operand_element<KIND>(o[ks][j], 0) +
                   operand_element<KIND>(w[ks][j], 1) * operand_element<KIND>(o[ks][j], 1);
        }
      }
    }
    delta = both_halves_sum(delta);
  }

  int covered = 0;  // (where the sequences seen so far end)
  for (; s < p.num_seqs && sq0 < block_end; ++s, sq0 = sq1) {
    // (asked for together)
    const int q_end = p.cu_q[s + 1], k_begin = p.cu_k[s], k_end = p.cu_k[s + 1], before = p.ctx != nullptr ? p.ctx[s] : 0;
    sq1 = covered = uniform(q_end);
    const int64_t q_lo = sq0 > r0 ? sq0 : r0, q_hi = sq1 < block_end ? sq1 : block_end;
    if (q_lo >= q_hi) continue;
    const int ctx = uniform(before);
    const int64_t k_first = uniform(k_begin);
    const int n_k = uniform(k_end) - static_cast<int>(k_first);
    const bool live = row >= q_lo && row < q_hi;
    const int pos = live ? ctx + static_cast<int>(row - sq0) : -1;
    const uint64_t live_lanes = __builtin_amdgcn_ballot_w64(live);
    const bool wave_live = live_lanes != 0, wave_full = live_lanes == ~0ull;
    const int wave_pos_lo = ctx + static_cast<int>(wave_row0 - sq0), wave_pos_hi = wave_pos_lo + 31;
    const int pos_min = ctx + static_cast<int>(q_lo - sq0), pos_max = ctx + static_cast<int>(q_hi - 1 - sq0);
    const int key_lo = p.window_left >= 0 ? (pos_min - p.window_left > 0 ? pos_min - p.window_left : 0) : 0;
    const int key_hi = pos_max < n_k - 1 ? pos_max : n_k - 1;

    float16_t acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = zero16();
    float m_run = kWideNegInf, l_lane = 0.0f;

    if (key_hi >= key_lo) {  // (the same for the whole workgroup)
      const int t0 = key_lo / kWideTile, t1 = key_hi / kWideTile;
      const int64_t head_base = (k_first * p.kv_heads + kvh) * (D * 2);
      auto fetch = [&](const void* from, int t, uint32_t to) {
        const int last = min(n_k - t * kWideTile, kWideTile) - 1;  // rows behind the sequence's last repeat it
        const char* const base = static_cast<const char*>(from) + head_base + static_cast<int64_t>(t) * kWideTile * stride;
        const uint32_t dst = lds0 + to + wave_of_block * (NF * 1024);
        if (last == kWideTile - 1) {
#pragma unroll
          for (int f = 0; f < NF; ++f) fetch_to_lds(base, fetch_offset(f), dst + f * 1024);
        } else {
          const int l = lane_now();
#pragma unroll
          for (int f = 0; f < NF; ++f) {
            const int r = ((wave_of_block * NF + f) * 64 + l) / T::kChunksPerRow;
            fetch_end_to_lds(base, fetch_offset(f) - static_cast<uint32_t>(max(r - last, 0)) * stride, dst + f * 1024);
          }
        }
      };
      auto rescale = [&](float m_new) {
        const float m_ref = m_new == kWideNegInf ? 0.0f : m_new;
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
      };
      auto step = [&](int t, int buf) {
        asm volatile("" : "+v"(at_rows), "+v"(at_columns));  // (the addresses of a step are worked out where they are used)
        fetched_barrier();  // tile t (asked for a step ago) is there, and every wave has left tile t - 1
        if (t < t1) fetch(p.k, t + 1, (buf ^ 1) * T::kBytes);
        const int key_first = kWideTile * t, key_last = key_first + kWideTile - 1;
        const bool seen = wave_live && !(wave_full && (key_first > wave_pos_hi || (p.window_left >= 0 && key_last < wave_pos_lo - p.window_left)));
        char* const k_lds = wide_lds + buf * T::kBytes;
        // operands are read kAhead products in front of their own
        constexpr int kAhead = 4;
        V8 operand[kAhead];
        float16_t c, odd = zero16();
        auto columns = [&](int x) { return tile_columns<KIND, T>(k_lds, at_columns, 16 * (x & 1), 2 * (x >> 1)); };
        if (seen) {
          char* const rows_lds = second ? wide_lds : k_lds;
#pragma unroll
          for (int x = 0; x < kAhead; ++x) operand[x] = tile_rows<KIND, T>(rows_lds, at_rows, 0, x);
#pragma unroll
          for (int i = 0; i < 16; ++i) c[i] = -delta;  // (nothing for S; dP comes out less dO . O)
#pragma unroll
          for (int x = 0; x < NKS; ++x) {
            __builtin_amdgcn_sched_barrier(0);
            if (x & 1) {
              odd = M::mfma(operand[x % kAhead], own[x], odd);
            } else {
              c = M::mfma(operand[x % kAhead], own[x], c);
            }
            if (x + kAhead < NKS) operand[x % kAhead] = tile_rows<KIND, T>(rows_lds, at_rows, 0, x + kAhead);
          }
          c += odd;
#pragma unroll
          for (int x = 0; x < kAhead; ++x) operand[x] = columns(x);
          if (!second) {
            const bool plain = wave_full && key_last < n_k && key_last <= wave_pos_lo && (p.window_left < 0 || key_first >= wave_pos_hi - p.window_left);
            if (!plain) {
              const int base = key_first + 4 * half;  // keys base + 8 c + j
              const int last = min(pos, n_k - 1) - base, first = p.window_left < 0 ? -base : pos - p.window_left - base;
#pragma unroll
              for (int i = 0; i < 16; ++i) {
                const int key = 8 * (i >> 2) + (i & 3);
                c[i] = key >= first && key <= last ? c[i] : kWideNegInf;
              }
            }
            // (the reference is raised only when a score of the wave exceeds its row's by more than 2^8)
            float mt = c[0];
#pragma unroll
            for (int i = 1; i < 15; i += 2) mt = max3_f32(mt, c[i], c[i + 1]);
            mt = max_f32(mt, c[15]);
            if (__builtin_amdgcn_ballot_w64(mt * p.scale_log2e > m_run + 8.0f) != 0)
              rescale(max_f32(m_run, both_halves_max(mt) * p.scale_log2e));  // (the scale is positive)
            const float m_ref = m_run == kWideNegInf ? 0.0f : m_run;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              c[i] = fast_exp2(__builtin_fmaf(c[i], p.scale_log2e, -m_ref));  // (exp2(-inf) = 0: masked keys)
              l_lane += c[i];
            }
            *reference = m_run;
          }
#pragma unroll
          for (int x = 0; x < 4; ++x) hand[(second ? 4 + x : x) * kWave] = float4_t{c[4 * x], c[4 * x + 1], c[4 * x + 2], c[4 * x + 3]};
        }
        handed_barrier();
        if (t < t1) fetch(p.v, t + 1, L::kV);
        if (!seen) return;
        if (second) {
          const float m_new = *reference;
          if (__builtin_amdgcn_ballot_w64(m_new != m_run) != 0) rescale(m_new);
        }
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const float4_t other = hand[(second ? x : 4 + x) * kWave];
#pragma unroll
          for (int j = 0; j < 4; ++j) c[4 * x + j] *= other[j];
        }
        add_products<KIND, NB, kAhead>(wide_weights<KIND>(c), operand, columns, acc);
      };
      fetched_barrier();  // the tiles' previous readers (an earlier sequence of this block) are done
      fetch(p.k, t0, 0);
      fetch(p.v, t0, L::kV);
      for (int t = t0; t <= t1; t += 2) {
        step(t, 0);
        if (t + 1 <= t1) step(t + 1, 1);
      }
    }

    // dQ = scale / l * sum_k p_k (dP_k - dO . O) K_k; the row's log-sum-exp (log2 domain) and -(dO . O) for the dkv kernel
    handed_barrier();  // (the last hand is read)
    if (!second) *reference = both_halves_sum(l_lane);
    handed_barrier();
    const float l_tot = *reference;
    const float f = l_tot > 0.0f ? p.scale / l_tot : 0.0f;
    const int l = lane_now();  // (worked out anew: kept, what follows from it would cost the loop registers)
    const int64_t at = wave_row0 + (l & 31);
    if (p.grad_dtype != ARENO_DT_F32) {  // as whole blocks of 32 elements, through the tiles' LDS
      using Stage = RowStage<4 * NB>;
      char* const stage = wide_lds + wave_of_block * (32 * Stage::kRowBytes);
      static_assert(kWideDqWaves * 32 * Stage::kRowBytes <= L::kHands, "the rows' place");
#pragma unroll
      for (int x = 0; x < 4 * NB; ++x) {
        const int nb = x >> 2, c = 4 * (x & 3);
        Stage::put(stage, l & 31, x, l >> 5, pack_pair<KIND>(acc[nb][c] * f, acc[nb][c + 1] * f), pack_pair<KIND>(acc[nb][c + 2] * f, acc[nb][c + 3] * f));
      }
      Stage::template take<32>(stage, l, [&](int r, int chunk, uint4_t w) {
        const int64_t to = wave_row0 + r;
        const int elem = 64 * (chunk >> 2) + (second ? 32 : 0) + 8 * (chunk & 3);
        if (to >= q_lo && to < q_hi) *reinterpret_cast<uint4_t*>(static_cast<char*>(p.grad_q) + ((to * p.q_heads + h) * D + elem) * 2) = w;
      });
    }
    if (at >= q_lo && at < q_hi) {
      if (p.grad_dtype == ARENO_DT_F32) {
#pragma unroll
        for (int x = 0; x < 4 * NB; ++x) {
          const int nb = x >> 2, c = 4 * (x & 3);
          GradStore<float>{}(p.grad_q, (at * p.q_heads + h) * D + 64 * nb + (second ? 32 : 0) + 2 * c + 4 * (l >> 5), acc[nb][c] * f, acc[nb][c + 1] * f,
                             acc[nb][c + 2] * f, acc[nb][c + 3] * f);
        }
      }
      if (l < 32) {
        // a row without visible keys gets a reference no score reaches: its probabilities come out as zeros
        p.row_stats[(h * p.q_tokens + at) * 2 + (second ? 1 : 0)] =
            second ? -delta : l_tot > 0.0f ? m_run + __builtin_log2f(l_tot) : __builtin_huge_valf();
      }
    }
  }
  const int l = lane_now();
  const int64_t at = wave_row0 + (l & 31);
  if (at >= covered && at < p.q_tokens) {  // behind the last sequence, the end of a padded pack
    const int64_t elem = (at * p.q_heads + h) * D + (second ? 32 : 0) + 4 * (l >> 5);
    store_grads<typename M::elem>(p.grad_dtype, [&](auto store) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int c = 0; c < 4; ++c) store(p.grad_q, elem + 64 * nb + 8 * c, 0.0f, 0.0f, 0.0f, 0.0f);
      }
    });
  }
}

// ---- dK, dV -------------------------------------------------------------------------------------------------------------
template <int D, int KW, int P>
struct WideShape {
  static constexpr int kPartWaves = 2 * KW;
  using Tile = LdsTile<D, kWideTile, kPartWaves>;
  static constexpr int kThreads = kPartWaves * P * kWave;
  static constexpr int kKeys = 32 * KW;                     // key rows of a block
  static constexpr int kStat = kWideTile * 2 * 4;           // the rows' log-sum-exp, then their -(dO . O)
  static constexpr int kBuffer = 2 * Tile::kBytes + kStat;  // Q, dO
  static constexpr int kPart = 2 * kBuffer;
  static constexpr int kHand = 16 * kWave * 4;              // P of a pair of waves
  static constexpr int kSums = (P - 1) * kPartWaves * D * 32 * 4;
  static constexpr int kTiles = P * kPart > kSums ? P * kPart : kSums;
  static constexpr int kLdsBytes = kTiles + P * KW * kHand;
};

template <int KIND, int D, int KW, int P>
__global__ __launch_bounds__((WideShape<D, KW, P>::kThreads)) __attribute__((amdgpu_waves_per_eu(1, 1))) void bwd_mfma32_wide_dkv_kernel(BwdParams p) {
  using M = Mfma32<KIND>;
  using V8 = typename M::vec8;
  using L = WideShape<D, KW, P>;
  using T = typename L::Tile;
  constexpr int NKS = D / 16, NB = D / 32, NF = T::kFetches;

  ask_for_arguments(p, p.k_order);
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave_of_block = uniform(tid >> 6);
  const int part = wave_of_block / L::kPartWaves, part_wave = wave_of_block % L::kPartWaves;
  const int wave = part_wave >> 1;   // whose 32 keys
  const bool second = part_wave & 1;  // V and dK
  const int kvh = static_cast<int>(blockIdx.x % static_cast<unsigned>(p.kv_heads));
  const int group = p.q_heads / p.kv_heads;
  const int block = uniform(block_in_launch_order(static_cast<int>(blockIdx.x / static_cast<unsigned>(p.kv_heads)), p.k_order, L::kKeys, false));
  const int64_t r0 = static_cast<int64_t>(block) * L::kKeys;
  const int64_t block_end = r0 + L::kKeys < p.k_tokens ? r0 + L::kKeys : p.k_tokens;

  static_assert(L::kPart % 256 == 0 && T::kBytes % 256 == 0, "places that the reads' exclusive-ors leave alone");
  // a wave's rows operand comes from the one tile, its columns operand from the other
  uint32_t at_rows = T::rows_base(lane & 31, lane >> 5) + part * L::kPart + (second ? T::kBytes : 0);
  uint32_t at_columns = T::columns_base(lane) + part * L::kPart + (second ? 0 : T::kBytes);
  const uint32_t lds0 = lds_address(wide_lds) + part * L::kPart;
  const uint32_t stride = static_cast<uint32_t>(p.q_heads) * (D * 2);
  float4_t* const hand = reinterpret_cast<float4_t*>(wide_lds + L::kTiles + (part * KW + wave) * L::kHand);
  auto fetch_row = [&](int f, int lane) { return ((part_wave * NF + f) * 64 + lane) / T::kChunksPerRow; };
  uint32_t fetch_offset[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int slot = (part_wave * NF + f) * 64 + lane, r = slot / T::kChunksPerRow;
    fetch_offset[f] = static_cast<uint32_t>(r) * stride + static_cast<uint32_t>((slot % T::kChunksPerRow) ^ T::twist(r)) * 16u;
  }

  // (the block's first sequence is looked up while the rows below are on their way)
  int s = uniform(seq_of_row(p.cu_k, p.num_seqs, r0));
  int64_t sk0 = uniform(p.cu_k[s]), sk1;
  V8 own[NKS];  // this lane's parts of its row of K or V (B operands)
  const int64_t row = r0 + 32 * wave + (lane & 31);
  {
    uint4_t w[NKS];
    const void* const from = second ? p.v : p.k;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) w[ks] = uint4_t{0u, 0u, 0u, 0u};
    if (row < p.k_tokens) {
      const int64_t elem = (row * p.kv_heads + kvh) * D + 8 * (lane >> 5);
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) w[ks] = load16(from, (elem + 16 * ks) * 2);
    }
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      // (waited for here: left to their first use inside the loop, that wait would cover every tile's fetches as well; in
      // accumulation registers, where the products read them as they are)
      asm volatile("" : "+a"(w[ks]));
      own[ks] = __builtin_bit_cast(V8, w[ks]);
    }
  }
  float16_t acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) acc[nb] = zero16();

  for (; s < p.num_seqs && sk0 < block_end; ++s, sk0 = sk1) {
    // (asked for together)
    const int k_end = p.cu_k[s + 1], q_begin = p.cu_q[s], q_end = p.cu_q[s + 1], before = p.ctx != nullptr ? p.ctx[s] : 0;
    sk1 = uniform(k_end);
    const int64_t k_lo = sk0 > r0 ? sk0 : r0, k_hi = sk1 < block_end ? sk1 : block_end;
    if (k_lo >= k_hi) continue;
    const int ctx = uniform(before);
    const int64_t q_first = uniform(q_begin);
    const int n_q = uniform(q_end) - static_cast<int>(q_first);
    const bool live = row >= k_lo && row < k_hi;
    const uint64_t live_lanes = __builtin_amdgcn_ballot_w64(live);
    const bool wave_live = live_lanes != 0, wave_full = live_lanes == ~0ull;
    const int wave_key_lo = static_cast<int>(r0 + 32 * wave - sk0), wave_key_hi = wave_key_lo + 31;
    // queries i (position ctx + i) that see one of the block's keys: key <= ctx + i <= key + window
    const int key_min = static_cast<int>(k_lo - sk0), key_max = static_cast<int>(k_hi - 1 - sk0);
    const int i_lo = key_min - ctx > 0 ? key_min - ctx : 0;
    int i_hi = n_q - 1;
    if (p.window_left >= 0 && key_max + p.window_left - ctx < i_hi) i_hi = key_max + p.window_left - ctx;
    if (i_hi < i_lo) continue;  // (the same for the whole workgroup)
    const int t0 = i_lo / kWideTile, t1 = i_hi / kWideTile;
    const int tiles = t1 - t0 + 1;
    // the stream: tiles of every q head of the group, head by head; this part takes steps part, part + P, ...
    const int stream_steps = tiles * group;
    const int steps = (stream_steps - part + P - 1) / P;  // this part's
    const int rounds = (stream_steps + P - 1) / P;        // the longest part's: every part keeps the barriers of all
    // the step whose tile is fetched next: its tile, where its rows of Q (and, a fixed way off, of dO) and statistics lie
    const int64_t tile_bytes = static_cast<int64_t>(kWideTile) * stride;
    const int64_t head_bytes = D * 2 - tiles * tile_bytes, head_stats = (p.q_tokens - static_cast<int64_t>(tiles) * kWideTile) * 8;
    const int64_t to_grad = static_cast<const char*>(p.grad_out) - static_cast<const char*>(p.q);
    int tile = t0 + part, ahead = tile;
    const char* q_ahead = static_cast<const char*>(p.q) + q_first * stride + kvh * group * (D * 2) + tile * tile_bytes;
    const char* stat_ahead = reinterpret_cast<const char*>(p.row_stats) + ((kvh * group) * p.q_tokens + q_first + tile * kWideTile) * 8;
    auto to_next_heads = [&] {
      while (ahead > t1) {
        ahead -= tiles;
        q_ahead += head_bytes;
        stat_ahead += head_stats;
      }
    };
    to_next_heads();
    while (tile > t1) tile -= tiles;
    // tiles this wave computes on (the first to the last that one of its keys is seen from), and those without a mask
    int seen_hi = t1, plain_hi = n_q / kWideTile - 1;
    const int seen_lo = max(wave_key_lo - ctx, 0) / kWideTile, plain_lo = max(wave_key_hi - ctx + kWideTile - 1, 0) / kWideTile;
    if (p.window_left >= 0) {
      seen_hi = wave_key_hi + p.window_left - ctx < 0 ? -1 : (wave_key_hi + p.window_left - ctx) / kWideTile;
      const int reach = wave_key_lo + p.window_left - ctx - (kWideTile - 1);
      plain_hi = reach < 0 ? -1 : min(plain_hi, reach / kWideTile);
    }
    if (!wave_live) seen_hi = -1;
    if (!wave_full) plain_hi = -1;
    auto fetch = [&](int buf) {
      const int last = min(n_q - ahead * kWideTile, kWideTile) - 1;  // rows behind the sequence's last repeat it
      const char* const qb = q_ahead;
      const char* const gb = q_ahead + to_grad;
      const uint32_t dst = lds0 + static_cast<uint32_t>(buf * L::kBuffer + part_wave * (NF * 1024));
      const int lane = lane_now();
      if (last == kWideTile - 1) {
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          fetch_to_lds(qb, fetch_offset[f], dst + f * 1024);
          fetch_to_lds(gb, fetch_offset[f], dst + T::kBytes + f * 1024);
        }
      } else {
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          const uint32_t off = fetch_offset[f] - static_cast<uint32_t>(max(fetch_row(f, lane) - last, 0)) * stride;
          fetch_end_to_lds(qb, off, dst + f * 1024);
          fetch_end_to_lds(gb, off, dst + T::kBytes + f * 1024);
        }
      }
      if (part_wave == 0) {
        fetch_words_to_lds(stat_ahead, static_cast<uint32_t>(min(lane & 31, last)) * 8u + (lane >> 5) * 4u,
                           lds0 + static_cast<uint32_t>(buf * L::kBuffer + 2 * T::kBytes));
      }
      ahead += P;
      q_ahead += P * tile_bytes;
      stat_ahead += P * kWideTile * 8;
      to_next_heads();
    };
    auto step = [&](int i, int buf) {
      fetched_barrier();  // the step's tile (asked for a step ago) is there, and every wave has left the one before
      if (i + 1 < steps) fetch(buf ^ 1);
      const int t = tile;
      tile += P;
      while (tile > t1) tile -= tiles;
      if (i >= steps || t < seen_lo || t > seen_hi) {
        handed_barrier();
        return;
      }
      asm volatile("" : "+v"(at_rows), "+v"(at_columns));  // (the addresses of a step are worked out where they are used)
      char* const lds = wide_lds + buf * L::kBuffer;
      // this lane's rows' statistics: rows 8 c + 4 (lane / 32) .. + 3
      auto stat = [&](int c) {
        return *reinterpret_cast<const float4_t*>(lds + 2 * T::kBytes + part * L::kPart + (second ? 128 : 0) + 32 * c + 16 * (lane_now() >> 5));
      };
      // operands are read kAhead products in front of their own
      constexpr int kAhead = 4;
      V8 operand[kAhead];
#pragma unroll
      for (int x = 0; x < kAhead; ++x) operand[x] = tile_rows<KIND, T>(lds, at_rows, 0, x);
      float16_t c = zero16(), odd = zero16();  // (two sums, as in the dq kernel: S has to come out the same)
      if (second) {  // dP comes out less dO . O
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const float4_t d = stat(x);
#pragma unroll
          for (int j = 0; j < 4; ++j) c[4 * x + j] = d[j];
        }
      }
#pragma unroll
      for (int x = 0; x < NKS; ++x) {
        __builtin_amdgcn_sched_barrier(0);
        if (x & 1) {
          odd = M::mfma(operand[x % kAhead], own[x], odd);
        } else {
          c = M::mfma(operand[x % kAhead], own[x], c);
        }
        if (x + kAhead < NKS) operand[x % kAhead] = tile_rows<KIND, T>(lds, at_rows, 0, x + kAhead);
      }
      c += odd;
      auto columns = [&](int x) { return tile_columns<KIND, T>(lds, at_columns, 16 * (x & 1), x >> 1); };
#pragma unroll
      for (int x = 0; x < kAhead; ++x) operand[x] = columns(x);
      float4_t* const mine = hand + lane_now();
      if (!second) {
        if (t < plain_lo || t > plain_hi) {
          const int lane = lane_now();
          const int base = kWideTile * t + 4 * (lane >> 5);  // queries base + 8 c + j
          const int key = wave_key_lo + (lane & 31);         // this lane's key position in the sequence
          const int first = key - ctx - base;
          int last = n_q - 1;
          if (p.window_left >= 0) last = min(last, key - ctx + p.window_left);
          last = live ? last - base : -1;
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int q = 8 * (e >> 2) + (e & 3);
            c[e] = q >= first && q <= last ? c[e] : kWideNegInf;
          }
        }
        // (a query without visible keys has +inf as its log-sum-exp: exp2(-inf) = 0 either way)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const float4_t lse = stat(x);
          float4_t pe;
#pragma unroll
          for (int j = 0; j < 4; ++j) pe[j] = c[4 * x + j] = fast_exp2(c[4 * x + j] * p.scale_log2e - lse[j]);
          mine[x * kWave] = pe;
        }
        handed_barrier();
      } else {
        handed_barrier();
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const float4_t pe = mine[x * kWave];
#pragma unroll
          for (int j = 0; j < 4; ++j) c[4 * x + j] *= pe[j];
        }
      }
      add_products<KIND, NB, kAhead>(wide_weights<KIND>(c), operand, columns, acc);
    };
    fetched_barrier();  // the tiles' previous readers (an earlier sequence of this block) are done
    if (steps > 0) fetch(0);
    for (int i = 0; i < rounds; i += 2) {
      step(i, 0);
      if (i + 1 < rounds) step(i + 1, 1);
    }
  }

  if constexpr (P > 1) {
    // the other parts' sums to part 0, in a fixed order: a float4 per lane at a time, lanes next to each other
    float4_t* const sums = reinterpret_cast<float4_t*>(wide_lds) + part_wave * kWave + lane_now();
    constexpr int kStep = L::kPartWaves * kWave, kFours = 4 * NB;  // (per part)
    __syncthreads();  // the tiles' last readers are done
    if (part > 0) {
#pragma unroll
      for (int x = 0; x < kFours; ++x) {
        const int nb = x >> 2, c = 4 * (x & 3);
        sums[((part - 1) * kFours + x) * kStep] = float4_t{acc[nb][c], acc[nb][c + 1], acc[nb][c + 2], acc[nb][c + 3]};
      }
    }
    __syncthreads();
    if (part == 0) {
#pragma unroll
      for (int other = 0; other < P - 1; ++other) {
#pragma unroll
        for (int x = 0; x < kFours; ++x) {
          const float4_t theirs = sums[(other * kFours + x) * kStep];
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[x >> 2][4 * (x & 3) + j] += theirs[j];
        }
      }
    }
  }
  handed_barrier();  // (every wave has read its last tile, or the sums)
  if (part > 0) return;

  // every gradient element is written, also the zeros of keys no query sees; in 16 bits through LDS, as whole rows
  const int l = lane_now();
  const int64_t first_row = r0 + 32 * wave;
  void* const out = second ? p.grad_k : p.grad_v;
  const float f = second ? p.scale : 1.0f;
  if (p.grad_dtype == ARENO_DT_F32) {
    const int64_t out_row = first_row + (l & 31);
    if (out_row < p.k_tokens) {
      const int64_t elem = (out_row * p.kv_heads + kvh) * D + 4 * (l >> 5);
#pragma unroll
      for (int x = 0; x < 4 * NB; ++x) {
        const int nb = x >> 2, c = 4 * (x & 3);
        GradStore<float>{}(out, elem + 8 * x, acc[nb][c] * f, acc[nb][c + 1] * f, acc[nb][c + 2] * f, acc[nb][c + 3] * f);
      }
    }
  } else {
    using Stage = RowStage<4 * NB>;
    char* const stage = wide_lds + part_wave * (32 * Stage::kRowBytes);
    static_assert(L::kPartWaves * 32 * Stage::kRowBytes <= L::kTiles, "the rows' place");
#pragma unroll
    for (int x = 0; x < 4 * NB; ++x) {
      const int nb = x >> 2, c = 4 * (x & 3);
      Stage::put(stage, l & 31, x, l >> 5, pack_pair<KIND>(acc[nb][c] * f, acc[nb][c + 1] * f), pack_pair<KIND>(acc[nb][c + 2] * f, acc[nb][c + 3] * f));
    }
    Stage::template take<32>(stage, l, [&](int r, int chunk, uint4_t w) {
      if (first_row + r < p.k_tokens) *reinterpret_cast<uint4_t*>(static_cast<char*>(out) + (((first_row + r) * p.kv_heads + kvh) * D + 8 * chunk) * 2) = w;
    });
  }
}

template <int KIND, int D, int KW, int P>
BwdLaunch launch_of() {
  using L = WideShape<D, KW, P>;
  const bwd_fn fn = bwd_mfma32_wide_dkv_kernel<KIND, D, KW, P>;
  static std::atomic<uint64_t> allowed_on{0};
  if (!allow_lds<L::kLdsBytes>(reinterpret_cast<const void*>(fn), allowed_on)) return BwdLaunch{nullptr, 0, 0, 0};
  return BwdLaunch{fn, L::kLdsBytes, L::kThreads, L::kKeys};
}
template <int KIND, int D>
BwdLaunch launch_of(int parts) {
  return parts == 2 ? launch_of<KIND, D, 1, 2>() : launch_of<KIND, D, 2, 1>();
}

}  // namespace

template <int KIND, int D>
BwdLaunch dq_launch_of() {
  using L = WideDqShape<D>;
  const bwd_fn fn = bwd_mfma32_wide_dq_kernel<KIND, D>;
  static std::atomic<uint64_t> allowed_on{0};
  if (!allow_lds<L::kLdsBytes>(reinterpret_cast<const void*>(fn), allowed_on)) return BwdLaunch{nullptr, 0, 0, 0};
  return BwdLaunch{fn, L::kLdsBytes, kWideDqWaves * kWave, L::kRows};
}
BwdLaunch dq32_wide_launch(const BwdParams& p) {
  if (p.head_dim == 192) return p.dtype == ARENO_DT_BF16 ? dq_launch_of<KV_BF16, 192>() : dq_launch_of<KV_F16, 192>();
  return p.dtype == ARENO_DT_BF16 ? dq_launch_of<KV_BF16, 256>() : dq_launch_of<KV_F16, 256>();
}
// The dkv kernel's shape: blocks of 64 keys, or of 32 with the stream in two parts, which end sooner where the launch is its
// longest blocks; with more than three rounds of workgroups what counts is the tiles' traffic, half of it per key in the larger
// blocks (and where blocks hold several sequences, the waves that wait in these).  The backward in us, in one part and two
// (what the 16-row kernels took); in brackets blocks of 32, steps: heads of 192: 16 / 16, 5 x 34 tokens (96, 1) 39.1, 31.0 (47.6); 24 / 8,
// 2 x 1 580 (792, 147) 683, 455 (599); 32 / 8, 248 x 12 (744, 12) 214, 170 (209); 8 / 2, 15 x 1 066 (1 000, 132) 764, 622 (678); 6 / 6, 8 x 1 926
// (2 892, 60) 687, 744 (725); of 256: 6 / 6,
// 4 x 535 (402, 16) 105, 93 (176); 32 / 8, 2 x 720 (360, 88) 356, 252 (633); 8 / 1, 1 x 1 000, window 512 (32, 136) 367, 216 (911); 12 / 4, 5 x 1 306 (820, 120)
// 539, 664 (978); 32 / 8, 6 x 1 161 (1 744, 144) 1 227, 1 268 (1 612); 28 / 4, 8 x 2 048 (2 048, 448) 3 684, 3 831 (4 569).  Over 1 971 launches 0.5 % more than the better one.
int dkv32_wide_parts(const BwdParams& p) {
  const int64_t seqs = std::max<int64_t>(p.num_seqs, 1), mean = std::max<int64_t>(p.q_tokens / seqs, 1), blocks = (p.k_tokens + 31) / 32 * p.kv_heads;
  const int64_t seen = p.window_left >= 0 ? std::min<int64_t>(mean, p.window_left + int64_t{32}) : mean;
  const int64_t steps = std::max<int64_t>(seen / kWideTile, 1) * (p.q_heads / p.kv_heads) * std::min(seqs, 1 + 31 / mean);
  return steps >= (blocks > 256 ? 4 : mean > 32 ? 1 : 2) && blocks <= (mean < 32 && steps >= 7 ? 2048 : p.head_dim == 192 ? 1024 : 512) ? 2 : 1;
}
BwdLaunch dkv32_wide_launch(const BwdParams& p, int64_t* groups) {
  int parts = dkv32_wide_parts(p);
  // (ARENO_BACKWARD_PARTS=1|2 fixes it, for tests and timing)
  if (fixed_by("ARENO_BACKWARD_PARTS", "1")) parts = 1;
  if (fixed_by("ARENO_BACKWARD_PARTS", "2")) parts = 2;
  BwdLaunch launch;
  if (p.head_dim == 192) {
    launch = p.dtype == ARENO_DT_BF16 ? launch_of<KV_BF16, 192>(parts) : launch_of<KV_F16, 192>(parts);
  } else {
    launch = p.dtype == ARENO_DT_BF16 ? launch_of<KV_BF16, 256>(parts) : launch_of<KV_F16, 256>(parts);
  }
  *groups = (p.k_tokens + launch.rows - 1) / std::max(launch.rows, 1);
  return launch;
}

}  // namespace areno
