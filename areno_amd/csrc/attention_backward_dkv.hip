// dK and dV of the causal varlen / dense attention ops on 32 x 32 x 16 matrix products (gfx950): 16-bit inputs, head dims
// 64 and 128.  The second launch of attention_backward_mfma.hip; reads the rows' statistics that the dq kernel left.  The reference: areno/accel/csrc/attention.cu:244-524.
//
// A wave owns 32 packed key rows of one kv head: K and V of them as B operands and both sums in registers.  It goes
// through the query rows that may see them, for every q head of the group, in tiles of 32 that the memory pipe puts into
// LDS:  S = Q . K^T,  dP = dO . V^T - dO . O,  P = exp2(scale S - lse),  dS = P * dP,  dV^T += dO^T . P,  dK^T += Q^T . dS.  A
// C tile of the first two is the B operand of the last two as it lies (mfma32_tiles.hpp).  S is summed in the order of the
// dq kernel with 32 rows per wave; the one with 16 sums it in another, so that behind it S and the log-sum-exp differ by
// S's own roundings (32 bits in both).
//
// A workgroup is four waves: KW waves own neighbouring keys and share a stream of tiles, and P such parts own the same keys
// and take every P-th tile of the stream each; the sums of parts 1 .. P - 1 go to part 0 through LDS at the end, in a fixed
// order.  (4, 1) for large launches, two workgroups per compute unit; (2, 2); (1, 4) for small ones, whose time is that of
// their longest block: there a wave has its tiles for itself, no barrier, and 512 registers.  In a (1, 4) launch of about
// one workgroup per compute unit it takes block i and then block `blocks - 1 - i`: their costs add up to the same.  (1, 1) is
// a workgroup of one wave, for many short sequences: in a block of 128 keys each of them is a stream that one wave of four
// computes on while all wait at its barriers.
//
// Bound: (4, 1) by the matrix cores (busy 58 % of the cycles, at the clock that they then leave, 1.7 GHz) and LDS; (1, 4) by
// what one wave issues, 350 instructions and 34 products of 32 cycles in 2 500.  Where the time was: 16 x 16 x 32 products
// read an operand of 1 KB each where these read one per two; the compiler waited for every operand right behind its read;
// the spilled addresses of a step (a scratch load waits for all the fetches in front of it).  Forward and backward, us, with the
// 16-row kernel and this (the kernel by itself under the profiler): 4 x 4 096 tokens, 32 / 8 heads of 128, bf16: 2 886, 2 357 (1 763, 1 091);
// 2 x 2 048, 28 / 4 heads: 394, 324 (256, 143).
#include <algorithm>
#include <atomic>

#include "attention_backward.hpp"
#include "mfma32_tiles.hpp"

namespace areno {
namespace {

constexpr int kDkvTile = 32;  // query rows per step
constexpr float kDkvNegInf = -__builtin_huge_valf();

template <int D, int KW, int P>
struct Dkv32Shape {
  using Tile = LdsTile<D, kDkvTile, KW>;
  static constexpr int kWaves = KW * P;
  static constexpr int kThreads = kWaves * kWave;
  static constexpr int kKeys = 32 * KW;                        // key rows of a block
  static constexpr int kStat = kDkvTile * 2 * 4;               // the rows' statistics
  static constexpr int kBuffer = 2 * Tile::kBytes + kStat;     // Q, dO
  static constexpr int kPart = 2 * kBuffer;
  static constexpr int kSums = (P - 1) * KW * D * 32 * 2 * 4;  // what parts 1 .. P - 1 hand to part 0
  static constexpr int kLdsBytes = P * kPart > kSums ? P * kPart : kSums;
};
extern __shared__ __attribute__((aligned(1024))) char dkv32_lds[];

template <int KIND, int D, int KW, int P, int OCC>
__global__ __launch_bounds__((Dkv32Shape<D, KW, P>::kThreads)) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void bwd_mfma32_dkv_kernel(BwdParams p) {
  using M = Mfma32<KIND>;
  using V8 = typename M::vec8;
  using L = Dkv32Shape<D, KW, P>;
  using T = typename L::Tile;
  constexpr int NKS = D / 16, NB = D / 32, NF = T::kFetches;
  constexpr bool kTight = D > 64 && OCC > 1;  // sums, K and V and the scores leave 32 registers for all the rest

  ask_for_arguments(p, p.k_order);
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave_of_block = uniform(tid >> 6);
  const int part = wave_of_block / KW, wave = wave_of_block % KW;
  const int l32 = lane & 31, half = lane >> 5;
  const int kvh = static_cast<int>(blockIdx.x % static_cast<unsigned>(p.kv_heads));
  const int group = p.q_heads / p.kv_heads;
  const int k_blocks = static_cast<int>((p.k_tokens + L::kKeys - 1) / L::kKeys);
  const int wg = static_cast<int>(blockIdx.x / static_cast<unsigned>(p.kv_heads));
  // (launched with a workgroup per pair of blocks, or with one per block: then in cost order, one block each)
  const bool paired = gridDim.x / static_cast<unsigned>(p.kv_heads) < static_cast<unsigned>(k_blocks);
  const int first_block = paired ? wg : uniform(block_in_launch_order(wg, p.k_order, L::kKeys, false));

  // (with the part's place: a multiple of 256, which the reads' exclusive-ors leave alone)
  static_assert(L::kPart % 256 == 0, "the parts' places");
  uint32_t at_rows = T::rows_base(l32, half) + part * L::kPart, at_columns = T::columns_base(lane) + part * L::kPart;
  const uint32_t lds0 = lds_address(dkv32_lds) + part * L::kPart;
  const uint32_t stride = static_cast<uint32_t>(p.q_heads) * (D * 2);
  // Fetch f of a wave fills kFetchRows rows; the chunk a lane fetches is the one that belongs where its bytes land.  A wave
  // that fetches whole tiles keeps its offsets, others work out their few anew.
  constexpr int kFetchRows = 64 / T::kChunksPerRow;
  auto fetch_row = [&](int f, int lane) { return kFetchRows * (NF * wave + f) + lane / T::kChunksPerRow; };
  auto fetch_offset = [&](int f, int lane) {
    const int r = fetch_row(f, lane);
    return static_cast<uint32_t>(r) * stride + static_cast<uint32_t>((lane % T::kChunksPerRow) ^ T::twist(r)) * 16u;
  };
  uint32_t kept_offset[NF];
  if constexpr (KW == 1) {
#pragma unroll
    for (int f = 0; f < NF; ++f) kept_offset[f] = fetch_offset(f, lane);
  }

  for (int turn = 0; turn < 2; ++turn) {
    const int block = turn == 0 ? first_block : k_blocks - 1 - first_block;
    // (no second block without pairs, and none for the middle one of an odd number of blocks)
    if (turn == 1 && (!paired || block <= first_block)) break;
    const int64_t r0 = static_cast<int64_t>(block) * L::kKeys;
    const int64_t block_end = r0 + L::kKeys < p.k_tokens ? r0 + L::kKeys : p.k_tokens;
    const int64_t row = r0 + 32 * wave + l32;  // this lane's key row (a column of the products)
    const bool row_exists = row < p.k_tokens;
    const int64_t row_elem = (row * p.kv_heads + kvh) * D;
    V8 kop[NKS], vop[NKS];
    {
      uint4_t kw[NKS], vw[NKS];
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) kw[ks] = vw[ks] = uint4_t{0u, 0u, 0u, 0u};
      if (row_exists) {
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          const int64_t off = (row_elem + 16 * ks + 8 * half) * 2;
          kw[ks] = load16(p.k, off);
          vw[ks] = load16(p.v, off);
        }
      }
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        // (waited for here: left to their first use inside the loop, that wait would cover every tile's fetches as well)
        if constexpr (OCC == 1) {
          asm volatile("" : "+a"(kw[ks]), "+a"(vw[ks]));  // (in accumulation registers, where the products read them as they are)
        } else {
          asm volatile("" : "+v"(kw[ks]), "+v"(vw[ks]));
        }
        kop[ks] = __builtin_bit_cast(V8, kw[ks]);
        vop[ks] = __builtin_bit_cast(V8, vw[ks]);
      }
    }
    float16_t acc_k[NB], acc_v[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc_k[nb] = acc_v[nb] = zero16();

    int s = uniform(seq_of_row(p.cu_k, p.num_seqs, r0));
    for (int64_t sk0 = uniform(p.cu_k[s]), sk1; s < p.num_seqs && sk0 < block_end; ++s, sk0 = sk1) {
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
      const int t0 = i_lo / kDkvTile, t1 = i_hi / kDkvTile;
      const int tiles = t1 - t0 + 1;
      // the stream: tiles of every q head of the group, head by head; this part takes steps part, part + P, ...
      const int stream_steps = tiles * group;
      const int steps = (stream_steps - part + P - 1) / P;  // this part's
      const int rounds = (stream_steps + P - 1) / P;        // the longest part's: every part keeps the barriers of all
      // the step whose tile is fetched next: its tile, where its rows of Q (and, a fixed way off, of dO) and statistics lie
      const int64_t tile_bytes = static_cast<int64_t>(kDkvTile) * stride;
      const int64_t head_bytes = D * 2 - tiles * tile_bytes, head_stats = (p.q_tokens - static_cast<int64_t>(tiles) * kDkvTile) * 8;
      const int64_t to_grad = static_cast<const char*>(p.grad_out) - static_cast<const char*>(p.q);
      int tile = t0 + part, ahead = tile;
      const char* q_ahead = static_cast<const char*>(p.q) + q_first * stride + kvh * group * (D * 2) + tile * tile_bytes;
      const char* stat_ahead = reinterpret_cast<const char*>(p.row_stats) + ((kvh * group) * p.q_tokens + q_first + tile * kDkvTile) * 8;
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
      int seen_lo = 0, seen_hi = t1, plain_lo = max(wave_key_hi - ctx + kDkvTile - 1, 0) / kDkvTile, plain_hi = n_q / kDkvTile - 1;
      if constexpr (KW > 1) {
        seen_lo = max(wave_key_lo - ctx, 0) / kDkvTile;
        if (p.window_left >= 0) seen_hi = wave_key_hi + p.window_left - ctx < 0 ? -1 : (wave_key_hi + p.window_left - ctx) / kDkvTile;
        if (!wave_live) seen_hi = -1;
      }
      if (p.window_left >= 0) {
        const int reach = wave_key_lo + p.window_left - ctx - (kDkvTile - 1);
        plain_hi = reach < 0 ? -1 : min(plain_hi, reach / kDkvTile);
      }
      if (!wave_full) plain_hi = -1;
      auto fetch = [&](int buf) {
        const int last = min(n_q - ahead * kDkvTile, kDkvTile) - 1;  // rows behind the sequence's last repeat it
        const char* const qb = q_ahead;
        const char* const gb = q_ahead + to_grad;
        const char* const sb = stat_ahead;
        const uint32_t dst = lds0 + static_cast<uint32_t>(buf * L::kBuffer + wave * (NF * 1024));
        const int lane = lane_now();
        if (last == kDkvTile - 1) {
#pragma unroll
          for (int f = 0; f < NF; ++f) {
            const uint32_t off = KW == 1 ? kept_offset[f] : fetch_offset(f, lane);
            fetch_to_lds(qb, off, dst + f * 1024);
            fetch_to_lds(gb, off, dst + T::kBytes + f * 1024);
          }
        } else {
#pragma unroll
          for (int f = 0; f < NF; ++f) {
            const uint32_t back = static_cast<uint32_t>(max(fetch_row(f, lane) - last, 0)) * stride;
            const uint32_t off = (KW == 1 ? kept_offset[f] : fetch_offset(f, lane)) - back;
            fetch_end_to_lds(qb, off, dst + f * 1024);
            fetch_end_to_lds(gb, off, dst + T::kBytes + f * 1024);
          }
        }
        if (wave == 0) {
          fetch_words_to_lds(sb, static_cast<uint32_t>(min(lane & 31, last)) * 8u + (lane >> 5) * 4u,
                             lds0 + static_cast<uint32_t>(buf * L::kBuffer + 2 * T::kBytes));
        }
        ahead += P;
        q_ahead += P * tile_bytes;
        stat_ahead += P * kDkvTile * 8;
        to_next_heads();
      };
      auto step = [&](int i, int buf) {
        // the step's tile (asked for a step ago) is there, and every wave of the part has left the one before
        if constexpr (KW == 1) {
          fetched();
        } else {
          fetched_barrier();
        }
        if (i + 1 < steps) fetch(buf ^ 1);
        if (KW > 1 && i >= steps) return;
        const int t = tile;
        tile += P;
        while (tile > t1) tile -= tiles;
        if (KW > 1 && (t < seen_lo || t > seen_hi)) return;
        // (where registers are short the addresses of a step are worked out where they are used)
        if constexpr (OCC > 1) asm volatile("" : "+v"(at_rows), "+v"(at_columns));
        char* const q_lds = dkv32_lds + buf * L::kBuffer;
        char* const g_lds = q_lds + T::kBytes;
        // The products' operands come out of LDS in one stream, each read kAhead products in front of its own (left
        // alone the compiler reads one, waits for it and reads the next): rows of Q and of dO, columns of dO and of Q.
        constexpr int kAhead = kTight ? 2 : 8;
        auto read = [&](int x) {
          if (x < NKS) return tile_rows<KIND, T>(q_lds, at_rows, 0, x);
          if (x < 2 * NKS) return tile_rows<KIND, T>(g_lds, at_rows, 0, x - NKS);
          const int y = x - 2 * NKS;
          if (y < 2 * NB) return tile_columns<KIND, T>(g_lds, at_columns, 16 * (y / NB), y % NB);
          return tile_columns<KIND, T>(q_lds, at_columns, 16 * (y / NB - 2), y % NB);
        };
        constexpr int kReads = 2 * NKS + 4 * NB;
        V8 operand[kAhead];
        // The statistics of the rows that this lane has values of, the log-sum-exps and (128 bytes on) -(dO . O): of rows
        // 8 c + 4 (lane / 32) .. + 3 at 32 c.  P's exponent is rounded once, in its fma: put into the products as a
        // contraction step (a row's log-sum-exp over the scale in three bf16 parts) it was rounded three times, took two
        // products more and no less time: backward of 4 x 4 096 tokens, 32 / 8 heads of 128, bf16: 1 851 -> 1 812 us; 12 x 100 .. 900,
        // 32 / 8 heads of 64: 123 -> 120.
        const char* const stats = q_lds + 2 * T::kBytes + part * L::kPart + 16 * (lane_now() >> 5);
        auto stat = [&](int which, int c) { return *reinterpret_cast<const float4_t*>(stats + 128 * which + 32 * c); };
#pragma unroll
        for (int x = 0; x < kAhead; ++x) operand[x] = read(x);
        float16_t sc = zero16(), dp;
        float4_t lse[4];  // (each read one group of rows in front of its use)
#pragma unroll
        for (int x = 0; x < NKS; ++x) {
          __builtin_amdgcn_sched_barrier(0);
          sc = M::mfma(operand[x % kAhead], kop[x], sc);
          operand[x % kAhead] = read(x + kAhead);
          // (dP comes out less dO . O)
#pragma unroll
          for (int c = 4 * x / NKS; c < 4 * (x + 1) / NKS; ++c) {
            const float4_t start = stat(1, c);
#pragma unroll
            for (int j = 0; j < 4; ++j) dp[4 * c + j] = start[j];
          }
        }
        if constexpr (!kTight) lse[0] = stat(0, 0);
        if (t < plain_lo || t > plain_hi) {
          const int lane = lane_now();
          const int base = kDkvTile * t + 4 * (lane >> 5);  // queries base + 8 c + j
          const int key = wave_key_lo + (lane & 31);        // this lane's key position in the sequence
          const int first = key - ctx - base;
          int last = n_q - 1;
          if (p.window_left >= 0) last = min(last, key - ctx + p.window_left);
          last = live ? last - base : -1;
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int q = 8 * (e >> 2) + (e & 3);
            sc[e] = q >= first && q <= last ? sc[e] : kDkvNegInf;
          }
        }
        V8 pop[2], dsop[2];
        uint32_t w[8], dw[8];
        // (a query without visible keys has +inf as its log-sum-exp: exp2(-inf) = 0)
#pragma unroll
        for (int x = 0; x < NKS; ++x) {
          __builtin_amdgcn_sched_barrier(0);
          dp = M::mfma(operand[(NKS + x) % kAhead], vop[x], dp);
          operand[(NKS + x) % kAhead] = read(NKS + x + kAhead);
          if (!kTight && 4 * (x + 1) % NKS == 0 && x + 1 < NKS) lse[4 * (x + 1) / NKS] = stat(0, 4 * (x + 1) / NKS);
          if constexpr (!kTight) {  // the exponentials between the products of dP
#pragma unroll
            for (int e = 16 / NKS * x; e < 16 / NKS * (x + 1); e += 2) {
              sc[e] = fast_exp2(__builtin_fmaf(sc[e], p.scale_log2e, -lse[e >> 2][e & 3]));
              sc[e + 1] = fast_exp2(__builtin_fmaf(sc[e + 1], p.scale_log2e, -lse[e >> 2][(e & 3) + 1]));
              w[e / 2] = pack_pair<KIND>(sc[e], sc[e + 1]);
            }
          }
        }
        if constexpr (kTight) {  // (P and dS at once, so that packed ones take the registers of those they come from)
          lse[0] = stat(0, 0);
#pragma unroll
          for (int e = 0; e < 16; e += 2) {
            __builtin_amdgcn_sched_barrier(0);
            if (e % 4 == 0 && e < 12) lse[e / 4 + 1] = stat(0, e / 4 + 1);
            const float p0 = fast_exp2(__builtin_fmaf(sc[e], p.scale_log2e, -lse[e >> 2][e & 3]));
            const float p1 = fast_exp2(__builtin_fmaf(sc[e + 1], p.scale_log2e, -lse[e >> 2][(e & 3) + 1]));
            w[e / 2] = pack_pair<KIND>(p0, p1);
            dw[e / 2] = pack_pair<KIND>(p0 * dp[e], p1 * dp[e + 1]);
          }
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) pop[b] = __builtin_bit_cast(V8, uint4_t{w[4 * b], w[4 * b + 1], w[4 * b + 2], w[4 * b + 3]});
#pragma unroll
        for (int x = 0; x < 2 * NB; ++x) {
          constexpr int kFrom = 2 * NKS;
          __builtin_amdgcn_sched_barrier(0);
          acc_v[x % NB] = M::mfma(operand[(kFrom + x) % kAhead], pop[x / NB], acc_v[x % NB]);
          if (kFrom + x + kAhead < kReads) operand[(kFrom + x) % kAhead] = read(kFrom + x + kAhead);
          if constexpr (!kTight) {  // dS between the products of dV
#pragma unroll
            for (int e = 8 / NB * x; e < 8 / NB * (x + 1); e += 2) dw[e / 2] = pack_pair<KIND>(sc[e] * dp[e], sc[e + 1] * dp[e + 1]);
          }
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) dsop[b] = __builtin_bit_cast(V8, uint4_t{dw[4 * b], dw[4 * b + 1], dw[4 * b + 2], dw[4 * b + 3]});
#pragma unroll
        for (int x = 0; x < 2 * NB; ++x) {
          constexpr int kFrom = 2 * NKS + 2 * NB;
          __builtin_amdgcn_sched_barrier(0);
          acc_k[x % NB] = M::mfma(operand[(kFrom + x) % kAhead], dsop[x / NB], acc_k[x % NB]);
          if (kFrom + x + kAhead < kReads) operand[(kFrom + x) % kAhead] = read(kFrom + x + kAhead);
        }
      };
      // the tiles' previous readers (an earlier sequence of this block, the sums of the block before) are done
      fetched_barrier();
      if (steps > 0) fetch(0);
      const int turns = KW == 1 ? steps : rounds;
      for (int i = 0; i < turns; i += 2) {
        step(i, 0);
        if (i + 1 < turns) step(i + 1, 1);
      }
    }

    if constexpr (P > 1) {
      // the other parts' sums to part 0, in a fixed order: a float4 per lane at a time, lanes next to each other
      float4_t* const sums = reinterpret_cast<float4_t*>(dkv32_lds) + wave * kWave + lane_now();
      constexpr int kStep = KW * kWave, kFours = 8 * NB;  // (per part)
      __syncthreads();  // the tiles' last readers are done
      if (part > 0) {
        float4_t* const mine = sums + (part - 1) * (kFours * kStep);
#pragma unroll
        for (int x = 0; x < 4 * NB; ++x) {
          const int nb = x >> 2, c = 4 * (x & 3);
          mine[x * kStep] = float4_t{acc_k[nb][c], acc_k[nb][c + 1], acc_k[nb][c + 2], acc_k[nb][c + 3]};
          mine[(4 * NB + x) * kStep] = float4_t{acc_v[nb][c], acc_v[nb][c + 1], acc_v[nb][c + 2], acc_v[nb][c + 3]};
        }
      }
      __syncthreads();
      if (part == 0) {
#pragma unroll
        for (int other = 0; other < P - 1; ++other) {
          const float4_t* const theirs = sums + other * (kFours * kStep);
#pragma unroll
          for (int x = 0; x < 4 * NB; ++x) {
            const float4_t dk = theirs[x * kStep], dv = theirs[(4 * NB + x) * kStep];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              acc_k[x >> 2][4 * (x & 3) + j] += dk[j];
              acc_v[x >> 2][4 * (x & 3) + j] += dv[j];
            }
          }
        }
      }
    }

    // Every gradient element is written, also the zeros of keys no query sees.  At head dim 64 16-bit ones as whole rows, through
    // LDS (16 x 20 .. 600 tokens, 16 heads: 34.4 -> 33.2 us); at 128 that spilled registers of the loop in (4, 1) and (2, 2),
    // and took the one wave that stores longer in (1, 4) (2 x 2 048, 28 / 4 heads: 139.4 -> 142.2).
    constexpr bool kWholeRows = D == 64;
    if constexpr (KW > 1 && kWholeRows) handed_barrier();  // (the other waves have read their last tile, or the sums)
    const int lane_ = lane_now();
    const int64_t first_row = r0 + 32 * wave, out_row = first_row + (lane_ & 31);
    if (kWholeRows && p.grad_dtype != ARENO_DT_F32) {
      if (part == 0) {
        using Stage = RowStage<4 * NB>;
        char* const stage = dkv32_lds + wave * (32 * Stage::kRowBytes);
        auto out = [&](void* grad, const float16_t (&acc)[NB], float f) {
#pragma unroll
          for (int x = 0; x < 4 * NB; ++x) {
            const int nb = x >> 2, c = 4 * (x & 3);
            Stage::put(stage, lane_ & 31, x, lane_ >> 5, pack_pair<KIND>(acc[nb][c] * f, acc[nb][c + 1] * f), pack_pair<KIND>(acc[nb][c + 2] * f, acc[nb][c + 3] * f));
          }
          Stage::template take<32>(stage, lane_, [&](int r, int chunk, uint4_t w) {
            if (first_row + r < p.k_tokens) *reinterpret_cast<uint4_t*>(static_cast<char*>(grad) + (((first_row + r) * p.kv_heads + kvh) * D + 8 * chunk) * 2) = w;
          });
        };
        out(p.grad_k, acc_k, p.scale);
        out(p.grad_v, acc_v, 1.0f);
      }
    } else if (part == 0 && out_row < p.k_tokens) {
      const int64_t out_elem = (out_row * p.kv_heads + kvh) * D + 4 * (lane_ >> 5);
      auto out = [&](auto store) {
#pragma unroll
        for (int x = 0; x < 4 * NB; ++x) {
          const int nb = x >> 2, c = 4 * (x & 3);
          store(p.grad_k, out_elem + 8 * x, acc_k[nb][c] * p.scale, acc_k[nb][c + 1] * p.scale, acc_k[nb][c + 2] * p.scale, acc_k[nb][c + 3] * p.scale);
          store(p.grad_v, out_elem + 8 * x, acc_v[nb][c], acc_v[nb][c + 1], acc_v[nb][c + 2], acc_v[nb][c + 3]);
        }
      };
      if constexpr (!kWholeRows) {
        store_grads<typename M::elem>(p.grad_dtype, out);
      } else {
        out(GradStore<float>{});
      }
    }
  }
}

template <int KIND, int D, int KW, int P, int OCC>
BwdLaunch launch_of() {
  using L = Dkv32Shape<D, KW, P>;
  const bwd_fn fn = bwd_mfma32_dkv_kernel<KIND, D, KW, P, OCC>;
  static std::atomic<uint64_t> allowed_on{0};
  if (!allow_lds<L::kLdsBytes>(reinterpret_cast<const void*>(fn), allowed_on)) return BwdLaunch{nullptr, 0, 0, 0};
  return BwdLaunch{fn, L::kLdsBytes, L::kThreads, L::kKeys};
}
constexpr int kLoneWave = 0;  // for the parts: one wave
template <int KIND, int D>
BwdLaunch launch_of(int parts) {
  if (parts == kLoneWave) return launch_of<KIND, D, 1, 1, D == 64 ? 2 : 1>();
  if (parts == 4) return launch_of<KIND, D, 1, 4, 1>();
  if (parts == 2) return launch_of<KIND, D, 2, 2, 2>();
  return launch_of<KIND, D, 4, 1, 2>();
}

constexpr int64_t kComputeUnits = 256;

}  // namespace

// The shape, from the launch's size (blocks of 32 keys of a kv head) and the steps of a block's streams, for sequences of the
// mean length, of which a window shows a block of keys its own queries and as many behind them.  Up to a workgroup per
// compute unit a launch is its longest block: four parts, unless its streams are so few steps that handing the sums
// over takes longer.  Blocks of several sequences are one wave's: in a wider one each sequence is a stream that one wave
// computes on while the others wait.  The more workgroups there are the longer a stream has to be for four parts and for two,
// and four pay only where a few blocks' streams are far longer than the rest (not in a window); one part, which two waves
// per SIMD share, is for launches that fill the chip many times over, sooner where no block of 128 holds two sequences.
// Lines drawn through 8 753 launches of 1 .. 1 000 sequences of 1 .. 4 096 tokens, ten head ratios, equal and ragged lengths,
// windows: the choice takes 0.8 % longer than the best of all shapes, and 3 % longer than the 16-row kernels in one.  The backward
// in us, sequences x tokens (blocks, steps):
//   one wave, two parts, four.  D = 128: 16 / 16 heads, 1 x 26 (16, 1) 11.1, 12.5, 14.3; 6 / 6, 6 x 64 (72, 2) 13.9, 16.6, 16.8; 24 / 8, 8 x 160 (328, 15)
// 54.6, 48.5, 45.9; 6 / 6, 5 x 474 (450, 14) 45.0, 43.3, 49.7; 32 / 2, 347 x 14 (316, 48) 208, 198, 163; 8 / 1, 29 x 768, window 512 (696, 136) 258, 197, 245;
// 32 / 2, 37 x 448 (1 036, 224) 566, 431, 538; 32 / 8, 2 x 1 380 (696, 172) 266, 230, 172.  D = 64: 28 / 4, 9 x 617 (696, 133) 175, 130, 110; 24 / 8, 36 x 75
// (680, 6) 39.6, 36.5, 44.3; 28 / 4, 12 x 347 (524, 70) 155, 112, 87; 28 / 4, 38 x 92 (440, 14) 49.0, 43.6, 47.1; 32 / 8, 2 x 2 048 (1 024, 256) 220, 172, 172.
//   one wave, one part, two (the 16-row kernels).  D = 128: 16 / 16, 4 096 x 8 (16 384, 4) 717, 854, 899 (948); 512 x 16 (4 096, 2) 111, 125, 135 (133); 32 x 128 (2 048, 4) 55.0,
// 50.6, 56.5 (57.3); 32 / 8, 61 x 128 (1 952, 16) 139, 127, 133 (155); 16 / 8, 196 x 128 (6 272, 8) 279, 259, 272; 16 / 16, 67 x 180, window 128 (6 032, 5) 184, 173, 191.
// D = 64: 16 / 16, 4 096 x 8 335, 485, 518 (481); 512 x 8 (2 048, 4) 42, 60, 64 (66); 512 x 4 (1 024, 8) 49, 78, 64 (71); 11 x 716 (3 952, 22) 124, 109, 123; 361 x 132, window 128
// (23 840, 4) 432, 408, 460.
//   one part, two, four.  D = 128: 28 / 4, 8 x 2 048 (2 048, 448) 997, 926, 980 (1 182); 32 / 8, 4 x 4 096 (4 096, 512) 1 822, 1 864, 2 027 (2 382); D = 64: 28 / 4, 3 x 4 096
// (1 536, 896) 887, 704, 764 (1 008).
BwdLaunch dkv32_launch(const BwdParams& p, int64_t* groups) {
  const int64_t blocks = (p.k_tokens + 31) / 32, workgroups = blocks * p.kv_heads;
  const int64_t seqs = std::max<int64_t>(p.num_seqs, 1), mean = std::max<int64_t>(p.q_tokens / seqs, 1), group = p.q_heads / p.kv_heads;
  const int64_t seen = p.window_left >= 0 ? std::min<int64_t>(mean, p.window_left + int64_t{32}) : mean;
  const int64_t steps = std::max<int64_t>(seen / kDkvTile, 1) * group * std::min(seqs, 1 + 31 / mean);  // (a block of 32 keys ends inside a sequence)
  const bool d64 = p.head_dim == 64, several = mean < 32;
  // equal lengths, as far as the sizes tell, whose ends are those of blocks of 32 keys, or of 128: no block has a second stream
  const bool whole = seqs == 1 || (p.q_tokens == seqs * mean && mean % 32 == 0), whole128 = whole && mean % 128 == 0;
  int parts;
  if (workgroups <= kComputeUnits) {
    parts = steps >= (whole ? (d64 ? 4 : 7) : several ? 6 : 2) ? 4 : kLoneWave;
  } else if (several) {
    parts = workgroups <= 2 * kComputeUnits && steps >= (d64 ? 12 : 48) ? 4 : kLoneWave;
  } else if (workgroups <= 2 * kComputeUnits) {
    parts = steps >= (whole || workgroups > 384 ? 20 : 12) ? 4 : steps > (whole ? 6 : 3) ? 2 : kLoneWave;
  } else if (workgroups <= 1152) {
    const bool few = seen == mean && workgroups <= 1024 && !(whole && seqs > 12);  // blocks with the longest streams
    parts = few && steps >= (d64 ? 64 : workgroups <= 640 ? 28 : 80) ? 4 : steps > 5 ? 2 : kLoneWave;
  } else {
    // (one part: 512 workgroups of 128 keys are a full round)
    const bool one = workgroups > 3000 || (!d64 && steps <= 64 && (whole128 ? workgroups > 1536 : workgroups > 1792 && workgroups <= 2048));
    const int64_t lone = workgroups > (d64 ? 8192 : 4096) ? 3 : d64 ? 16 : one && whole128 ? 3 : 6;
    parts = steps <= lone ? kLoneWave : one ? 1 : 2;
  }
  if (parts == kLoneWave && workgroups > 0x7fffffffLL) parts = 1;
  // Pairs of blocks, whose costs add up to the same for one sequence, or two, where every pair then has a compute unit
  // and single blocks come round a second time: 1 x 1 978, 16 / 8 heads of 128 (496 blocks): the backward 117 us, 120 with single ones; 2 x 2 819,
  // 8 / 2 (354): 221, 232.  Far fewer pairs than units leave these idle (2 x 2 341, 8 / 2, 294: 256, 215), of many sequences single
  // blocks end closer together (13 x 451, 8 / 2, 368: 91.9, 76.6), and at head dim 64, where two workgroups share a unit, they
  // always do (1 x 3 091, 6 / 6, 582: 105, 95).
  bool pairs = !d64 && p.num_seqs <= 2 && workgroups >= kComputeUnits * 5 / 4 && (blocks + 1) / 2 * p.kv_heads <= kComputeUnits;
  // ARENO_BACKWARD_PARTS=1w|1|2|4s|4 (read at every launch; one wave, 4 with single blocks and in pairs) fixes the choice: the
  // same dK and dV up to the order of the last sums, so this is for tests of the kernels a launch of the test's size would
  // not take, and for timing
  const char* const name = "ARENO_BACKWARD_PARTS";
  if (fixed_by(name, "1")) parts = 1;
  if (fixed_by(name, "2")) parts = 2;
  if (workgroups <= 0x7fffffffLL) {
    if (fixed_by(name, "1w")) parts = kLoneWave;
    if (fixed_by(name, "4s")) parts = 4, pairs = false;
    if (fixed_by(name, "4")) parts = 4, pairs = true;
  }
  BwdLaunch launch;
  if (p.head_dim == 64) {
    launch = p.dtype == ARENO_DT_BF16 ? launch_of<KV_BF16, 64>(parts) : launch_of<KV_F16, 64>(parts);
  } else {
    launch = p.dtype == ARENO_DT_BF16 ? launch_of<KV_BF16, 128>(parts) : launch_of<KV_F16, 128>(parts);
  }
  *groups = parts != 4 ? (p.k_tokens + launch.rows - 1) / std::max(launch.rows, 1) : pairs ? (blocks + 1) / 2 : blocks;
  return launch;
}

}  // namespace areno
