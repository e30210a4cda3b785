// Causal attention over packed new tokens (the varlen op's forward; areno/accel/csrc/attention.cu:145-242 in the
// reference) on the matrix cores: 16-bit inputs, head dims 64, 128, 192 and 256.
//
// A workgroup of four waves computes one query block of one kv head -- 128 rows, row r being (token r / fold, q head
// r % fold) as in prefill_mfma.hip -- from its first visible key to its last.  No block is cut, so nothing is left
// to merge; the blocks of a launch are taken longest first (varlen_blocks.hpp), and two or three workgroups share a compute unit
// (four at head dim 64), so one's waits and softmax fall into the other's products.  Per step of 64 keys (32 at the wide
// heads, and at head dim 128 where short_tiles_are_faster) a wave, which owns 32 of the rows:
//   * passes one barrier and asks for the next step's K and V tiles, which the memory pipe writes into LDS by itself
//     (two buffers; mfma32_tiles.hpp);
//   * S^T = K . Q^T on 32 x 32 x 16 products, Q in registers; a lane holds half of the keys of one query row;
//   * the softmax of prefill_mfma.hip (the lazily raised reference), one lane swap where a row's halves meet;
//   * O^T += V^T . P^T with the probabilities as they lie.
// Measured against the kernel of prefill_mfma.hip and its merge, which it replaces for packed K / V but for few heads over
// long sequences (equal_shares_are_faster), bf16, us: 32 prompts of 33 .. 512 tokens, 28 / 4 heads of 128, with the cache
// write: 128 -> 40; 2 x 2 048: 166 -> 74; 4 x 4 096, 32 / 8 heads: 725 -> 520 (1 060 TFLOP/s); 256 tokens alone, 8 / 2 heads:
// 46 -> 11; 256 x 24: 43 -> 34; 1 024 x 24: 154 -> 159; 4 x 300 .. 1 000, 16 / 8 heads of 256, window 512: 88 -> 32;
// 16 x 20 .. 600, 16 heads of 64, fp16: 50 -> 16.  What it does not spend any more: a ~10 us fill and drain
// per query block with nothing beside it, the partials of cut blocks (up to 67 MB written and read), a third of the
// loop's vector instructions (staging, half the lane swaps).  Bound at length by the matrix cores and the LDS
// reads behind them (an operand read per product), at short lengths by a block's chain of steps.
#include <algorithm>
#include <atomic>

#include "cache_row_quant.hpp"
#include "mfma32_tiles.hpp"
#include "page_write.hpp"
#include "varlen_blocks.hpp"

namespace areno {
namespace {

constexpr int kVmWaves = 4;
constexpr int kVmThreads = kVmWaves * kWave;
constexpr int kVmRows = 32 * kVmWaves;  // query rows of a workgroup

struct VarlenMfmaParams {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  const int32_t* cu_seqlens;
  int32_t tokens;
  int32_t num_seqs;
  int32_t q_heads;
  int32_t kv_heads;
  int32_t group;
  int32_t head_parts;    // workgroups of a block per kv head: up to 16 of its q heads each
  int32_t fold;          // row r of a block is (token r / fold, q head r % fold of the part)
  int32_t fold_magic;    // ceil(2^16 / fold)
  int32_t block_tokens;  // kVmRows / fold
  BlockDivision block_division;
  int32_t window_left;
  float scale_log2e;
  PageWrite pages;  // (of the instances that write them)
};

// What the i-th workgroup of a head computes (block_place); false: nothing.  A lane
// holds the blocks of sequences lane, lane + 64, ... in registers: a step of the bisection is a sum over the wave.
// (Read again from cu_seqlens at every step, 1 024 sequences of 24 tokens, 28 / 4 heads, took 355 us instead of 159, and
// a prefix sum by the whole workgroup, as in prefill_mfma.hip, 154.)
struct BlockAt {
  int j, q_begin, n_new;  // block j of the sequence whose n_new tokens start at q_begin
  int idle;               // of a workgroup without a block: its place among those
};
template <int ROUNDS>
__device__ __forceinline__ bool find_block(const VarlenMfmaParams& p, int i, BlockAt& at) {
  const int lane = threadIdx.x & (kWave - 1);
  int begin[ROUNDS], tokens[ROUNDS], blocks[ROUNDS], most = 0;
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int s = 64 * r + lane;
    begin[r] = p.cu_seqlens[min(s, p.num_seqs)];
    tokens[r] = max(p.cu_seqlens[min(s + 1, p.num_seqs)] - begin[r], 0);
  }
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    blocks[r] = p.block_division(tokens[r] + p.block_tokens - 1);
    most = max(most, blocks[r]);
  }
  BlockPlace place;
  const bool found = block_place(
      i, wave_reduce(most, [](int a, int b) { return max(a, b); }),
      [&](int j) {
        int n = 0;
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) n += max(0, blocks[r] - j);
        return wave_reduce(n, [](int a, int b) { return a + b; });
      },
      place);
  if (!found) {
    at.idle = place.nth;
    return false;
  }
  at.j = place.j;
  int nth = place.nth;
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const uint64_t has = __builtin_amdgcn_ballot_w64(blocks[r] > place.j);
    const bool mine = (has >> lane & 1) != 0 && __builtin_popcountll(has & ((uint64_t{1} << lane) - 1)) == nth;
    const uint64_t chosen = __builtin_amdgcn_ballot_w64(mine);
    if (chosen != 0) {
      const int from = __builtin_ctzll(chosen);
      at.q_begin = __builtin_amdgcn_readlane(begin[r], from);
      at.n_new = __builtin_amdgcn_readlane(tokens[r], from);
    }
    nth -= __builtin_popcountll(has);  // (below zero behind the chosen one: no lane has that rank)
  }
  return true;
}

// (the output is taken from 8-byte alignment on; the same instruction stores it)
typedef uint4_t uint4_at8_t __attribute__((aligned(8)));
extern __shared__ __attribute__((aligned(1024))) char vm_lds[];
constexpr int kSchedMatrix = 0x8, kSchedLdsRead = 0x100;  // instruction classes of sched_group_barrier

template <int D, bool WRITE, int TILE>
struct VmShape {
  static constexpr int kTile = TILE;  // keys per step
  using Tile = LdsTile<D, kTile, kVmWaves>;
  static constexpr int kBuffer = 2 * Tile::kBytes;  // K, V
  static constexpr int kQueries = kBuffer + (D <= 128 ? kVmRows * D * 2 : 0);  // the end of the query rows, which start where the second tile will lie
  static constexpr int kPlaces = 2 * kBuffer > kQueries ? 2 * kBuffer : kQueries;  // the pages of the block's tokens, then their places in these
  static constexpr int kLdsBytes = WRITE ? kPlaces + 2 * kVmRows * 8 : kPlaces;
};

// A token's row of one kv head (of K, or `second`: of V) into the pages: quantized or copied, chunk `sub` of 16 bytes per
// lane, a row's lanes next to each other.  The bits are those of areno_hip_cache_write: the same closed forms over the same lanes.
template <int KIND, int D>
__device__ __forceinline__ void write_page_chunk(const PageWrite& w, uint4_t raw, bool second, int64_t id, int64_t slot, int kvh, int kv_heads, int sub, bool live) {
  const bool store = live && id >= 0 && id < w.num_blocks && slot >= 0 && slot < w.block_size;
  const int64_t dst_row = (id * w.block_size + slot) * kv_heads + kvh;
  void* const pool = second ? w.v : w.k;
  constexpr bool kWholeGroups = (D & (D - 1)) == 0;  // a row's lanes are a power of two, as its maximum wants them
  if (kWholeGroups && is_quantized_dtype(w.cache_dtype)) {
    float x[8], amax = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x[2 * j] = operand_element<KIND>(raw[j], 0);
      x[2 * j + 1] = operand_element<KIND>(raw[j], 1);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(x[j]));
    amax = lane_group_max<kWholeGroups ? D / 8 : 1>(amax);
    if (store) store_row_slice(x, amax, sub, dst_row, D, pool, second ? w.v_scale : w.k_scale, w.cache_dtype, w.scale_dtype);
  } else if (store) {
    // (whole rows that nothing here reads again: kept out of the way of the tiles in L2; the case below 57.5 -> 55.1 us)
    __builtin_nontemporal_store(raw, reinterpret_cast<uint4_t*>(static_cast<char*>(pool) + (dst_row * D + sub * 8) * 2));
  }
}

// (Two waves per SIMD -- three with steps of 32 keys at head dim 128, four at 64 -- are what the tiles leave room for, and the scheduler is told so: where it
// takes three to be within reach it saves registers for them and waits for every operand read right behind it --
// 8 192 tokens, 8 / 1 heads of 128: 208 instead of 172 us.)
//
// WRITE: the launch also stores the tokens' K and V in the pages of a cache, which nothing in it reads.  A block's workgroup
// has the rows of its own tokens in LDS when it is done -- they are the last keys that its rows see -- so they cost no
// fetch, and their stores go out behind the output's, while the next workgroup starts.  The pass with a launch of its own for
// the pages and with this, us (both with the output's stores as they were then): 32 prompts of 33 .. 512 tokens, 28 / 4 heads of 128, bf16: 61.5 -> 57.6; 2 x 3 000 .. 6 000, 16 / 8
// heads of 256, window 1 024: 176.6 -> 165; 24 x 48 .. 387 into fp8 pages 40.0 -> 38.8; 2 x 9 .. 74: 21.7 -> 17.7 (the host's).
//
// PAST_L2: the output's stores leave L2 to the tiles (output_past_l2).
template <int KIND, int D, bool WRITE, int TILE, bool PAST_L2>
__global__ __launch_bounds__(kVmThreads) __attribute__((amdgpu_waves_per_eu(D == 128 && TILE == 32 ? 3 : 2, D == 64 ? 4 : D == 128 && TILE == 32 ? 3 : 2))) void varlen_mfma_kernel(VarlenMfmaParams p) {
  using S = VmShape<D, WRITE, TILE>;
  using T = typename S::Tile;
  using M = Mfma32<KIND>;
  using V8 = typename M::vec8;
  constexpr int TK = S::kTile;
  constexpr int KT = TK / 32;   // 32-key score tiles per step
  constexpr int NKS = D / 16;   // contraction steps of a score tile
  constexpr int NB = D / 32;    // 32-element blocks of the head
  constexpr int NF = T::kFetches;

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = uniform(tid >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  const int vheads = p.kv_heads * p.head_parts;
  const int vhead = static_cast<int>(blockIdx.x % static_cast<unsigned>(vheads));
  const int kvh = p.head_parts > 1 ? vhead / p.head_parts : vhead;
  const int head0 = kvh * p.group + 16 * (vhead - kvh * p.head_parts);
  const int group_here = min(16, (kvh + 1) * p.group - head0);
  const int tq = p.block_tokens;

  BlockAt at;
  {
    const int i = static_cast<int>(blockIdx.x / static_cast<unsigned>(vheads));
    bool found;
    if (p.num_seqs <= 64) {
      found = find_block<1>(p, i, at);
    } else if (p.num_seqs <= 256) {
      found = find_block<4>(p, i, at);
    } else {
      found = find_block<16>(p, i, at);
    }
    if (!found) {
      // (the same for the whole workgroup; the grid covers the most blocks the token count allows and one more).  Rows
      // behind the last sequence -- the end of a padded pack -- become zeros, over the workgroups that have no block
      const int end = p.cu_seqlens[p.num_seqs], rest = max(p.tokens - end, 0);
      const int front = WRITE ? p.cu_seqlens[0] : 0;  // (tokens in front of the first sequence: their pages are written as well)
      if (rest + front <= 0) return;
      const int idle = static_cast<int>(gridDim.x / static_cast<unsigned>(vheads)) - i + at.idle;  // so many
      if constexpr (WRITE) {
        constexpr int kChunks = D / 8;
        if (head0 == kvh * p.group) {  // (the first of a kv head's parts)
          const int64_t chunks = static_cast<int64_t>(rest + front) * kChunks;
          for (int64_t c = at.idle * kVmThreads + tid; c < 2 * chunks; c += static_cast<int64_t>(idle) * kVmThreads) {
            const bool second = c >= chunks;
            const int64_t nth = (c - (second ? chunks : 0)) / kChunks, token = nth < front ? nth : nth - front + end;
            const int sub = static_cast<int>(c % kChunks);
            const uint4_t raw = load16(second ? p.v : p.k, ((token * p.kv_heads + kvh) * D + sub * 8) * 2);
            write_page_chunk<KIND, D>(p.pages, raw, second, p.pages.block_ids[token], p.pages.block_offsets[token], kvh, p.kv_heads, sub, true);
          }
        }
      }
      const int per_token = group_here * (D / 4);
      const int64_t words = static_cast<int64_t>(rest) * per_token;
      for (int64_t w = at.idle * kVmThreads + tid; w < words; w += static_cast<int64_t>(idle) * kVmThreads) {
        const int64_t elem = ((end + w / per_token) * p.q_heads + head0) * D + 4 * (w % per_token);
        *reinterpret_cast<uint2_t*>(static_cast<char*>(p.out) + elem * 2) = uint2_t{0u, 0u};
      }
      return;
    }
  }
  const int q_begin = uniform(at.q_begin), n_new = uniform(at.n_new);
  const int tok0 = uniform(at.j) * tq;
  const int tok_cnt = min(tq, n_new - tok0);

  // ---- this lane's query row -------------------------------------------------------------------------------------
  auto token_of_row = [&](int r) { return (r * p.fold_magic) >> 16; };
  const int r = 32 * wave + l32;
  const int t_row = token_of_row(r);
  const int hh = r - t_row * p.fold;
  const bool live = t_row < tok_cnt && hh < group_here;
  const int q_pos = live ? tok0 + t_row : -1;
  // Up to head dim 128 the query rows come through LDS, where the second tile will lie, as whole rows: a lane needs 16 bytes
  // here and there of one row, and asked for as such they are 64 pieces an instruction (the kernel with steps of 64 keys, us:
  // 4 x 4 096, 32 / 8 heads: 548 -> 540; 16 x 20 .. 600, 16 heads of 64: 16.4 -> 15.9).  The wide heads' rows are twice what a buffer
  // holds.  Rows that do not exist repeat the block's first.
  constexpr bool kRowsThroughLds = D <= 128;
  V8 qop[NKS];
  if constexpr (!kRowsThroughLds) {
    const int64_t row_elem = (static_cast<int64_t>(q_begin + tok0 + t_row) * p.q_heads + head0 + hh) * D;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      uint4_t w = {0u, 0u, 0u, 0u};
      if (live) w = load16(p.q, (row_elem + 16 * ks + 8 * h) * 2);
      qop[ks] = __builtin_bit_cast(V8, w);
    }
  } else {
    const char* const rows = static_cast<const char*>(p.q) + (static_cast<int64_t>(q_begin + tok0) * p.q_heads + head0) * (D * 2);
    constexpr int kFetchRows = 64 / T::kChunksPerRow;
#pragma unroll
    for (int f = 0; f < 32 / kFetchRows; ++f) {
      const int row = kFetchRows * f + lane / T::kChunksPerRow, t = token_of_row(32 * wave + row), head = 32 * wave + row - t * p.fold;
      const bool there = t < tok_cnt && head < group_here;
      const uint32_t off = there ? static_cast<uint32_t>(t * p.q_heads + head) * (D * 2) : 0u;
      fetch_to_lds(rows, off + static_cast<uint32_t>((lane % T::kChunksPerRow) ^ T::twist(row)) * 16u,
                   lds_address(vm_lds) + S::kBuffer + wave * (32 * T::kRowBytes) + f * 1024);
    }
  }
  const bool wave_live = 32 * wave < tok_cnt * p.fold;
  const int wave_qmin = tok0 + token_of_row(32 * wave);
  const int wave_qmax = tok0 + min(tok_cnt - 1, token_of_row(32 * wave + 31));

  // ---- the stream of key tiles -----------------------------------------------------------------------------------
  const int key_hi = tok0 + tok_cnt - 1;  // the last key any row of the block sees
  const int key_lo = p.window_left >= 0 ? max(0, tok0 - p.window_left) : 0;
  const int ta = key_lo / TK, tb = key_hi / TK;
  const float lazy = TK == 64 ? 8.0f : D == 128 && tb - ta < 4 ? 1.0f : 2.0f;  // (log2: by how much a score may exceed its row's reference)
  const int64_t stride = static_cast<int64_t>(p.kv_heads) * D * 2;
  const int64_t head_base = (static_cast<int64_t>(q_begin) * p.kv_heads + kvh) * (D * 2);
  const char* const k_base = static_cast<const char*>(p.k) + head_base;
  const char* const v_base = static_cast<const char*>(p.v) + head_base;
  const uint32_t lds0 = lds_address(vm_lds);
  int fetch_row[NF];
  uint32_t fetch_chunk[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int slot = (wave * NF + f) * 64 + lane;
    fetch_row[f] = slot / T::kChunksPerRow;
    fetch_chunk[f] = static_cast<uint32_t>((slot % T::kChunksPerRow) ^ T::twist(fetch_row[f])) * 16u;
  }
  auto fetch = [&](int t, int buf) {
    const int rows = key_hi + 1 - t * TK;  // rows of the tile that exist; the ones behind repeat the last
    const char* kb = k_base + static_cast<int64_t>(t) * TK * stride;
    const char* vb = v_base + static_cast<int64_t>(t) * TK * stride;
    const uint32_t dst = lds0 + static_cast<uint32_t>(buf * S::kBuffer + wave * (NF * 1024));
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const uint32_t off = static_cast<uint32_t>(min(fetch_row[f], rows - 1)) * static_cast<uint32_t>(stride) + fetch_chunk[f];
      fetch_to_lds(kb, off, dst + f * 1024);
      fetch_to_lds(vb, off, dst + T::kBytes + f * 1024);
    }
  };

  float16_t acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) acc[nb] = zero16();
  float m_run = kNegInf, l_lane = 0.0f;

  uint32_t at_rows = T::rows_base(l32, h), at_columns = T::columns_base(lane);
  auto step = [&](int t, int buf) {
    // (wide heads: the 32 addresses of a step are worked out where they are used, instead of being kept in registers
    // that the sums need)
    if constexpr (D > 128) asm volatile("" : "+v"(at_rows), "+v"(at_columns));
    fetched_barrier();  // tile t (asked for a step ago) is there, and every wave has left tile t - 1
    if (t < tb) fetch(t + 1, buf ^ 1);
    const int k0 = t * TK;
    if (!wave_live || k0 > wave_qmax) return;
    if (p.window_left >= 0 && k0 + TK - 1 < wave_qmin - p.window_left) return;
    char* kt_lds = vm_lds + buf * S::kBuffer;
    char* vt_lds = vm_lds + buf * S::kBuffer + T::kBytes;
    float16_t s[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) s[kt] = zero16();
    // Wide heads: the products' operands in one stream, each read kAhead products in front of its own (the compiler, short of
    // registers, waits for most of them right behind the read): rows of K, then columns of V.  Two sequences of 3 000 .. 6 000
    // tokens, 16 / 8 heads of 256, window 1 024: 162 -> 158 us (under the profiler); up to head dim 128 it changes the time by -7 to +3 % and is not used.
    constexpr int kScores = NKS * KT, kReads = kScores + 2 * KT * NB, kAhead = D == 256 ? 3 : 4;
    auto read = [&](int x) {
      if (x < kScores) return tile_rows<KIND, T>(kt_lds, at_rows, 32 * (x % KT), x / KT);
      return tile_columns<KIND, T>(vt_lds, at_columns, 16 * ((x - kScores) / NB), (x - kScores) % NB);
    };
    V8 operand[kAhead];
    if constexpr (D > 128) {
#pragma unroll
      for (int x = 0; x < kAhead; ++x) operand[x] = read(x);
#pragma unroll
      for (int x = 0; x < kScores; ++x) {
        __builtin_amdgcn_sched_barrier(0);
        s[x % KT] = M::mfma(operand[x % kAhead], qop[x / KT], s[x % KT]);
        operand[x % kAhead] = read(x + kAhead);
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) s[kt] = M::mfma(tile_rows<KIND, T>(kt_lds, at_rows, 32 * kt, ks), qop[ks], s[kt]);
      }
      // four operand reads ahead of the products: left alone the compiler waits for
      // every pair of reads right behind it (4 x 4 096 tokens, 32 / 8 heads of 128: 577 -> 557 us)
      __builtin_amdgcn_sched_group_barrier(kSchedLdsRead, kAhead, 0);
#pragma unroll
      for (int x = 0; x < NKS * KT - kAhead; ++x) {
        __builtin_amdgcn_sched_group_barrier(kSchedMatrix, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kSchedLdsRead, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(kSchedMatrix, kAhead, 0);
    }
    if (k0 + TK - 1 > wave_qmin || (p.window_left >= 0 && k0 < wave_qmax - p.window_left)) {
      const int hi = q_pos - k0 - 4 * h;
      const int lo = p.window_left >= 0 ? hi - p.window_left : -0x40000000;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = 32 * kt + 8 * (i >> 2) + (i & 3);
          s[kt][i] = key <= hi && key >= lo ? s[kt][i] : kNegInf;
        }
      }
    }
    // online softmax as in prefill_mfma.hip: the reference value is raised only when a tile exceeds it by 2^8, by 2^2 with steps
    // of 32 keys, whose first tile sets a lower one, and at head dim 128 by 2 where a block has no more than four of them.  Relative
    // error against 64 bits with 2^8 and 2^2, in bf16, and of the kernel with longer steps that it replaces: 256 wide, 300 .. 1 000
    // tokens, window 512: 2.026e-3, 1.992e-3, 2.020e-3; 192 wide: 1.985e-3, 1.955e-3, 1.957e-3; 128 wide, 33 .. 900 tokens: 1.973e-3,
    // 1.949e-3, 1.960e-3 (fp16 2.467e-4, 2.436e-4, 2.450e-4).  It costs 2 to 4 % of the time.  With 2^2, with 2, and with longer steps, 128 wide,
    // sequences of 64 tokens: 1.8202e-3, 1.8137e-3, 1.8177e-3, of 48: 1.7902e-3, 1.7872e-3, 1.7888e-3; 2 everywhere would cost 3 % more.
    float mt = max3_f32(s[0][0], s[0][1], s[0][2]);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
      for (int i = kt == 0 ? 3 : 0; i < 16; i += 2) mt = max3_f32(mt, s[kt][i], s[kt][i + 1 < 16 ? i + 1 : i]);
    }
    if (__builtin_amdgcn_ballot_w64(mt * p.scale_log2e > m_run + lazy) != 0) {
      uint32_t a = __builtin_bit_cast(uint32_t, mt), b = a;
      swap_rows32(a, b);
      mt = max_f32(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
      const float m_new = max_f32(m_run, mt * p.scale_log2e);
      const float m_ref = m_new == kNegInf ? 0.0f : m_new;
      const float alpha = settled(fast_exp2(m_run - m_ref));
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
    const float m_safe = m_run == kNegInf ? 0.0f : m_run;
    V8 pop[2 * KT];
#pragma unroll
    for (int b = 0; b < 2 * KT; ++b) {
      uint32_t w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = 8 * (b & 1) + 2 * j;
        w[j] = pack_pair<KIND>(fast_exp2(__builtin_fmaf(s[b >> 1][i], p.scale_log2e, -m_safe)),
                               fast_exp2(__builtin_fmaf(s[b >> 1][i + 1], p.scale_log2e, -m_safe)));
        l_lane = M::add_pair(w[j], l_lane);  // sums the probabilities as rounded for the product
      }
      pop[b] = __builtin_bit_cast(V8, uint4_t{w[0], w[1], w[2], w[3]});
    }
#pragma unroll
    for (int b = 0; b < 2 * KT; ++b) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int x = kScores + b * NB + nb;
        if constexpr (D > 128) {
          __builtin_amdgcn_sched_barrier(0);
          acc[nb] = M::mfma(operand[x % kAhead], pop[b], acc[nb]);
          if (x + kAhead < kReads) operand[x % kAhead] = read(x + kAhead);
        } else {
          acc[nb] = M::mfma(read(x), pop[b], acc[nb]);
        }
      }
    }
  };

  fetch(ta, 0);
  // the tokens' places in the cache, into LDS with the first tile (asked for at the block's end, which is when they are
  // needed, 1 560 blocks of 32 prompts of 33 .. 512 tokens take 56.2 us instead of 52.7, without a store)
  const bool writes = WRITE && head0 == kvh * p.group;  // (the first of a kv head's parts)
  if (writes && kWave * wave < 2 * tok_cnt) {
    const uint32_t words = static_cast<uint32_t>(2 * tok_cnt), word = min(static_cast<uint32_t>(kWave * wave + lane), words - 1) * 4u;
    const int64_t first = static_cast<int64_t>(q_begin + tok0) * 8;
    fetch_words_to_lds(reinterpret_cast<const char*>(p.pages.block_ids) + first, word, lds0 + S::kPlaces + wave * (kWave * 4));
    fetch_words_to_lds(reinterpret_cast<const char*>(p.pages.block_offsets) + first, word, lds0 + S::kPlaces + kVmRows * 8 + wave * (kWave * 4));
  }
  if constexpr (kRowsThroughLds) {
    fetched();  // (its own rows: no barrier)
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qop[ks] = tile_rows<KIND, T>(vm_lds + S::kBuffer + wave * (32 * T::kRowBytes), at_rows, 0, ks);
  }
  // (the query rows are waited for here: left to their first use inside the loop, that wait would cover every step's
  // fetches as well)
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    uint4_t w = __builtin_bit_cast(uint4_t, qop[ks]);
    asm volatile("" : "+v"(w));
    qop[ks] = __builtin_bit_cast(V8, w);
  }
  for (int t = ta; t <= tb; t += 2) {
    step(t, 0);
    if (t + 1 <= tb) step(t + 1, 1);
  }

  if (writes) {
    constexpr int kChunks = D / 8;  // of a row
    const int chunks = tok_cnt * kChunks, thread = wave * kWave + lane_now();
    const int64_t* const places = reinterpret_cast<const int64_t*>(vm_lds + S::kPlaces);
    for (int first = 0; first < 2 * chunks; first += kVmThreads) {  // K's, then V's
      const int c = min(first + thread, 2 * chunks - 1), sub = (first + thread) % kChunks;
      const bool second = c >= chunks;
      const int nth = (c - (second ? chunks : 0)) / kChunks;
      const int key = tok0 + nth, t = key / TK, row = key % TK;
      uint4_t raw;
      if (t >= tb - 1) {  // the last two tiles lie in LDS, as their last barrier left them
        raw = *reinterpret_cast<const uint4_t*>(vm_lds + ((t - ta) & 1) * S::kBuffer + (second ? T::kBytes : 0) + row * T::kRowBytes +
                                                ((sub ^ T::twist(row)) << 4));
      } else {
        raw = load16(second ? v_base : k_base, static_cast<int64_t>(key) * stride + sub * 16);
      }
      write_page_chunk<KIND, D>(p.pages, raw, second, places[nth], places[kVmRows + nth], kvh, p.kv_heads, sub, first + thread < 2 * chunks);
    }
    handed_barrier();  // (the tile in front of the last is read)
  }

  // The output through LDS (RowStage), where the tile in front of the last one lay: every wave has left it.  Against pieces of
  // 8 bytes from the accumulators, as whole rows past L2, the kernel in us (whole rows kept in L2): 32 prompts of
  // 33 .. 512 tokens, 28 / 4 heads of 128, with the pages: 57.8 -> 47.6 (50.0); 2 x 3 000 .. 6 000, 16 / 8 heads of 256, window 1 024: 197 ->
  // 180 (187); 16 x 20 .. 600, 16 heads of 64: 16.5 -> 15.5 (16.8); 2 x 2 048: 84.8 -> 81.0 (82.7); 4 x 4 096, 32 / 8: 558 -> 545 (545).
  uint32_t a = __builtin_bit_cast(uint32_t, l_lane), b = a;
  swap_rows32(a, b);
  const float l_tot = __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
  const float inv = 1.0f / l_tot;  // (rows that do not exist are not stored)
  char* const rows_lds = vm_lds + ((tb - ta + 1) & 1) * S::kBuffer + wave * (S::kBuffer / kVmWaves);
  constexpr int kBlocks = S::kBuffer / kVmWaves / (32 * 64);  // blocks of 32 elements that a wave's part holds of its rows
  constexpr int kRounds = (NB + kBlocks - 1) / kBlocks, kHere = NB / kRounds, kRowChunks = kHere * 4;
  static_assert(NB % kRounds == 0, "the output's parts");
  using Stage = RowStage<kRowChunks>;
  const int l = lane_now();
#pragma unroll
  for (int round = 0; round < kRounds; ++round) {
#pragma unroll
    for (int x = 0; x < kRowChunks; ++x) {
      const int nb = round * kHere + x / 4, c = x % 4;
      Stage::put(rows_lds, l & 31, x, l >> 5, pack_pair<KIND>(acc[nb][4 * c] * inv, acc[nb][4 * c + 1] * inv),
                 pack_pair<KIND>(acc[nb][4 * c + 2] * inv, acc[nb][4 * c + 3] * inv));
    }
    Stage::template take<32>(rows_lds, l, [&](int row, int chunk, uint4_t w) {
      const int t_here = token_of_row(32 * wave + row), head_here = 32 * wave + row - t_here * p.fold;
      if (t_here < tok_cnt && head_here < group_here) {
        const int64_t elem = (static_cast<int64_t>(q_begin + tok0 + t_here) * p.q_heads + head0 + head_here) * D + round * (32 * kHere) + 8 * chunk;
        uint4_at8_t* const to = reinterpret_cast<uint4_at8_t*>(static_cast<char*>(p.out) + elem * 2);
        if constexpr (PAST_L2) {
          __builtin_nontemporal_store(w, to);
        } else {
          *to = w;
        }
      }
    });
  }
}

typedef void (*vm_fn)(VarlenMfmaParams);
struct VmLaunch {
  vm_fn fn;  // nullptr: no such kernel, or its LDS size was refused
  int lds_bytes;
};
template <int KIND, int D, bool WRITE, int TILE, bool PAST_L2>
VmLaunch vm_launch_of() {
  static std::atomic<uint64_t> allowed_on{0};
  constexpr int kLdsBytes = VmShape<D, WRITE, TILE>::kLdsBytes;
  const vm_fn fn = varlen_mfma_kernel<KIND, D, WRITE, TILE, PAST_L2>;
  return {allow_lds<kLdsBytes>(reinterpret_cast<const void*>(fn), allowed_on) ? fn : nullptr, kLdsBytes};
}
template <int KIND, bool WRITE, bool PAST_L2>
VmLaunch vm_lookup(int head_dim, bool short_tiles) {
  switch (head_dim) {
    case 64: return vm_launch_of<KIND, 64, WRITE, 64, PAST_L2>();
    case 128: return short_tiles ? vm_launch_of<KIND, 128, WRITE, 32, PAST_L2>() : vm_launch_of<KIND, 128, WRITE, 64, PAST_L2>();
    case 192: return vm_launch_of<KIND, 192, WRITE, 32, PAST_L2>();
    case 256: return vm_launch_of<KIND, 256, WRITE, 32, PAST_L2>();
    default: return {nullptr, 0};
  }
}
template <int KIND>
VmLaunch vm_lookup(int head_dim, bool short_tiles, bool write, bool past_l2) {
  if (write) return past_l2 ? vm_lookup<KIND, true, true>(head_dim, short_tiles) : vm_lookup<KIND, true, false>(head_dim, short_tiles);
  return past_l2 ? vm_lookup<KIND, false, true>(head_dim, short_tiles) : vm_lookup<KIND, false, false>(head_dim, short_tiles);
}

// The output's stores past L2 leave it to the tiles, 2 to 12 % of the kernel from 4 MB on, and cost the reader behind it nothing there; up to
// 2 MB they gain nothing and cost it up to 2 us.  With and without, attention and a product with its output's width,
// us: 16 heads of 64, 256 tokens (0.5 MB): 15.4, 13.8; 8 / 2 of 128, 500 (1 MB): 21.7, 19.4; 28 / 4, 500 (3.6 MB): 41.9, 42.8; 8 / 2,
// 4 448 (9.1 MB): 33.6, 34.7; 28 / 4, 8 333 (60 MB): 210.1, 209.7; 16 / 8 of 256, 16 384 (134 MB): 903, 934.  (Two instances: decided inside the
// kernel, per store or per block, it costs heads of 256 and short steps 2 to 4 %.)
bool output_past_l2(int64_t tokens, int32_t q_heads, int32_t head_dim) { return tokens * q_heads * head_dim * 2 > (int64_t{2} << 20); }

// Few heads over long sequences: such a launch has fewer blocks than the chip has places for, and lasts as long as its
// longest block, one chain of steps over all its keys.  The kernel of prefill_mfma.hip, which cuts the blocks' steps
// into equal shares and merges them, is the faster one there, us (shares, this kernel; q / kv heads):
//   64 wide:  6 144 tokens, 1/1: 60, 76;  8 192, 2/1: 66, 101;  4 096, 3/3: 46, 52;  12 288, 4/4: 150, 153
//             4 096, 1/1: 65, 52;  32 768, 2/1: 430, 420;  32 768, 3/3: 610, 525;  8 192, 5/1: 144, 103
//   128 wide: 6 144, 1/1: 72, 101;  16 384, 1/1: 127, 263;  8 192, 2/1: 96, 136;  4 096, 3/3: 62, 70;  12 288, 4/4: 217, 223
//             4 096, 1/1: 78, 69;  4 096, 4/1: 80, 70;  32 768, 3/3: 880, 791;  8 192, 5/1: 217, 146
//   192 wide: 4 096, 1/1: 62, 101;  16 384, 2/1: 379, 381;  8 192, 3/3: 173, 198;  12 288, 3/3: 309, 300;  2 048, 1/1: 74, 55
//   256 wide: 2 048, 2/1: 63, 77;  16 384, 1/1: 246, 542;  12 288, 3/3: 366, 418;  12 288, 4/4: 471, 453;  2 048, 5/1: 116, 78
//   with a window: 16 384, 1/1, 256 wide, window 8 192: 206, 285;  128 wide, 4 096: 89, 77;  2/1, 256 wide, 8 192: 368, 290
// The lengths are not known on the host: they are taken to be about equal (two of 8 192, 1/1: 100, 134; four: 134, 139).
bool equal_shares_are_faster(int64_t tokens, int32_t num_seqs, int32_t q_heads, int32_t group, int32_t head_dim, int32_t window_left) {
  if (static_cast<int64_t>(q_heads) * num_seqs > (group == 1 ? 4 : 3)) return false;  // chains side by side
  const int64_t mean = tokens / num_seqs;
  // a block sees half a sequence on the average, or all of a shorter window
  const bool cut = window_left >= 0 && window_left + int64_t{1} < mean;
  const int64_t length = cut ? (window_left + int64_t{1}) / 2 : mean;
  const int64_t blocks = (cut ? 2 : 1) * tokens * q_heads / kVmRows;
  if (head_dim <= 128) return length >= 4096 && blocks >= 48 && blocks <= 384;
  return head_dim == 192 ? length >= 4096 && blocks <= 256 : length >= 2048 && blocks <= 320;
}

// Head dim 128: steps of 32 keys leave room for three workgroups per compute unit, whose starts, ends and softmax fall into
// each other's products; steps of 64, two workgroups, are fewer, which counts where a launch is the chain of its longest
// blocks.  Sequences of up to 64 keys fill no more than one long step.  Where blocks cost alike -- a window, or sequences of equal
// length as far as the sizes tell -- 32 wins as soon as there are more blocks than the 512 places of the longer steps, or a few less: a second
// round is spared; the more keys, the more blocks it takes, up to 900.  Where lengths differ the longest ones decide for longer, and the line
// lies higher, up to 1 400 blocks (of the tokens, half a block more per sequence).  In us, 64 and 32 keys (blocks, keys seen):
//   equal: 28 / 4 heads, 16 x 200 (740, 200) 17.8, 13.1; 2 x 2 048 (912, 2 048) 81, 74; 4 x 4 096 (3 648) 476, 468; 32 / 8, 1 x 4 096 (1 024) 146, 141;
// 16 / 16, 4 x 250 (144) 11.8, 12.5; 28 / 4, 1 x 2 048 (452) 45.0, 49;
//   ragged: 28 / 4, 64 x 12 .. 52 (588, 32) 11.7, 8.2; 64 x 25 .. 390 (2 913, 195) 60.8, 52; 16 x 64 .. 960 (1 716, 474) 52.3, 47; 8 / 2, 4 x 3 334 on average
// (840) 137, 149.
// Of 2 576 launches of 1 .. 64 sequences of 12 .. 8 192 tokens, seven head ratios, equal and two kinds of ragged lengths, with and without a
// window, most of them near the lines, the choice takes 1.3 % more than the better one, 64 keys everywhere 5.6 %, 32 everywhere 4.0 %, one line
// for all of them (550 + 3 / 20 of the keys) 2.1 %; it is slower than 64 keys by more than 3 % in 165, most with one sequence far longer
// than the rest, that line in 431.  At head dim 64, where four workgroups share a unit with 64 keys, five with 32 gain and lose as much.
bool short_tiles_are_faster(int64_t tokens, int32_t num_seqs, int64_t vheads, int block_tokens, int32_t window_left) {
  const int64_t mean = tokens / num_seqs, window = window_left + int64_t{1} + block_tokens;
  const int64_t seen = window_left >= 0 ? std::min(mean, window) : mean;
  if (seen <= 64) return true;
  const bool alike = num_seqs == 1 || (mean * num_seqs == tokens && mean % 16 == 0) || seen < mean;
  return (tokens / block_tokens + num_seqs / 2) * vheads >= std::min<int64_t>(alike ? 425 + seen / 4 : 300 + 2 * seen, alike ? 900 : 1400);
}

}  // namespace

// Called by launch_prefill_mfma behind its checks (types, scale, sizes, alignment, workspace), so that a packed call is
// taken or refused, by the matrix cores or the generic kernel, as it is there.  ARENO_ERR_UNSUPPORTED: a launch for
// the kernel of prefill_mfma.hip.  `pages` (optional): where the launch also stores K and V.
int launch_varlen_mfma(const void* q, const void* k, const void* v, void* out, int32_t dtype, int64_t tokens,
                       int32_t q_heads, int32_t kv_heads, int32_t head_dim, const int32_t* cu_seqlens, int32_t num_seqs,
                       int32_t window_left, float softmax_scale, const PageWrite* pages, void* stream) {
  const char* op = "areno_hip_varlen_attention";
  const bool bf16 = dtype == ARENO_DT_BF16;
  const int group = q_heads / kv_heads, head_parts = (group + 15) / 16;
  const bool short_tiles = short_tiles_are_faster(tokens, num_seqs, kv_heads * head_parts, kVmRows / (head_parts > 1 ? 16 : group), window_left);
  const bool past_l2 = output_past_l2(tokens, q_heads, head_dim);
  const VmLaunch l = bf16 ? vm_lookup<KV_BF16>(head_dim, short_tiles, pages != nullptr, past_l2) : vm_lookup<KV_F16>(head_dim, short_tiles, pages != nullptr, past_l2);
  if (l.fn == nullptr) return ARENO_ERR_UNSUPPORTED;
  if (equal_shares_are_faster(tokens, num_seqs, q_heads, group, head_dim, window_left)) return ARENO_ERR_UNSUPPORTED;
  const int64_t vheads = static_cast<int64_t>(kv_heads) * head_parts;
  // offsets inside a key tile and inside a block's query rows are 32 bits wide
  if (static_cast<int64_t>(kv_heads) * head_dim * 2 * 64 > 0x7fffffffLL) return ARENO_ERR_UNSUPPORTED;
  if (static_cast<int64_t>(kVmRows / (head_parts > 1 ? 16 : group)) * q_heads * head_dim * 2 > 0xffffffffLL) return ARENO_ERR_UNSUPPORTED;
  VarlenMfmaParams p;
  p.q = q;
  p.k = k;
  p.v = v;
  p.out = out;
  p.cu_seqlens = cu_seqlens;
  p.tokens = static_cast<int32_t>(tokens);
  p.num_seqs = num_seqs;
  p.q_heads = q_heads;
  p.kv_heads = kv_heads;
  p.group = group;
  p.head_parts = head_parts;
  p.fold = head_parts > 1 ? 16 : group;
  p.fold_magic = (65536 + p.fold - 1) / p.fold;
  p.block_tokens = kVmRows / p.fold;
  p.block_division = block_division(p.block_tokens);
  p.window_left = window_left;
  p.scale_log2e = softmax_scale * kLog2e;
  p.pages = pages != nullptr ? *pages : PageWrite{};
  const int64_t blocks = (tokens / p.block_tokens + num_seqs + 1) * vheads;
  if (blocks * kVmThreads > 0xffffffffLL) return ARENO_ERR_UNSUPPORTED;  // (a launch counts its work items in 32 bits)
  hipLaunchKernelGGL(l.fn, dim3(static_cast<unsigned>(blocks)), dim3(kVmThreads), l.lds_bytes,
                     static_cast<hipStream_t>(stream), p);
  return check_launch(op);
}

}  // namespace areno
