// What the kernels on 32 x 32 x 16 matrix products share (varlen_mfma.hip, attention_backward_*.hip): the products, LDS tiles that
// the memory pipe fills directly (no registers, no staging instructions), and the two ways a wave reads an operand out
// of such a tile.
//
// Layouts of v_mfma_f32_32x32x16: A is 32 rows x 16 contraction elements, lane l holds row l % 32, elements
// 8 (l / 32) .. + 7; B the same with columns for rows; C has column l % 32 and, in register i, row
// 8 (i / 4) + 4 (l / 32) + i % 4.  A C tile whose rows are the streamed index is the B operand of the next product as
// it lies: registers 8 b .. 8 b + 7 are one block of 16 streamed rows, in an order that the A operand of that product
// is read in as well (tile_columns below).
#pragma once

#include <atomic>

#include "decode_mfma_kernels.hpp"

namespace areno {

typedef __attribute__((ext_vector_type(16))) float float16_t;

template <int KIND>
struct Mfma32;
template <>
struct Mfma32<KV_BF16> {
  using elem = __bf16;
  using vec8 = bf16x8_t;
  static __device__ __forceinline__ float16_t mfma(vec8 a, vec8 b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  // c + the sum of a pair of packed values
  static __device__ __forceinline__ float add_pair(uint32_t pair, float c) {
    const bf16x2_t ones = __builtin_bit_cast(bf16x2_t, 0x3f803f80u);
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pair), ones, c, false);
  }
};
template <>
struct Mfma32<KV_F16> {
  using elem = _Float16;
  using vec8 = half8_t;
  static __device__ __forceinline__ float16_t mfma(vec8 a, vec8 b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ float add_pair(uint32_t pair, float c) {
    const half2_t ones = __builtin_bit_cast(half2_t, 0x3c003c00u);
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, pair), ones, c, false);
  }
};

// one of the two 16-bit elements of an operand's word
template <int KIND>
__device__ __forceinline__ float operand_element(uint32_t word, int hi) {
  const uint32_t bits = hi ? word >> 16 : word & 0xffffu;
  return KIND == KV_BF16 ? bf16_bits_to_float(bits) : f16_bits_to_float(bits);
}

__device__ __forceinline__ float16_t zero16() {
  float16_t z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.0f;
  return z;
}

// A tile of ROWS x D 16-bit elements in LDS, rows back to back.  The 16-byte chunks of a row are permuted by a
// function of the row, so that neither kind of read meets a bank twice: 16 lanes that read the same chunk of 16 rows,
// and 32 lanes that read four neighbouring chunks of four rows.  (The permutation is applied by the lane that fetches
// a chunk: the memory pipe writes a wave's 64 chunks back to back.)
template <int D, int ROWS, int WAVES>
struct LdsTile {
  static constexpr int kChunksPerRow = D / 8;
  static constexpr int kRowBytes = D * 2;
  static constexpr int kBytes = ROWS * kRowBytes;
  static constexpr int kFetches = kBytes / 1024 / WAVES;  // per wave, 64 chunks each
  static_assert(kBytes % (1024 * WAVES) == 0, "a tile is a whole number of fetches per wave");

  // chunk c of row r lies at place c ^ twist(r) of its group of kGroup chunks
  static constexpr int kGroup = D % 128 == 0 ? 16 : 8;  // (rows of 128 or 384 bytes: odd rows start half way round)
  static __device__ __forceinline__ int twist(int row) {
    if constexpr (kGroup == 16) return ((row & 3) << 2) | ((row >> 2) & 3);
    return (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
  }
  // byte offsets of what a lane reads, less the part that a read's constants add (rows_at, columns_at)
  static __device__ __forceinline__ uint32_t rows_base(int l32, int h) {
    return static_cast<uint32_t>(l32 * kRowBytes + ((twist(l32) ^ h) << 4));
  }
  static __device__ __forceinline__ uint32_t columns_base(int lane) {
    const int i = lane & 15, row = 4 * (lane >> 5) + (i >> 2);
    return static_cast<uint32_t>(row * kRowBytes + ((twist(row) ^ (((lane >> 3) & 2) + ((i & 3) >> 1))) << 4) + 8 * (i & 1));
  }
};

// One wave instruction that moves 64 chunks of 16 bytes from memory into LDS: lane l's chunk, at base + offset,
// lands at lds + 16 l (in m0: an operand, so that the compiler knows).  Asm, so that the compiler does not wait for it at
// the next LDS read: the caller waits (fetched_barrier) before anything is read and leaves none in flight at the
// kernel's end.
__device__ __forceinline__ void fetch_to_lds(const char* base, uint32_t offset, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(offset), "s"(base), "{m0}"(lds) : "memory");
}
// The same for the offsets of a tile that the sequence ends in.  (Another text, so that the compiler keeps the two paths
// apart instead of clamping every tile's rows.)
__device__ __forceinline__ void fetch_end_to_lds(const char* base, uint32_t offset, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 ; end" : : "v"(offset), "s"(base), "{m0}"(lds) : "memory");
}
// the same for 64 words of 4 bytes
__device__ __forceinline__ void fetch_words_to_lds(const char* base, uint32_t offset, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, %1" : : "v"(offset), "s"(base), "{m0}"(lds) : "memory");
}
// The wave's fetches have landed and its LDS reads are in registers (what a wave waits for that shares its tiles with none).
__device__ __forceinline__ void fetched() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" : : : "memory"); }
// The wave's fetches have landed and its LDS reads are in registers; then every wave's have: the tiles asked for may be
// read and the tiles read so far may be fetched over.
__device__ __forceinline__ void fetched_barrier() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory"); }

// Every wave's LDS accesses are done; fetches stay in flight.
__device__ __forceinline__ void handed_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory"); }

// The lane's number, worked out where it is needed (the sums leave no register to keep it in).
__device__ __forceinline__ int lane_now() {
  int x;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(x));
  return x;
}

__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char*)p));
}

// A operand of rows: row row0 + lane % 32 of the tile (row0 a multiple of 16), contraction elements
// 16 ks + 8 (lane / 32) .. + 7.  `base` = rows_base: the rest of the address is constant.
template <int KIND, typename T>
__device__ __forceinline__ typename Mfma32<KIND>::vec8 tile_rows(const char* tile, uint32_t base, int row0, int ks) {
  const int c = 2 * ks;
  const uint32_t off = (base ^ static_cast<uint32_t>((c % T::kGroup) << 4)) + (c / T::kGroup) * (T::kGroup * 16) + row0 * T::kRowBytes;
  return *reinterpret_cast<const typename Mfma32<KIND>::vec8*>(tile + off);
}

// A operand of columns: head elements 32 nb + lane % 32 as rows, the 16 tile rows row0 .. + 15 as the contraction index
// in the order a C tile leaves them (register order: rows 4 h .. + 3, then 8 + 4 h .. + 3).  A transposing read takes
// four rows of 16 elements per 16 lanes: lane i of the 16 supplies the address of row i / 4, elements 4 (i % 4) .. + 3,
// and receives element i of the four rows.  `base` = columns_base.
template <int KIND, typename T>
__device__ __forceinline__ typename Mfma32<KIND>::vec8 tile_columns(char* tile, uint32_t base, int row0, int nb) {
  const int c = 4 * nb;
  uint32_t w[4];
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    // (eight rows further on the twist differs by 2)
    const uint32_t off = (base ^ static_cast<uint32_t>(((c % T::kGroup) ^ (2 * half)) << 4)) + (c / T::kGroup) * (T::kGroup * 16) +
                         (row0 + 8 * half) * T::kRowBytes;
    const uint2_t u = __builtin_bit_cast(uint2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(tile + off)));
    w[2 * half] = u[0];
    w[2 * half + 1] = u[1];
  }
  return __builtin_bit_cast(typename Mfma32<KIND>::vec8, uint4_t{w[0], w[1], w[2], w[3]});
}

// Rows of 16-bit elements on their way from a wave's registers to memory, through a part of LDS that is the wave's alone: a
// lane of a C tile holds four elements here and there of a row, and stored from there they are 64 pieces of 8 bytes an
// instruction, which the memory pipe takes one by one.  The 16-byte chunks of a row are permuted by a function of the row, so
// that lanes that put the same chunk of different rows meet different banks.
template <int CHUNKS>  // of a row
struct RowStage {
  static constexpr int kRowBytes = CHUNKS * 16;
  static constexpr int kTwist = (CHUNKS & (CHUNKS - 1)) == 0 ? CHUNKS - 1 : 3;
  static_assert(CHUNKS % 4 == 0, "the twist stays inside a row");
  static __device__ __forceinline__ char* place(char* stage, int row, int chunk) {
    return stage + row * kRowBytes + ((chunk ^ (row & kTwist)) << 4);
  }
  // four elements, the first or (`half`) the second ones of a chunk
  static __device__ __forceinline__ void put(char* stage, int row, int chunk, int half, uint32_t lo, uint32_t hi) {
    *reinterpret_cast<uint2_t*>(place(stage, row, chunk) + 8 * half) = uint2_t{lo, hi};
  }
  // The rows that were put, chunk by chunk: store(row, chunk, its 16 bytes), a row's lanes next to each other.  (The wave's LDS
  // accesses take place in their order.)
  template <int ROWS, typename Store>
  static __device__ __forceinline__ void take(char* stage, int lane, const Store& store) {
    static_assert(ROWS * CHUNKS % 64 == 0, "whole instructions");
    asm volatile("" : : : "memory");
#pragma unroll
    for (int x = 0; x < ROWS * CHUNKS / 64; ++x) {
      const int i = x * 64 + lane, row = i / CHUNKS, chunk = i % CHUNKS;
      store(row, chunk, *reinterpret_cast<const uint4_t*>(place(stage, row, chunk)));
    }
    asm volatile("" : : : "memory");
  }
};

// more than 64 KB of LDS has to be allowed once per device; one bit per device (the attribute belongs to the device's copy)
template <int BYTES>
bool allow_lds(const void* fn, std::atomic<uint64_t>& allowed_on) {
  if constexpr (BYTES > 64 * 1024) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return false;
    if ((allowed_on.load(std::memory_order_acquire) >> device & 1) == 0) {
      if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, BYTES) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
      allowed_on.fetch_or(uint64_t{1} << device, std::memory_order_release);
    }
  }
  return true;
}

}  // namespace areno
