// Rows of a paged cache into LDS without passing registers, and the chunk order in which they lie there.  Included by
// sink_attn.hip.
#pragma once

#include "lds_copy.h"

namespace hymeta {
namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

// Lane (g4 = lane / 16, n = lane % 16) of the result: column n of the block of 4 keys x 16 columns its 16 lanes address, 4
// columns a lane.
__device__ __forceinline__ bf16x4 read_transposed(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_bf16x4*)(p));
}

// Rows lie in LDS one behind the other, `Chunks` 16-byte chunks each.  A fragment read asks for the same chunk of 16 rows at
// once, a transposed read for four neighbouring chunks of 4 rows; a chunk's number is XOR-ed with bits of its row so that
// either spreads over all banks (16 chunks of 16 bytes): the two low bits of the row move groups of four chunks, where the
// pitch does not do that already, the next two the chunks within a group.
template <int Chunks>
struct ChunkOrder {
  static_assert(Chunks % 4 == 0, "rows of whole 64 bytes");
  static __device__ __forceinline__ int twist(int row) {
    const int within = (row >> 2) & 3;
    if (Chunks % 16 == 0) return ((row & 3) << 2) | within;
    if (Chunks % 16 == 8) return ((row & 2) << 1) | within;
    return within;
  }
};

// Keys [j0, j0 + Keys) of a sequence into an LDS image of Keys rows of Chunks chunks (KeyChunks of the key, then those of the
// value, if it lies elsewhere in the cache row), by waves `wave` of `Waves`; keys past `last` repeat it (their weights are
// zero).  Tiles start at multiples of Keys; pages hold a power of two of rows.
template <int KeyChunks, int ValueChunks, int Keys, int Waves>
struct RowCopy {
  static constexpr int kChunks = KeyChunks + ValueChunks, kInstr = Keys * kChunks / 64, kPerWave = (kInstr + Waves - 1) / Waves;
  typedef ChunkOrder<kChunks> Order;
  static_assert(Keys * kChunks % 64 == 0, "whole instructions");
  const char* cache;              // the cache, at the head's key
  const int32_t* bt;
  int64_t row_bytes;
  int value_off;                  // from the key to the value, in bytes
  int shift, mask, wave;
  uint32_t place[kPerWave];       // this lane's byte offset from the tile's first row, per instruction

  __device__ __forceinline__ RowCopy(const void* cache_, int64_t row_bytes_, int64_t key_off, int value_off_, int block_size, const int32_t* tables, int wave_)
      : cache(static_cast<const char*>(cache_) + key_off), bt(tables), row_bytes(row_bytes_), value_off(value_off_),
        shift(__builtin_ctz(block_size)), mask(block_size - 1), wave(wave_) {
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
      const int chunk = 64 * (wave + Waves * i) + (threadIdx.x & 63), row = chunk / kChunks;
      place[i] = static_cast<uint32_t>(row * row_bytes) + inside(chunk % kChunks, row);
    }
  }
  // byte offset, from the key, of what lies at chunk `slot` of row `row` of the image
  __device__ __forceinline__ uint32_t inside(int slot, int row) const {
    const int c = slot ^ Order::twist(row);
    return static_cast<uint32_t>(ValueChunks == 0 || c < KeyChunks ? 16 * c : value_off + 16 * (c - KeyChunks));
  }
  __device__ __forceinline__ void issue(int j0, int last, char* image) const {
    if (mask + 1 >= Keys) {
      const int64_t row = (static_cast<int64_t>(__builtin_amdgcn_readfirstlane(bt[j0 >> shift])) << shift) + (j0 & mask);
      const char* base = cache + row * row_bytes;
      if (j0 + Keys - 1 <= last) {
#pragma unroll
        for (int i = 0; i < kPerWave; ++i)
          if (kInstr % Waves == 0 || wave + Waves * i < kInstr) copy16_to_lds(base, place[i], image + 1024 * (wave + Waves * i));
        return;
      }
      for (int at = wave; at < kInstr; at += Waves) {
        const int chunk = 64 * at + (threadIdx.x & 63), r = chunk / kChunks;
        copy16_to_lds(base + min(r, last - j0) * row_bytes + inside(chunk % kChunks, r), image + 1024 * at);
      }
      return;
    }
    for (int at = wave; at < kInstr; at += Waves) {          // small pages: every row's page is looked up
      const int chunk = 64 * at + (threadIdx.x & 63), r = chunk / kChunks, j = min(j0 + r, last);
      const int64_t row = (static_cast<int64_t>(bt[j >> shift]) << shift) + (j & mask);
      copy16_to_lds(cache + row * row_bytes + inside(chunk % kChunks, r), image + 1024 * at);
    }
  }
};

}  // namespace
}  // namespace hymeta
