// Attention over rows whose value is the first C elements of a key of C + 64 (HYMETA_KV_VALUE_IN_KEY), C = 256, 384 or
// 512, bf16 on the matrix cores: one pass over the keys for all the value columns.  Included by sink_attn.hip.
//
// A wave cannot hold the queries of its rows (D registers of 4 bytes per 2 elements: 72 at C = 512 for 16 rows) beside
// accumulators of all C value columns of enough rows to reuse what it reads from LDS.  In a prompt a workgroup of 8
// waves therefore splits its work in two ways: for the scores every wave owns 16 of the workgroup's 128 rows, for the
// weighted values every wave owns C / 8 of the columns of ALL 128 rows, and the weights pass from the first to the
// second through LDS, as the fragments the second product reads.  Each score is computed once, and what is read from LDS
// is used by 8 row blocks.
//
// Key rows lie in LDS as they lie in the pages, copied there without passing registers; the values are read from the same
// image, transposed by the LDS read itself.  16-byte chunks of row R are XOR-ed with (R / 2) % 8 within their group of 8
// chunks: with the row pitch an odd multiple of 128 bytes that spreads the 16 rows of a fragment read, and the 4 rows of
// a transposed read, over all banks.
#pragma once

#include <type_traits>

#include "row_attn.h"

namespace hymeta {
namespace {

// Scores of a lane's row against N keys at distances dist - i in the base-2 domain (scores times log2 e; the bias'
// coefficient is the same in both), from the products of the query with the keys.
template <int N>
__device__ __forceinline__ void finish_scores(const hymeta_sink_attention_args& a, float (&s)[N], float dist, float ba, float bb) {
  if (a.softcap > 0.f) {
    const float cap_in = a.scale / a.softcap, cap2 = a.softcap * 1.4426950408889634f;
#pragma unroll
    for (int i = 0; i < N; ++i) s[i] = cap2 * tanh_fast(s[i] * cap_in);
  } else {
    const float scale2 = a.scale * 1.4426950408889634f;
#pragma unroll
    for (int i = 0; i < N; ++i) s[i] *= scale2;
  }
  if (a.bias_mode == HYMETA_BIAS_LOG_DISTANCE) {
#pragma unroll
    for (int i = 0; i < N; ++i) s[i] = fmaf(-ba, __log2f(fmaf(bb, dist - static_cast<float>(i), 1.f)), s[i]);
  }
}

// Tiles of Keys keys of a sequence's key/value head into LDS images of Keys rows of D elements, by waves `wave` of `Waves`.  Pages
// hold a power of two of rows.  An instruction takes 64 chunks of 16 bytes; those of 8 rows (D / 64 instructions) repeat from 8
// rows to 8 rows but for a chunk's place, and with the row pitch an odd multiple of 128 bytes that differs in one bit: the lanes'
// places of 8 rows are enough.  Where a tile's first row lies is looked up for 64 tiles at once:
// a load in front of every tile's copies waits for all that are on their way.  So does a register that lies in scratch memory;
// with 512 + 64 the prompts' form has none left over, works its places out on every tile and parks the queries' last two steps in
// LDS.  8192 rows x 16 heads on 512 + 64 1618 -> 1440 us, a decode step of 64 sequences x 4096 70.8 -> 64.4.
template <int D, int Keys, int Waves>
struct LatentCopy {
  static constexpr int kChunks = D / 8, kInstr = Keys * kChunks / 64, kEight = kChunks / 8;
  static constexpr int kShare = Waves == 1 ? 1 : Waves / (Keys / 8), kPlaces = (kEight + kShare - 1) / kShare;       // waves to 8 rows
  static_assert(kChunks % 16 == 8 && Keys % 8 == 0 && (Waves == 1 || Waves == kShare * (Keys / 8)), "the row pitch is an odd multiple of 128 bytes");
  const char* cache;
  const int32_t* bt;
  int64_t row_bytes;
  int shift, mask, wave;
  static constexpr bool kKept = Waves == 1;       // the lanes' places are kept: where eight waves share a tile, registers are short
  uint32_t place[kKept ? kPlaces : 1];
  int tile_row;                   // lane = tile % 64: the cache row of a tile's first key, for 64 tiles from the last refill on

  __device__ __forceinline__ LatentCopy(const hymeta_sink_attention_args& a, const int32_t* tables, int g, int wave_)
      : cache(static_cast<const char*>(a.kv_cache) + static_cast<int64_t>(g) * D * 2), bt(tables),
        row_bytes(static_cast<int64_t>(a.num_kv_heads) * D * 2), shift(__builtin_ctz(a.block_size)), mask(a.block_size - 1), wave(wave_), tile_row(0) {
  }
  // this lane's byte offset from the tile's first row in the wave's i-th instruction over its 8 rows
  __device__ __forceinline__ uint32_t place_of(int i, int lane) const {
    const int eight = wave / kShare, chunk = 64 * (wave % kShare + kShare * i) + lane;
    const int r = static_cast<int>(__umul24(chunk >> 3, (512 + kEight - 1) / kEight) >> 9);          // chunk / kChunks below 8 rows
    const int pos = chunk - r * kChunks;
    return __umul24(8 * eight + r, static_cast<uint32_t>(row_bytes)) + 16 * (pos ^ ((4 * eight + (r >> 1)) & 7));
  }
  // whether tiles of Keys rows of one page can be copied from lanes' 32-bit offsets
  __device__ __forceinline__ bool fits() const { return mask + 1 >= Keys && row_bytes < (1 << 24); }
  // (a tile behind the last key: that one's row)
  template <typename F>
  __device__ __forceinline__ void refill(int t, int tiles, int last, const F& key_of, bool begin = false) {
    const int tile = t + ((static_cast<int>(threadIdx.x) - t) & 63);
    if (tile < tiles) {
      const int j = min(key_of(tile), last);
      tile_row = (bt[j >> shift] << shift) + (j & mask);
    }
    if constexpr (kKept) {
      if (begin) {                                // (under the load)
#pragma unroll
        for (int i = 0; i < kPlaces; ++i) place[i] = place_of(i, threadIdx.x & 63);
      }
    }
    asm volatile("" : "+v"(tile_row));            // (waited for here and not on every tile)
  }
  // tile t, all of it in one page and seen by some row
  __device__ __forceinline__ void issue_whole(int t, char* image) const {
    const char* base = cache + static_cast<int64_t>(__builtin_amdgcn_readlane(tile_row, t & 63)) * row_bytes;
    if constexpr (Waves == 1) {
#pragma unroll
      for (int e = 0; e < Keys / 8; ++e) {
#pragma unroll
        for (int i = 0; i < kEight; ++i) copy16_to_lds(base, e & 1 ? place[i] ^ 64 : place[i], image + 1024 * (kEight * e + i));
        base += 8 * row_bytes;
      }
    } else {
      char* rows = image + 1024 * (kEight * (wave / kShare) + wave % kShare);
      int lane = threadIdx.x & 63;
      asm volatile("" : "+v"(lane));              // (worked out here each time)
#pragma unroll
      for (int i = 0; i < kPlaces; ++i)
        if (kEight % kShare == 0 || i + 1 < kPlaces || wave % kShare < kEight % kShare) copy16_to_lds(base, place_of(i, lane), rows + 1024 * kShare * i);
    }
  }
  // tile t with its rows past the first `rows` repeating the last of those (their weights are zero)
  __device__ __forceinline__ void issue_part(int t, int rows, char* image) const {
    const char* base = cache + static_cast<int64_t>(__builtin_amdgcn_readlane(tile_row, t & 63)) * row_bytes;
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));                // (nothing of this is kept in registers over the other tiles)
    for (int at = wave; at < kInstr; at += Waves) {
      const int chunk = 64 * at + lane, row = chunk / kChunks;
      copy16_to_lds(base, __umul24(min(row, rows - 1), static_cast<uint32_t>(row_bytes)) + 16 * ((chunk % kChunks) ^ ((row >> 1) & 7)), image + 1024 * at);
    }
  }
  // pages that do not fit: keys [j0, j0 + Keys), those past `last` repeating it
  __device__ __forceinline__ void issue(int j0, int last, char* image) const {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));                // (nothing of this is kept in registers over the other tiles)
    for (int at = wave; at < kInstr; at += Waves) {
      const int chunk = 64 * at + lane, row = chunk / kChunks, j = min(j0 + row, last);
      const int64_t src = (static_cast<int64_t>(bt[j >> shift]) << shift) + (j & mask);
      copy16_to_lds(cache + src * row_bytes + 16 * ((chunk % kChunks) ^ ((row >> 1) & 7)), image + 1024 * at);
    }
  }
};

constexpr int kWideWaves = 8, kWideRows = 16 * kWideWaves;
static_assert(kWideRows == kPortionRows, "the merge finds a row's block");

template <int C>
struct WideSmem {
  static constexpr int kImage = kWideKeys * (C + 64) * 2;
  static constexpr int kParked = C == 512 ? 2 : 0;      // the queries' last steps that find no registers
  char k[3][kImage];                              // tiles t, t + 1 and, on its way, t + 2
  u32x4 q[kParked ? kWideWaves : 1][kParked ? kParked : 1][64];
  u32x4 p[2][kWideWaves][2][64];                  // weights of a tile, high and low bf16 parts, by row block and lane
  float corr[2][kWideRows];                       // what a row's sums so far are multiplied with before the tile
  int moved[2][kWideWaves];                       // whether a row block has any factor but 1
};

// Portions of prompts: grid = their blocks of 128 rows x slices of the keys at most x key/value heads; a row is a (query, head)
// pair, the heads of a key/value head side by side, so that a portion of a few tokens fills its blocks.  Sequences with one row
// are left to the decode form.
//
// Per tile of 32 keys a workgroup issues 800 matrix instructions (C = 512) against 480 LDS reads of 1 KB; a step computes
// the scores of tile t + 1 and adds tile t's values, which do not depend on each other: the two waves of a SIMD do them in
// opposite order, so that one's softmax runs under the other's products.  One barrier per tile.  Bound by the matrix
// and the vector pipes, busy 51 and 40 % of the time (the waves wait 29 % of theirs): 8192 rows x 16 heads on 512 + 64: 1.44 ms = 1.20
// PFLOP/s of the products issued (both parts of the weights counted), where launches over value slices of 128, each repeating the
// scores, took 11.3 ms.  Fragments of the keys three ahead (two and five: level).  Plain: neither a bias nor a cap on the scores.
template <int C, bool Plain>
__global__ __launch_bounds__(64 * kWideWaves) void latent_prefill_kernel(hymeta_sink_attention_args a, PortionSlices ps) {
  constexpr int D = C + 64, kRowB = 2 * D, kSteps = D / 32, CB = C / 128, kParked = WideSmem<C>::kParked, kAhead = 3;
  __shared__ __attribute__((aligned(16))) WideSmem<C> sm;
  const int group = a.num_heads / a.num_kv_heads, g = blockIdx.x % a.num_kv_heads, item = blockIdx.x / a.num_kv_heads, split = item % ps.splits;
  const PieceAt block = portion_block(a, item / ps.splits, ps);
  const int s = block.seq, row0 = block.row0, q = block.rows, rows = q * group;
  if (s < 0) return;
  const int r0 = ((rows - 1) / kWideRows - block.index) * kWideRows;        // (the longest rows first)
  const int lane = threadIdx.x & 63, n = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ctx = a.seq_lens[s] - q;

  // this lane's row for the scores
  const int r = r0 + 16 * wave + n;
  const bool ok = r < rows;
  const int qi = ok ? r / group : 0, h = g * group + (ok ? r % group : 0);
  const int pos = ok ? ctx + qi : -1;
  const float ba = !Plain && a.bias_mode ? a.bias_a[h] : 0.f, bb = !Plain && a.bias_mode == HYMETA_BIAS_LOG_DISTANCE ? a.bias_b[h] : 0.f;
  bf16x8 qf[kSteps - kParked];
  {
    const uint16_t* qrow = static_cast<const uint16_t*>(a.q) + static_cast<int64_t>(row0 + qi) * a.q_stride_t + static_cast<int64_t>(h) * D;
#pragma unroll
    for (int st = 0; st < kSteps; ++st) {
      const u32x4 x = ok ? ld16g(qrow + 32 * st + 8 * g4) : u32x4{0u, 0u, 0u, 0u};
      if (st < kSteps - kParked) qf[st] = __builtin_bit_cast(bf16x8, x);
      else sm.q[wave][st - (kSteps - kParked)][lane] = x;
    }
  }
  // positions the block's and the wave's rows span
  const int p_hi = ctx + (min(rows, r0 + kWideRows) - 1) / group;
  const int w_lo = ctx + min(rows - 1, r0 + 16 * wave) / group, w_hi = ctx + min(rows - 1, r0 + 16 * wave + 15) / group;
  const int w_first = first_key(a, w_hi);
  const bool full = r0 + 16 * wave + 16 <= rows;
  const BlockKeys keys = block_keys<kWideKeys>(a, ctx + r0 / group, p_hi);
  const int splits = keys.slices(ps);
  if (split >= splits) return;
  const bool sink = a.sink && splits == 1;            // (of several slices of the keys none has the sink: the merge adds it)
  float m = sink ? (a.sink_logits ? a.sink_logits[h] * 1.4426950408889634f : 0.f) : -INFINITY;
  float l = sink && g4 == 0 ? 1.f : 0.f;              // the sink's exp(m - m), counted once per row
  const int per = (keys.tiles + splits - 1) / splits, t0 = split * per, tiles = min(keys.tiles - t0, per);          // this slice's
  auto key0 = [&](int t) { return keys.first(t0 + t); };

  f32x4v o[kWideWaves][CB];                           // O^T: this wave's columns x the rows of block rb
#pragma unroll
  for (int rb = 0; rb < kWideWaves; ++rb)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) o[rb][cb] = f32x4v{0.f, 0.f, 0.f, 0.f};

  LatentCopy<D, kWideKeys, kWideWaves> copy(a, a.block_tables + static_cast<int64_t>(s) * a.block_table_stride, g, wave);
  // LDS offsets of this lane's fragments: keys (even and odd 32-element steps), values
  const int swz = (n >> 1) & 7;
  // (the others are one bit away, and worked out where they are used: registers are short)
  const int koff = n * kRowB + 16 * (g4 ^ swz);
  const int vrow = 4 * g4 + (n >> 2);
  auto value_place = [&](int block) __attribute__((always_inline)) {
    return vrow * kRowB + 16 * ((2 * block + ((n & 3) >> 1)) ^ ((vrow >> 1) & 7)) + 8 * (n & 1);
  };
  const int voff = value_place(wave * CB);
  const float scale2 = a.scale * 1.4426950408889634f;
  auto scores = [&](int t, const char* img, int buf) {
    const int j0 = key0(t);
    f32x4v acc[2] = {};
    // fragment f: step f / 2 of the head, keys 16 (f % 2) ..; kAhead of them ahead
    u32x4 kf[kAhead + 1];
    bf16x8 parked[kParked + 1];
    int even = koff;
    asm volatile("" : "+v"(even));
    const int odd = even ^ 64;
    auto load = [&](int f) __attribute__((always_inline)) {
      const int st = f >> 1, late = st - (kSteps - kParked);
      kf[f % (kAhead + 1)] = ld16(img + (st & 1 ? odd : even) + (f & 1) * 16 * kRowB + (st >> 1) * 128);
      if (late >= 0 && (f & 1) == 0) parked[late < 0 ? 0 : late] = __builtin_bit_cast(bf16x8, sm.q[wave][late < 0 ? 0 : late][lane]);
    };
#pragma unroll
    for (int f = 0; f < kAhead; ++f) load(f);
#pragma unroll
    for (int f = 0; f < 2 * kSteps; ++f) {
      if (f + kAhead < 2 * kSteps) load(f + kAhead);
      __builtin_amdgcn_sched_barrier(0);
      const int st = f >> 1, late = st - (kSteps - kParked);
      acc[f & 1] = mfma16(__builtin_bit_cast(bf16x8, kf[f % (kAhead + 1)]), late < 0 ? qf[late < 0 ? st : 0] : parked[late < 0 ? 0 : late], acc[f & 1]);
    }
    // the lane holds the scores of its row against keys j0 + 16 ks + 4 g4 + e
    const bool masked = !(full && j0 + kWideKeys - 1 <= w_lo && j0 >= w_first);
    float sc[2][4], mx = -INFINITY;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int e = 0; e < 4; ++e) sc[ks][e] = acc[ks][e];
      if constexpr (Plain) {
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[ks][e] *= scale2;
      } else {
        finish_scores(a, sc[ks], static_cast<float>(pos - (j0 + 16 * ks + 4 * g4)), ba, bb);
      }
    }
    if (masked) {
      const int first = first_key(a, pos);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = j0 + 16 * ks + 4 * g4 + e;
          sc[ks][e] = (j <= pos && (j >= first || j < a.keep_first)) ? sc[ks][e] : -INFINITY;
        }
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = fmaxf(mx, sc[ks][e]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const bool up = mx > m + kLazyMax2;               // (from -inf: at the first visible key)
    float corr = 1.f;
    if (up) {
      corr = __builtin_amdgcn_exp2f(m - mx);
      m = mx;
    }
    const float ref = m == -INFINITY ? 0.f : m;       // nothing visible yet: every weight is exp2(-inf) = 0
    float sum = 0.f;
    u32x4 hi, lo;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float p0 = __builtin_amdgcn_exp2f(sc[ks][2 * e] - ref), p1 = __builtin_amdgcn_exp2f(sc[ks][2 * e + 1] - ref);
        sum += p0 + p1;
        const uint32_t w = pack_bf16x2(p0, p1);
        hi[2 * ks + e] = w;
        lo[2 * ks + e] = pack_bf16x2(p0 - lo_bf(w), p1 - hi_bf(w));
      }
    l = l * corr + sum;
    sm.p[buf][wave][0][lane] = hi;
    sm.p[buf][wave][1][lane] = lo;
    if (g4 == 0) sm.corr[buf][16 * wave + n] = corr;
    const int any = __any(up);
    if (lane == 0) sm.moved[buf][wave] = any;
  };
  auto values = [&](const char* img, int buf) {
    bf16x8 vf[CB];
    int at = voff;
    asm volatile("" : "+v"(at));
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      // columns 16 (wave CB + cb) ..: CB runs of 2 chunks, 4 runs to a group of 8 chunks (CB = 3: not on its boundary)
      const int col = 4 % CB == 0 ? at ^ (32 * cb) : value_place(wave * CB + cb);
      const bf16x4 v0 = read_transposed(img + col), v1 = read_transposed(img + col + 16 * kRowB);
      vf[cb] = bf16x8{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
    }
    int moved = 0;
#pragma unroll
    for (int rb = 0; rb < kWideWaves; ++rb) moved |= sm.moved[buf][rb];
    if (__builtin_amdgcn_readfirstlane(moved)) {
#pragma unroll
      for (int rb = 0; rb < kWideWaves; ++rb) {
        const float f = sm.corr[buf][16 * rb + n];
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) o[rb][cb] *= f;
      }
    }
    u32x4 pf[2][2];
#pragma unroll
    for (int part = 0; part < 2; ++part) pf[0][part] = sm.p[buf][0][part][lane];
#pragma unroll
    for (int rb = 0; rb < kWideWaves; ++rb) {
      if (rb + 1 < kWideWaves) {
#pragma unroll
        for (int part = 0; part < 2; ++part) pf[(rb + 1) & 1][part] = sm.p[buf][rb + 1][part][lane];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int part = 0; part < 2; ++part)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) o[rb][cb] = mfma16(vf[cb], __builtin_bit_cast(bf16x8, pf[rb & 1][part]), o[rb][cb]);
    }
  };

  const bool fits = copy.fits();
  const int whole = p_hi + 1 - key0(tiles - 1) >= kWideKeys ? tiles : tiles - 1, looked_up = fits ? tiles : 0;
  auto copy_tile = [&](int t, char* image) __attribute__((always_inline)) {
    if (!fits) copy.issue(key0(t), p_hi, image);
    else if (t < whole) copy.issue_whole(t, image);
    else copy.issue_part(t, p_hi + 1 - key0(t), image);
  };
  if (tiles > 0) {
    copy.refill(0, looked_up, p_hi, key0);
    copy_tile(0, sm.k[0]);
    if (tiles > 1) copy_tile(1, sm.k[1]);
    copies_landed_barrier();
    scores(0, sm.k[0], 0);
    copies_landed_barrier();
  }
  auto walk = [&](auto scores_first) {
    constexpr bool kScoresFirst = decltype(scores_first)::value;
    int i0 = 0, i1 = 1, i2 = 2;
    for (int t = 0; t < tiles; ++t) {
      // image i2 held tile t - 1, read for the last time before the barrier
      if (t + 2 < tiles) copy_tile(t + 2, sm.k[i2]);
      if (!kScoresFirst) values(sm.k[i0], t & 1);
      if (t + 1 < tiles) scores(t + 1, sm.k[i1], (t + 1) & 1);
      if (kScoresFirst) values(sm.k[i0], t & 1);
      if ((t & 31) == 29) copy.refill(t + 3, looked_up, p_hi, key0);
      copies_landed_barrier();
      const int i = i0;
      i0 = i1, i1 = i2, i2 = i;
    }
  };
  if (wave < kWideWaves / 2) walk(std::true_type{});
  else walk(std::false_type{});
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (splits > 1) {
    float* parts = ps.parts + split * partial_row_floats(C);
    const size_t stride = ps.splits * partial_row_floats(C);
    if (g4 == 0 && ok) {
      float* part = parts + (static_cast<size_t>(row0 + qi) * a.num_heads + h) * stride;
      part[C] = m, part[C + 1] = l;
    }
#pragma unroll
    for (int rb = 0; rb < kWideWaves; ++rb) {
      const int ro = r0 + 16 * rb + n;
      if (ro >= rows) continue;
      float* part = parts + (static_cast<size_t>(row0 + ro / group) * a.num_heads + g * group + ro % group) * stride + wave * 16 * CB;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) *reinterpret_cast<f32x4v*>(part + 16 * cb + 4 * g4) = o[rb][cb];
    }
    return;
  }
  if (g4 == 0) {
    float inv = l > 0.f ? 1.f / l : 0.f;
    if (a.head_gate && ok) inv *= sigmoid_exact(bf2f(static_cast<const uint16_t*>(a.head_gate)[static_cast<int64_t>(row0 + qi) * a.head_gate_stride_t + h]));
    sm.corr[0][16 * wave + n] = inv;
  }
  __syncthreads();
#pragma unroll
  for (int rb = 0; rb < kWideWaves; ++rb) {
    const int ro = r0 + 16 * rb + n;
    if (ro >= rows) continue;
    const int64_t token = row0 + ro / group;
    const int64_t col = static_cast<int64_t>(g * group + ro % group) * C + wave * 16 * CB;
    const float inv = sm.corr[0][16 * rb + n];
    uint16_t* out = static_cast<uint16_t*>(a.out) + token * a.num_heads * C + col;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      f32x4v v = o[rb][cb] * inv;
      if (a.elem_gate) {
        float gate[4];
        ActBf16::ld4(static_cast<const uint16_t*>(a.elem_gate) + token * a.elem_gate_stride_t + col + 16 * cb + 4 * g4, gate);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= ActBf16::sigmoid(gate[e]);
      }
      *reinterpret_cast<u32x2*>(out + 16 * cb + 4 * g4) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    }
  }
}

// Decode: a workgroup of 4 waves per (sequence with one row, key/value head, slice of the keys, slice of 16 query heads).
// Every wave is on its own until the end: it takes 16 of each tile's 64 keys, copies them into an LDS ring of its own two
// tiles ahead of their use and keeps statistics and all C value columns of its rows; no barrier stands between the copies.
// The waves' sums are merged through LDS (a tree of two steps) into one partial per slice.  Two row blocks in a wave (28
// heads) need 400 registers, of which 256 can be addressed by everything but the matrix instructions: the compiler spills
// 460.  The head slices of a (sequence, slice of keys) follow each other on one die instead, whose L2 has the keys for the
// second.  Bound by memory, and by what stands around a slice's few tiles (queries, first tile, merge): 64 sequences x 4096 keys
// of 512 + 64, 16 heads: 64 us, 53 of them this kernel (4.8 TB/s), where four launches over value slices took 280.
constexpr int kLatentWaves = 4, kLatentKeys = 16, kLatentHeads = 16;

template <int C>
struct LatentDecodeSmem {
  static constexpr int kStage = kLatentKeys * (C + 64) * 2, kRowF = C + 4;
  static constexpr int kRing = 2 * kLatentWaves * kStage, kMerge = 2 * kLatentHeads * kRowF * 4;
  char bytes[kRing > kMerge ? kRing : kMerge];
};

template <int C>
__global__ __launch_bounds__(64 * kLatentWaves) void latent_decode_kernel(hymeta_sink_attention_args a, int splits) {
  constexpr int D = C + 64, kRowB = 2 * D, kSteps = D / 32, kTile = kLatentWaves * kLatentKeys;
  typedef LatentDecodeSmem<C> Smem;
  __shared__ __attribute__((aligned(16))) Smem sm;
  const int group = a.num_heads / a.num_kv_heads, slices = (group + kLatentHeads - 1) / kLatentHeads;
  // workgroups go to the chip's 8 dies round robin by their number
  const int turn = blockIdx.x >> 3, item = (turn / slices) * 8 + (blockIdx.x & 7);
  if (item >= a.num_seqs * a.num_kv_heads * splits) return;
  const int h_first = (turn % slices) * kLatentHeads, h_count = min(kLatentHeads, group - h_first);
  const int split = item % splits, g = item / splits % a.num_kv_heads, s = item / splits / a.num_kv_heads;
  const int t = a.query_start_loc[s];
  if (a.query_start_loc[s + 1] - t != 1) return;
  const int pos = a.seq_lens[s] - 1;
  const int lane = threadIdx.x & 63, n = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the sequence's tiles of 64 keys: those of the kept first keys that lie before the window's first tile, then the window's
  const int first = first_key(a, pos);
  const int from = first / kTile * kTile;
  const int kept = bounded(a) ? min((a.keep_first + kTile - 1) / kTile * kTile, from) / kTile : 0;
  const int tiles = pos < 0 ? 0 : kept + (pos - from) / kTile + 1, per = (tiles + splits - 1) / splits;
  const int v_lo = split * per, v_hi = min(tiles, v_lo + per) - 1;
  auto key0 = [&](int v) { return (v < kept ? v * kTile : from + (v - kept) * kTile) + kLatentKeys * wave; };

  // (in front of the queries, whose loads the first tile's copies would otherwise wait for)
  LatentCopy<D, kLatentKeys, 1> copy(a, a.block_tables + static_cast<int64_t>(s) * a.block_table_stride, g, 0);
  const bool fits = copy.fits();
  const int looked_up = fits ? v_hi + 1 : 0;
  if (v_lo <= v_hi) copy.refill(v_lo, looked_up, pos, key0, true);
  bf16x8 qf[kSteps];
  f32x4v o[C / 16];
  float m = -INFINITY, l = 0.f;
  const bool ok = n < h_count;
  const int h = g * group + h_first + (ok ? n : 0);
  const float ba = a.bias_mode ? a.bias_a[h] : 0.f, bb = a.bias_mode == HYMETA_BIAS_LOG_DISTANCE ? a.bias_b[h] : 0.f;
  {
    const uint16_t* qrow = static_cast<const uint16_t*>(a.q) + static_cast<int64_t>(t) * a.q_stride_t + static_cast<int64_t>(h) * D;
#pragma unroll
    for (int st = 0; st < kSteps; ++st) qf[st] = ok ? __builtin_bit_cast(bf16x8, ld16g(qrow + 32 * st + 8 * g4)) : bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
  }
#pragma unroll
  for (int cb = 0; cb < C / 16; ++cb) o[cb] = f32x4v{0.f, 0.f, 0.f, 0.f};
  constexpr int kLoads = LatentCopy<D, kLatentKeys, 1>::kInstr;
  char* ring = sm.bytes + wave * 2 * Smem::kStage;
  const int swz = (n >> 1) & 7;
  const int koff[2] = {n * kRowB + 16 * (g4 ^ swz), n * kRowB + 16 * ((4 + g4) ^ swz)};
  int voff[4];                                        // columns 16 cb: chunks 2 cb, 2 cb + 1; four cb to a group of 8 chunks
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    const int R = 4 * g4 + (n >> 2);
    voff[cb] = R * kRowB + 16 * ((2 * cb + ((n & 3) >> 1)) ^ ((R >> 1) & 7)) + 8 * (n & 1);
  }

  // (a wave whose 16 keys lie past the last one copies the last one and skips them)
  const int whole = key0(tiles - 1) + kLatentKeys - 1 <= pos ? tiles : tiles - 1;
  auto copy_tile = [&](int v, char* image) __attribute__((always_inline)) {
    if (!fits) copy.issue(min(key0(v), pos), pos, image);
    else if (v < whole) copy.issue_whole(v, image);
    else copy.issue_part(v, max(1, pos + 1 - key0(v)), image);
  };
  if (v_lo <= v_hi) {
    copy_tile(v_lo, ring);
    if (v_lo < v_hi) copy_tile(v_lo + 1, ring + Smem::kStage);
  }
  for (int v = v_lo; v <= v_hi; ++v) {
    const int j0 = key0(v);
    char* img = ring + ((v - v_lo) & 1) * Smem::kStage;
    if (v < v_hi) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (j0 <= pos) {
      f32x4v acc[2] = {};
#pragma unroll
      for (int st = 0; st < kSteps; ++st)
        acc[st & 1] = mfma16(__builtin_bit_cast(bf16x8, ld16(img + koff[st & 1] + (st >> 1) * 128)), qf[st], acc[st & 1]);
      // the lane holds the scores of its row against keys j0 + 4 g4 + e
      float sc[4], mx = -INFINITY;
#pragma unroll
      for (int e = 0; e < 4; ++e) sc[e] = acc[0][e] + acc[1][e];
      finish_scores(a, sc, static_cast<float>(pos - (j0 + 4 * g4)), ba, bb);
      if (!(j0 + kLatentKeys - 1 <= pos && j0 >= first)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = j0 + 4 * g4 + e;
          sc[e] = (j <= pos && (j >= first || j < a.keep_first)) ? sc[e] : -INFINITY;
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = fmaxf(mx, sc[e]);
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const bool up = mx > m + kLazyMax2;
      if (__any(up)) {
        const float corr = up ? __builtin_amdgcn_exp2f(m - mx) : 1.f;
        m = up ? mx : m;
        l *= corr;
#pragma unroll
        for (int cb = 0; cb < C / 16; ++cb) o[cb] *= corr;
      }
      const float ref = m == -INFINITY ? 0.f : m;     // nothing visible yet: every weight is exp2(-inf) = 0
      u32x2 hi, lo;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float p0 = __builtin_amdgcn_exp2f(sc[2 * e] - ref), p1 = __builtin_amdgcn_exp2f(sc[2 * e + 1] - ref);
        l += p0 + p1;
        hi[e] = pack_bf16x2(p0, p1);
        lo[e] = pack_bf16x2(p0 - lo_bf(hi[e]), p1 - hi_bf(hi[e]));
      }
      const bf16x4 ph = __builtin_bit_cast(bf16x4, hi), pl = __builtin_bit_cast(bf16x4, lo);
#pragma unroll
      for (int cb = 0; cb < C / 16; ++cb) {
        const bf16x4 vf = read_transposed(img + voff[cb & 3] + (cb >> 2) * 128);
        o[cb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(vf, ph, o[cb], 0, 0, 0);
        o[cb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(vf, pl, o[cb], 0, 0, 0);
      }
    }
    if (v + 2 <= v_hi) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");        // the tile's last reads are in registers
      if (((v - v_lo) & 31) == 30) copy.refill(v + 2, looked_up, pos, key0);
      copy_tile(v + 2, img);
    }
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  float* lds = reinterpret_cast<float*>(sm.bytes);
  auto put = [&](float* to) {
    if (n >= h_count) return;
    float* pr = to + n * Smem::kRowF;
    if (g4 == 0) pr[C] = m, pr[C + 1] = l;
#pragma unroll
    for (int cb = 0; cb < C / 16; ++cb) *reinterpret_cast<f32x4v*>(pr + 16 * cb + 4 * g4) = o[cb];
  };
  auto take = [&](const float* rows) {
    if (n >= h_count) return;
    const float* pr = rows + n * Smem::kRowF;
    const float mp = pr[C], lp = pr[C + 1], mm = fmaxf(m, mp);
    const float f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mm);       // (a wave that saw no key)
    const float fp = mp == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mp - mm);
#pragma unroll
    for (int cb = 0; cb < C / 16; ++cb) o[cb] = o[cb] * f + *reinterpret_cast<const f32x4v*>(pr + 16 * cb + 4 * g4) * fp;
    l = l * f + lp * fp;
    m = mm;
  };
  __syncthreads();                                    // every wave is done with its ring
  if (wave >= 2) put(lds + (wave - 2) * kLatentHeads * Smem::kRowF);
  __syncthreads();
  if (wave < 2) take(lds + wave * kLatentHeads * Smem::kRowF);
  __syncthreads();
  if (wave == 1) put(lds);
  __syncthreads();
  if (wave == 0) {
    take(lds);
    put(static_cast<float*>(a.workspace) + (((static_cast<size_t>(s) * a.num_kv_heads + g) * splits + split) * group + h_first) * Smem::kRowF);
  }
}

}  // namespace
}  // namespace hymeta
