// Varlen prefill attention: causal sliding window over the real keys plus an
// always-visible block of meta keys, one softmax (flash-attention forward).
//
// A workgroup owns 128 (query, head) rows of one (sequence, kv-head): the
// query heads of a kv-head lie side by side, so that they share every key and
// a chunk of a few queries still fills its waves.  Each wave owns 32 rows; the
// keys are walked in tiles of 64, copied straight into LDS images (256-byte
// rows, 16-byte chunks permuted within the row).  Two workgroups run on a
// compute unit, in steps of their own.
//
// A wave's step is a software pipeline over three tiles: the products of the
// scores of tile t + 1 (S^T = K Q^T) and of the output of tile t - 1 (O^T +=
// V^T P^T), with the exponentials of tile t and the maximum of tile t + 1
// placed between them, so that the matrix pipe runs under the wave's own vector
// work.  S^T leaves row n's scores of 32 of the 64 keys on lane n and the
// others on lane n + 32; packed to bf16 they are the second product's operand
// as they lie, the values being read transposed (ds_read_b64_tr_b16) in the
// same order of keys.
//
// Bound by the matrix pipe and its clock: with nothing but the products left in
// the loop, one prompt of 8192 x 28 heads (4 kv-heads, window 4097) takes 263 us,
// with everything 359 (1.0 PFLOP/s); copies cost 6 %, barriers and the look at
// the reference 3 % each.  Against a workgroup per head with operands through
// registers, one tile at a time: 647 -> 359 us here, a chunk of 2048 at 32k of
// 7 heads on one kv-head 365 -> 238, one prompt of 32768 (window 4097) 1968 ->
// 1709, eight of 4096 1739 -> 962, four chunks of 5 tokens behind 7922 65 -> 26.
// Eight waves to a workgroup, which read the keys half as often: level at
// prompts of 8192 and more, 3 to 20 % slower below and with few heads.  The
// step's scalar work counts as much as its vector work (twice as many scalar
// instructions and branches per tile: 415 us): what a tile needs is worked out
// in front of the loop.
// Keys are read through a block table (chunked / prefix prefill) or from the
// packed [token, kv-head, dim] tensor of the step.
#include "lds_copy.h"

namespace hymeta {
namespace {

constexpr int kTile = 32;            // granularity required of the meta-key count
constexpr int kTileK = 64;           // keys per step
constexpr int kRowsPerWave = 32;
constexpr int kWaves = 4, kRows = kRowsPerWave * kWaves;
constexpr int kCopies = 16 / kWaves;  // copies of 4 rows a wave makes per image
constexpr int kPitch = 2 * kHeadDim;
constexpr int kImage = kTileK * kPitch;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLazyLog2 = 8.f;     // the softmax reference may trail the true row maximum by a factor 2^8

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

__device__ __forceinline__ f32x16 mfma32(const u32x4& a, const u32x4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// max of three as ONE instruction: v_maximum3_f32 (NaN-propagating, so the compiler adds no
// canonicalising v_max per MFMA output as it does for fmaxf, and no wait states as after inline asm).
__device__ __forceinline__ float max3(float a, float b, float c) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c);
}

// 4 keys x 16 dims block read column-major: lane i of a 16-lane group gets dim i of the 4 keys.
__device__ __forceinline__ u32x2 tr_read(const char* p) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p)));
}

// Sum of a packed bf16 pair and c, in fp32.
__device__ __forceinline__ float add_pair(uint32_t pair, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), __builtin_bit_cast(bf16x2, 0x3f803f80u), c, false);
}

// 16-byte chunks of a row are permuted so that the rows of one fragment read hit distinct banks: a key read asks for one chunk
// of 16 rows, a transposed value read for four neighbouring chunks of four rows.
__device__ __forceinline__ int key_twist(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }
__device__ __forceinline__ int value_twist(int row) { return (row & 3) << 2; }

// A quotient of wave-uniform values as one: the division runs on the vector unit, and what follows from it would stay there.
__device__ __forceinline__ int quotient(int a, int b) { return __builtin_amdgcn_readfirstlane(a / b); }

}  // namespace

// grid = (blocks of 128 rows x key slices x kv-heads (fastest), num_seqs (+1: the meta-query rows)).
//
// splits > 1 (few workgroups, long key ranges: a short chunk of a long sequence): a workgroup walks
// only its share of the tiles and leaves an un-normalised partial (fp32 O, the reference exponent
// and the row sum per row) in the workspace; a second launch merges the slices in slice order.
template <bool PAGED>
__global__ __launch_bounds__(64 * kWaves, 2) void swa_prefill_kernel(hymeta_swa_prefill_args a, float scale_log2, int splits,
                                                                 int64_t part_rows) {
  __shared__ __attribute__((aligned(16))) char s_k[2][kImage];
  __shared__ __attribute__((aligned(16))) char s_v[2][kImage];

  const int lane = threadIdx.x & 63, n = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int seq = blockIdx.y;
  const int group = quotient(a.num_heads, a.num_kv_heads);
  const int item = quotient(blockIdx.x, a.num_kv_heads), kvh = blockIdx.x - item * a.num_kv_heads;
  const int block = quotient(item, splits), split = item - block * splits;
  const bool meta_rows = seq == a.num_seqs;  // this workgroup computes the meta-query rows
  const int M = a.meta_key != nullptr ? a.num_meta : 0;
  const int meta_tiles = (M + kTileK - 1) / kTileK;
  const int out_row0 = a.meta_query != nullptr ? a.num_meta : 0;

  int Lq, Lk;                 // query count, key count
  const uint16_t* qbase;
  int64_t q_stride_t, q_stride_h;
  int64_t out_first;          // output row of the sequence's first query
  int64_t k_first = 0;        // un-paged: first key row of the sequence
  if (meta_rows) {
    Lq = a.num_meta;
    Lk = 0;
    qbase = static_cast<const uint16_t*>(a.meta_query);
    q_stride_t = a.meta_q_stride_t, q_stride_h = a.meta_q_stride_h;
    out_first = 0;
  } else {
    const int q_first = a.cu_seqlens_q[seq];
    Lq = a.cu_seqlens_q[seq + 1] - q_first;
    if constexpr (PAGED) {
      Lk = a.seq_lens_k[seq];
    } else {
      k_first = a.cu_seqlens_k[seq];
      Lk = a.cu_seqlens_k[seq + 1] - static_cast<int>(k_first);
    }
    qbase = static_cast<const uint16_t*>(a.q) + static_cast<int64_t>(q_first) * a.q_stride_t;
    q_stride_t = a.q_stride_t, q_stride_h = a.q_stride_h;
    out_first = out_row0 + q_first;
  }
  const int rows = Lq * group;
  const int r0 = ((rows + kRows - 1) / kRows - 1 - block) * kRows;   // the blocks with the most keys first
  if (r0 < 0) return;                        // workgroup-uniform
  const int w0 = r0 + wave * kRowsPerWave;   // first row of this wave
  const bool active = w0 < rows;             // idle waves still copy tiles and meet the barriers
  const int pos_shift = Lk - Lq;             // query i sits at key position i + pos_shift (bottom-right aligned)

  // this lane's row
  const int r = w0 + n;
  const bool ok = r < rows;
  const int qi = ok ? r / group : 0, h = kvh * group + (ok ? r - qi * group : 0);
  u32x4 qf[8];
  {
    const uint16_t* qrow = qbase + static_cast<int64_t>(qi) * q_stride_t + static_cast<int64_t>(h) * q_stride_h + 8 * hh;
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      qf[st] = u32x4{0u, 0u, 0u, 0u};
      if (ok) qf[st] = ld16g(qrow + 16 * st);
    }
  }

  // Tile ranges: of the workgroup's rows and (real keys) of this wave's.
  const int p_lo = quotient(min(w0, rows - 1), group) + pos_shift, p_hi = quotient(min(w0 + kRowsPerWave - 1, rows - 1), group) + pos_shift;
  int tw_lo = 0, tw_hi = -1, T_lo = 0, T_hi = -1;
  if (!meta_rows && Lk > 0) {
    auto tiles_of = [&](int first, int last, int& lo, int& hi) __attribute__((always_inline)) {
      if (last < 0) return;
      lo = (a.window_left >= 0 && first - a.window_left > 0 ? first - a.window_left : 0) / kTileK;
      hi = min(last, Lk - 1) / kTileK;
    };
    if (active) tiles_of(p_lo, p_hi, tw_lo, tw_hi);
    tiles_of(quotient(r0, group) + pos_shift, quotient(min(r0 + kRows - 1, rows - 1), group) + pos_shift, T_lo, T_hi);
  }
  const int all_tiles = meta_tiles + (T_hi - T_lo + 1);
  // this workgroup's share of the tile sequence (all of it when there is one slice)
  const int per_split = quotient(all_tiles + splits - 1, splits);
  const int t_begin = min(split * per_split, all_tiles);
  const int t_end = min(t_begin + per_split, all_tiles);
  // Tile t holds the real keys from 64 (t + t_real) on, if t >= meta_tiles.
  const int t_real = T_lo - meta_tiles;
  // first and last tile that this wave's rows see (with meta keys: from the first on)
  const int seen_lo = active ? (meta_tiles > 0 ? 0 : tw_lo - t_real) : all_tiles + 1, seen_hi = active && tw_hi >= 0 ? tw_hi - t_real : meta_tiles - 1;
  // real tiles that every row of the wave sees whole: [clear_lo, clear_hi)
  const int clear_lo = max(meta_tiles, (a.window_left >= 0 ? max(p_hi - a.window_left + kTileK - 1, 0) / kTileK : 0) - t_real);
  const int clear_hi = max(min(p_lo + 1, Lk), 0) / kTileK - t_real;

  // ---- copies: an instruction takes four rows of an image, lane = row lane / 16, chunk lane % 16 as it lies in LDS; the
  // wave's i-th the rows 4 (wave + 4 i) ..
  const int32_t* bt = PAGED ? a.block_tables + static_cast<int64_t>(seq) * a.block_table_stride : nullptr;
  const int64_t k_row = 2 * (PAGED ? a.cache_stride_pos : a.k_stride_t), v_row = 2 * (PAGED ? a.cache_stride_pos : a.v_stride_t);
  const char* kglob;
  const char* vglob;
  if constexpr (PAGED) {
    kglob = static_cast<const char*>(a.key_cache) + 2 * kvh * a.cache_stride_h;
    vglob = static_cast<const char*>(a.value_cache) + 2 * kvh * a.cache_stride_h;
  } else {
    kglob = static_cast<const char*>(a.key) + 2 * kvh * a.k_stride_h + k_first * k_row;
    vglob = static_cast<const char*>(a.value) + 2 * kvh * a.v_stride_h + k_first * v_row;
  }
  auto chunk_of = [&](int ln, bool value) __attribute__((always_inline)) -> uint32_t {      // (16 rows on: the same)
    return 16 * ((ln & 15) ^ (value ? value_twist(ln >> 4) : key_twist(4 * wave + (ln >> 4))));
  };
  const uint32_t kplace = (lane >> 4) * static_cast<uint32_t>(k_row) + chunk_of(lane, false);
  const uint32_t vplace = (lane >> 4) * static_cast<uint32_t>(v_row) + chunk_of(lane, true);
  const char* kwave = kglob + 4 * wave * k_row;
  const char* vwave = vglob + 4 * wave * v_row;
  // Tiles [whole_lo, whole_hi) are 64 rows at one stride (whole tiles within a page, four rows within 32 bits): a base per tile
  // and an offset per lane.  Every other one's rows are found one by one.
  const bool regular = (PAGED ? a.block_size % kTileK == 0 : true) && max(k_row, v_row) < (1 << 27);
  const int whole_lo = meta_tiles, whole_hi = regular ? Lk / kTileK - t_real : 0;
  // Paged: lane = tile % 64 holds where a tile's first row lies, for 64 tiles from the last refill on.
  int64_t tile_at = 0;
  auto refill = [&](int t) __attribute__((always_inline)) {
    if (!PAGED) return;
    const int tile = t + ((lane - t) & 63);
    if (tile < whole_lo || tile >= min(whole_hi, t_end)) return;
    const int j = (tile + t_real) * kTileK, at = j / a.block_size;
    tile_at = 2 * (bt[at] * a.cache_stride_block + (j - at * a.block_size) * a.cache_stride_pos);
  };
  auto place_of = [&](int t, int64_t row_bytes) __attribute__((always_inline)) -> int64_t {
    if (!PAGED) return static_cast<int64_t>(t + t_real) * kTileK * row_bytes;
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(tile_at), t & 63);
    const int hi = __builtin_amdgcn_readlane(static_cast<int>(tile_at >> 32), t & 63);
    return (static_cast<int64_t>(hi) << 32) | lo;
  };
  auto copy_tile = [&](int t, bool value, char* image) __attribute__((always_inline)) {
    if (t >= whole_lo && t < whole_hi) {
      const int64_t row_bytes = value ? v_row : k_row;
      const char* base = (value ? vwave : kwave) + place_of(t, row_bytes);
#pragma unroll
      for (int i = 0; i < kCopies; ++i) {
        copy16_to_lds(base, value ? vplace : kplace, image + 1024 * (wave + kWaves * i));
        base += 4 * kWaves * row_bytes;
      }
      return;
    }
    // rows past the last repeat it (their weights are zero)
    int ln = lane;
    asm volatile("" : "+v"(ln));               // (nothing of this is kept in registers over the other tiles)
    for (int i = 0; i < kCopies; ++i) {
      const int row = 4 * (wave + kWaves * i) + (ln >> 4);
      const char* from;
      if (t < meta_tiles) {
        from = static_cast<const char*>(value ? a.meta_value : a.meta_key) + 2 * (min(t * kTileK + row, M - 1) * a.meta_stride_t + kvh * a.meta_stride_h);
      } else {
        const int j = min((t + t_real) * kTileK + row, Lk - 1);
        from = value ? vglob : kglob;
        if (PAGED) {
          const int at = j / a.block_size;
          from += 2 * (bt[at] * a.cache_stride_block + (j - at * a.block_size) * a.cache_stride_pos);
        } else {
          from += j * (value ? v_row : k_row);
        }
      }
      copy16_to_lds(from + chunk_of(ln, value), image + 1024 * (wave + kWaves * i));
    }
  };

  // ---- LDS offsets of this lane's fragments
  int koff[8], voff[4];
#pragma unroll
  for (int st = 0; st < 8; ++st) koff[st] = n * kPitch + 16 * ((2 * st + hh) ^ key_twist(n));
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    const int R = 4 * hh + ((lane & 15) >> 2), chunk = 4 * cb + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    voff[cb] = R * kPitch + 16 * (chunk ^ value_twist(R)) + 8 * (lane & 1);
  }

  f32x16 o[4];                               // O^T: columns 32 cb + 8 i + 4 hh + e of the lane's row, i, e < 4
#pragma unroll
  for (int cb = 0; cb < 4; ++cb)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[cb][i] = 0.f;
  float ref = 0.f, l = 0.f;                  // reference of the exponentials (base 2, a lazy running maximum), sum of the weights
  bool unset = true;                         // the row has not seen a key
  float late = 1.f;                          // what `o` is to be multiplied with behind the weights that are not in it yet
  f32x16 sa[2], sb[2];                       // scores: keys 32 x + 8 i + 4 hh + e of a tile, element 4 i + e of [x]
  u32x4 pa[4], pb[4];                        // weights: keys 8 i + 4 hh + e and 32 further, e < 4, of [i]

  // fragment f of a step: f < 16 of the keys (step f / 2 of the head, half f % 2 of the tile), else of the values (16 keys
  // (f - 16) / 4, columns 32 (f % 4) ..)
  auto fragment = [&](const char* kimg, const char* vimg, int f) __attribute__((always_inline)) {
    if (f < 16) return ld16(kimg + koff[f >> 1] + (f & 1) * 32 * kPitch);
    const char* v = vimg + voff[f & 3] + ((f - 16) >> 2) * 8 * kPitch;
    const u32x2 lo = tr_read(v), hi = tr_read(v + 32 * kPitch);
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  };
  // After the scores of tile t: mask them, move the reference where they ask for it, then of all the wave's rows to their
  // maxima so far, whose weights are 1 and not rounded.  The weights that are not in `o` yet follow the reference before: what
  // the move asks of `o` is done a step later, behind them (`late`).  (Steps of whole powers of two, which scale those weights as
  // well, round the greatest weight like the others: over 2048 keys an error of 0.00217 where it is 0.00207, and 1 and 3/4 beside each
  // other give a difference 8 times as far off.)
  auto settle = [&](int t, f32x16 (&s)[2], float mx) __attribute__((always_inline)) {
    if (t < clear_lo || t >= clear_hi) {
      const bool is_meta = t < meta_tiles;
      const int pos0 = (is_meta ? t : t + t_real) * kTileK;
      // visible key positions of this lane's query: [lo, hi], as one unsigned range test
      const int qp = qi + pos_shift;
      const int lo = is_meta || a.window_left < 0 ? 0 : max(qp - a.window_left, 0), hi = is_meta ? M - 1 : min(qp, Lk - 1);
      const unsigned span = static_cast<unsigned>(hi - lo);
      int ahead = pos0 + 4 * hh - lo;
      asm volatile("" : "+v"(ahead));          // (keeps the compiler from working this out on every tile)
      mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        const bool in = hi >= lo && static_cast<unsigned>(ahead + 32 * (i >> 4) + 8 * ((i & 15) >> 2) + (i & 3)) <= span;
        s[i >> 4][i & 15] = in ? s[i >> 4][i & 15] : -INFINITY;
        mx = __builtin_elementwise_maximum(mx, s[i >> 4][i & 15]);
      }
    }
    const float over = fmaf(mx, scale_log2, -ref);
    if (__any(over > kLazyLog2 || (unset && mx > -INFINITY) || late != 1.f)) {
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) o[cb] *= late;
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float top = fmaf(mx, scale_log2, -ref);
      const bool move = __any(top > kLazyLog2 || (unset && mx > -INFINITY)), up = move && (top > 0.f || (unset && mx > -INFINITY));
      late = up ? (unset ? 0.f : __builtin_amdgcn_exp2f(-top)) : 1.f;
      ref += up ? top : 0.f;
      unset = unset && !up;
      l *= late;
    }
  };
  // One step: scores of tile t + 1 into `next`, weights of tile t (scores `cur`) into `p`, output of tile t - 1 (weights `q`).
  // A slot is one product, the read of a fragment a few products ahead and a slice of the vector work.
  constexpr int kAhead = 4;
  auto step = [&](const char* kimg, const char* vimg, f32x16 (&cur)[2], f32x16 (&next)[2], u32x4 (&p)[4], u32x4 (&q)[4]) __attribute__((always_inline)) -> float {
    u32x4 fr[32];
    float mx = 0.f;
#pragma unroll
    for (int f = 0; f < kAhead; ++f) fr[f] = fragment(kimg, vimg, f);
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int i = 0; i < 16; ++i) next[x][i] = 0.f;
#pragma unroll
    for (int f = 0; f < 32; ++f) {
      if (f + kAhead < 32) fr[f + kAhead] = fragment(kimg, vimg, f + kAhead);
      if (f < 16) next[f & 1] = mfma32(fr[f], qf[f >> 1], next[f & 1]);
      else o[f & 3] = mfma32(fr[f], q[(f - 16) >> 2], o[f & 3]);
      // weights: 16 pairs of scores, ten of them under the first product, six under the second
      const int lo = f < 16 ? f * 10 / 16 : 10 + (f - 16) * 6 / 10, hi = f < 16 ? (f + 1) * 10 / 16 : 10 + (f - 15) * 6 / 10;
#pragma unroll
      for (int j = lo; j < (hi < 16 ? hi : 16); ++j) {
        const int i = j >> 2, e = j & 3;
        const float p0 = __builtin_amdgcn_exp2f(fmaf(cur[e >> 1][4 * i + 2 * (e & 1)], scale_log2, -ref));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(cur[e >> 1][4 * i + 2 * (e & 1) + 1], scale_log2, -ref));
        p[i][e] = pack_bf16x2(p0, p1);
        l = add_pair(p[i][e], l);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (lo <= 4 * i + 3 && 4 * i + 3 < hi) asm volatile("" : "+v"(p[i]), "+v"(l));      // here, not where they are used
      // the next tile's maximum
      if (f == 20) mx = __builtin_elementwise_maximum(next[0][0], next[1][0]);
      if (f > 20) {
#pragma unroll
        for (int j = 1 + (f - 21) * 15 / 11; j < 1 + (f - 20) * 15 / 11; ++j) mx = max3(mx, next[0][j], next[1][j]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("" : "+v"(mx));
    return mx;
  };
  // The same without a tile t - 1 that this wave's rows see.
  auto lead = [&](const char* kimg, f32x16 (&cur)[2], f32x16 (&next)[2], u32x4 (&p)[4]) __attribute__((always_inline)) -> float {
#pragma unroll
    for (int i = 0; i < 32; ++i) next[i >> 4][i & 15] = 0.f;
#pragma unroll
    for (int f = 0; f < 16; ++f) next[f & 1] = mfma32(fragment(kimg, kimg, f), qf[f >> 1], next[f & 1]);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int i = j >> 2, e = j & 3;
      const float p0 = __builtin_amdgcn_exp2f(fmaf(cur[e >> 1][4 * i + 2 * (e & 1)], scale_log2, -ref));
      const float p1 = __builtin_amdgcn_exp2f(fmaf(cur[e >> 1][4 * i + 2 * (e & 1) + 1], scale_log2, -ref));
      p[i][e] = pack_bf16x2(p0, p1);
      l = add_pair(p[i][e], l);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = max3(mx, next[0][i], next[1][i]);
    return mx;
  };
  auto blank = [&](f32x16 (&s)[2], u32x4 (&p)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 32; ++i) s[i >> 4][i & 15] = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = u32x4{0u, 0u, 0u, 0u};
  };

  blank(sa, pa), blank(sb, pb);
  if (t_begin < t_end) {
    refill(t_begin);
    copy_tile(t_begin, false, s_k[0]);
    copies_landed_barrier();
    if (t_begin + 1 < t_end) copy_tile(t_begin + 1, false, s_k[1]);
    settle(t_begin, sa, lead(s_k[0], sb, sa, pa));     // the first tile's scores
    // tile t: keys and values in images (t - t_begin) & 1
    auto arrive = [&](int t, int even) __attribute__((always_inline)) {
      copies_landed_barrier();               // keys of t + 1 and values of t - 1 are there, and nobody reads the images they leave
      if (t + 2 < t_end) copy_tile(t + 2, false, s_k[even]);
      copy_tile(t, true, s_v[even]);
    };
    auto iterate = [&](int t, int even, f32x16 (&cur)[2], f32x16 (&next)[2], u32x4 (&p)[4], u32x4 (&q)[4]) __attribute__((always_inline)) {
      arrive(t, even);
      if (t + 1 < seen_lo || t - 1 > seen_hi) {
        blank(next, p);
        return;
      }
      const float mx = step(s_k[1 - even], s_v[1 - even], cur, next, p, q);
      if (t + 1 < t_end) settle(t + 1, next, mx);
    };
    auto finish = [&](int last, u32x4 (&p)[4]) __attribute__((always_inline)) {
      copies_landed_barrier();
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) o[cb] *= late;
#pragma unroll
      for (int f = 16; f < 32; ++f) o[f & 3] = mfma32(fragment(s_v[last], s_v[last], f), p[(f - 16) >> 2], o[f & 3]);
    };
    arrive(t_begin, 0);
    {
      const float mx = lead(s_k[1], sa, sb, pa);
      if (t_begin + 1 < t_end) settle(t_begin + 1, sb, mx);
    }
    int t = t_begin + 1;
    for (; t + 1 < t_end; t += 2) {
      if (((t - t_begin) & 31) == 31) refill(t);
      iterate(t, 1, sb, sa, pb, pa);
      iterate(t + 1, 0, sa, sb, pa, pb);
    }
    if (t < t_end) {
      iterate(t, 1, sb, sa, pb, pa);
      finish(1, pb);
    } else {
      finish(0, pa);
    }
  }
  l += __shfl_xor(l, 32, 64);
  if (!ok) return;

  if (splits > 1) {
    // partial of this key slice: O un-normalised (fp32), the row's reference exponent and its sum
    const int64_t prow = (split * part_rows + out_first + qi) * a.num_heads + h;
    float* po = static_cast<float*>(a.workspace);
    float* pm = po + static_cast<int64_t>(splits) * part_rows * a.num_heads * kHeadDim;
    float* pl = pm + static_cast<int64_t>(splits) * part_rows * a.num_heads;
    if (hh == 0) pm[prow] = unset ? -INFINITY : ref, pl[prow] = l;
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4*>(po + prow * kHeadDim + 32 * cb + 8 * i + 4 * hh) = f32x4{o[cb][4 * i], o[cb][4 * i + 1], o[cb][4 * i + 2], o[cb][4 * i + 3]};
    return;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  uint16_t* out = static_cast<uint16_t*>(a.out) + (out_first + qi) * a.out_stride_t + static_cast<int64_t>(h) * a.out_stride_h;
#pragma unroll
  for (int cb = 0; cb < 4; ++cb)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<u32x2*>(out + 32 * cb + 8 * i + 4 * hh) =
          u32x2{pack_bf16x2(o[cb][4 * i] * inv, o[cb][4 * i + 1] * inv), pack_bf16x2(o[cb][4 * i + 2] * inv, o[cb][4 * i + 3] * inv)};
}

// One wave per (output row, head): out = sum_s 2^(m_s - m) O_s / sum_s 2^(m_s - m) l_s, slices in order.
__global__ __launch_bounds__(256) void swa_prefill_merge_kernel(hymeta_swa_prefill_args a, int splits, int64_t part_rows) {
  const int lane = threadIdx.x & 63;
  const int64_t pair = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);     // row * H + head
  if (pair >= part_rows * a.num_heads) return;
  const float* po = static_cast<const float*>(a.workspace);
  const float* pm = po + static_cast<int64_t>(splits) * part_rows * a.num_heads * kHeadDim;
  const float* pl = pm + static_cast<int64_t>(splits) * part_rows * a.num_heads;
  float m = -INFINITY;
  for (int s = 0; s < splits; ++s) m = fmaxf(m, pm[s * part_rows * a.num_heads + pair]);
  float o0 = 0.f, o1 = 0.f, l = 0.f;
  for (int s = 0; s < splits; ++s) {
    const float ms = pm[s * part_rows * a.num_heads + pair], ls = pl[s * part_rows * a.num_heads + pair];
    if (ms == -INFINITY && ls == 0.f) continue;           // a slice without a visible key for this query (of nothing but NaN: its sum is one)
    const float w = __builtin_amdgcn_exp2f(ms - m);
    const f32x2 v = *reinterpret_cast<const f32x2*>(po + (s * part_rows * a.num_heads + pair) * kHeadDim + 2 * lane);
    o0 += w * v[0];
    o1 += w * v[1];
    l += w * ls;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const int64_t row = pair / a.num_heads;
  const int head = static_cast<int>(pair % a.num_heads);
  uint32_t* op = reinterpret_cast<uint32_t*>(reinterpret_cast<uint16_t*>(a.out) + row * a.out_stride_t +
                                             static_cast<int64_t>(head) * a.out_stride_h) + lane;
  *op = pack_bf16x2(o0 * inv, o1 * inv);
}

}  // namespace hymeta

using namespace hymeta;

constexpr int kMaxPrefillSplits = 8;

static size_t prefill_partial_bytes(int64_t rows, int heads, int splits) {
  return static_cast<size_t>(splits) * rows * heads * (kHeadDim + 2) * sizeof(float);
}

// Key slices for a call: only where the rows would leave most compute units idle and every slice
// still walks a fair number of tiles (a bound from the window or max_seqlen_k; unknown: 1).  Rows are
// counted in blocks of 128 (256) queries of one head.  The blocks launched are fewer where a kv-head
// has several heads and a sequence few queries, as those lie side by side: 8 queries of 7 heads behind
// 32768 keys are one block in 8 slices (77 us).
extern "C" int hymeta_meta_swa_prefill_splits(int32_t total_q, int32_t num_heads, int32_t num_meta, int32_t meta_rows,
                                              int32_t window_left, int32_t max_seqlen_k) {
  if (total_q <= 0 || num_heads <= 0) return 1;
  const int64_t wgs256 = (static_cast<int64_t>(total_q) + 255) / 256 * num_heads + static_cast<int64_t>(num_heads) * ((meta_rows + 255) / 256);
  if (wgs256 >= 128) return 1;
  const int64_t wgs128 = (static_cast<int64_t>(total_q) + 127) / 128 * num_heads + static_cast<int64_t>(num_heads) * ((meta_rows + 127) / 128);
  int64_t keys = max_seqlen_k > 0 ? max_seqlen_k : -1;
  if (window_left >= 0 && (keys < 0 || window_left + 128 < keys)) keys = window_left + 128;
  if (keys < 0) return 1;
  const int64_t tiles = (keys + kTileK - 1) / kTileK + 1 + (num_meta + kTileK - 1) / kTileK;
  int64_t splits = 512 / (wgs128 > 0 ? wgs128 : 1);          // two workgroups fit a compute unit
  if (splits > tiles / 8) splits = tiles / 8;
  if (splits > kMaxPrefillSplits) splits = kMaxPrefillSplits;
  return splits < 2 ? 1 : static_cast<int>(splits);
}

extern "C" size_t hymeta_meta_swa_prefill_workspace_bytes(int32_t out_rows, int32_t num_heads, int32_t num_splits) {
  if (out_rows <= 0 || num_heads <= 0 || num_splits == 1) return 0;
  return prefill_partial_bytes(out_rows, num_heads, num_splits <= 0 ? kMaxPrefillSplits : num_splits);
}

extern "C" int hymeta_meta_swa_prefill(const hymeta_swa_prefill_args* args, hymeta_stream_t stream) {
  if (!hymeta::args_ok(args)) return HYMETA_ERR_INVALID_ARG;
  hymeta_swa_prefill_args a = *args;
  if (a.num_seqs < 0 || a.total_q < 0 || a.num_heads <= 0 || a.num_kv_heads <= 0) return HYMETA_ERR_INVALID_ARG;
  if (a.head_dim != kHeadDim) return HYMETA_ERR_UNSUPPORTED;
  if (a.num_heads % a.num_kv_heads != 0) return HYMETA_ERR_INVALID_ARG;
  if ((a.meta_key == nullptr) != (a.meta_value == nullptr)) return HYMETA_ERR_INVALID_ARG;
  if (a.meta_key == nullptr) a.num_meta = 0;
  if (a.num_meta < 0 || a.num_meta % kTile != 0) return HYMETA_ERR_UNSUPPORTED;
  if (a.meta_query != nullptr && a.num_meta == 0) return HYMETA_ERR_INVALID_ARG;
  const bool have_rows = a.num_seqs > 0 && a.total_q > 0;
  if (!have_rows && a.meta_query == nullptr) return HYMETA_OK;
  if (!a.out) return HYMETA_ERR_INVALID_ARG;
  const bool paged = a.block_tables != nullptr;
  if (have_rows) {
    if (!a.q || !a.cu_seqlens_q) return HYMETA_ERR_INVALID_ARG;
    if (paged) {
      if (!a.key_cache || !a.value_cache || !a.seq_lens_k || a.block_size <= 0) return HYMETA_ERR_INVALID_ARG;
      if (a.block_size % 16 != 0) return HYMETA_ERR_UNSUPPORTED;
    } else if (!a.key || !a.value || !a.cu_seqlens_k) {
      return HYMETA_ERR_INVALID_ARG;
    }
  }
  const int64_t strides[] = {a.q_stride_t, a.q_stride_h, a.k_stride_t, a.k_stride_h, a.v_stride_t, a.v_stride_h,
                             a.out_stride_t, a.out_stride_h, a.cache_stride_block, a.cache_stride_pos,
                             a.cache_stride_h, a.meta_q_stride_t, a.meta_q_stride_h, a.meta_stride_t, a.meta_stride_h};
  for (int64_t st : strides)
    if (st % 8 != 0) return HYMETA_ERR_UNSUPPORTED;
  const uintptr_t ptrs = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.key) |
                         reinterpret_cast<uintptr_t>(a.value) | reinterpret_cast<uintptr_t>(a.key_cache) |
                         reinterpret_cast<uintptr_t>(a.value_cache) | reinterpret_cast<uintptr_t>(a.meta_query) |
                         reinterpret_cast<uintptr_t>(a.meta_key) | reinterpret_cast<uintptr_t>(a.meta_value) |
                         reinterpret_cast<uintptr_t>(a.out);
  if (ptrs % 16 != 0) return HYMETA_ERR_UNSUPPORTED;

  const float scale = a.scale > 0.f ? a.scale : 1.f / sqrtf(static_cast<float>(a.head_dim));
  int max_rows = have_rows ? a.max_seqlen_q : 0;
  if (have_rows && max_rows <= 0) max_rows = a.total_q;
  if (a.meta_query != nullptr && a.num_meta > max_rows) max_rows = a.num_meta;
  const int seqs = have_rows ? a.num_seqs : 0;
  if (!have_rows) a.num_seqs = 0;
  // key slices: the library's choice needs a workspace that holds it (without one: a single slice)
  const int64_t out_rows = static_cast<int64_t>(have_rows ? a.total_q : 0) + (a.meta_query != nullptr ? a.num_meta : 0);
  int splits = a.num_splits > 0 ? a.num_splits
                                : hymeta_meta_swa_prefill_splits(have_rows ? a.total_q : 0, a.num_heads, a.num_meta,
                                                                 a.meta_query != nullptr ? a.num_meta : 0, a.window_left, a.max_seqlen_k);
  if (splits > kMaxPrefillSplits) return HYMETA_ERR_UNSUPPORTED;
  if (splits > 1 && (a.workspace == nullptr || a.workspace_bytes < prefill_partial_bytes(out_rows, a.num_heads, splits))) {
    if (a.num_splits > 1) return HYMETA_ERR_WORKSPACE;
    splits = 1;
  }
  if (splits > 1 && reinterpret_cast<uintptr_t>(a.workspace) % 16 != 0) return HYMETA_ERR_UNSUPPORTED;
  const int64_t blocks = (static_cast<int64_t>(max_rows) * (a.num_heads / a.num_kv_heads) + kRows - 1) / kRows;
  dim3 grid(static_cast<unsigned>(blocks * splits * a.num_kv_heads), seqs + (a.meta_query != nullptr ? 1 : 0));
  hipStream_t s = begin_launches(stream);
  const float sl2 = scale * kLog2e;
  if (paged) hipLaunchKernelGGL((swa_prefill_kernel<true>), grid, dim3(64 * kWaves), 0, s, a, sl2, splits, out_rows);
  else hipLaunchKernelGGL((swa_prefill_kernel<false>), grid, dim3(64 * kWaves), 0, s, a, sl2, splits, out_rows);
  if (splits > 1) {
    if (hipGetLastError() != hipSuccess) return HYMETA_ERR_LAUNCH;
    const int64_t pairs = out_rows * a.num_heads;
    hipLaunchKernelGGL(swa_prefill_merge_kernel, dim3(static_cast<unsigned>((pairs + 3) / 4)), dim3(256), 0, s, a, splits, out_rows);
  }
  return launch_status();
}
