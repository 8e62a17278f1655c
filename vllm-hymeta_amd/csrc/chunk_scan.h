// Linear attention with decays over the bf16 rows of prompts' portions, in chunks of 64 rows on the matrix cores: the
// kernel behind lightning attention and the decay scan.  With S the state before a chunk, i and j rows of the chunk, n its
// number of rows, l_j the log2 decays, c_i = l_0 + ... + l_i their running sums and b_j the input weights:
//   o_i   = 2^(c_i) S^T q_i + sum_{j <= i} 2^(c_i - c_j) b_j (q_i . k_j) v_j + skip v_i
//   S_new = 2^(c_{n-1}) S + sum_j k_j (2^(c_{n-1} - c_j) b_j v_j)^T
#pragma once

#include "act_types.h"
#include "row_copy.h"

namespace hymeta {
namespace {

struct ChunkScanArgs {
  const uint16_t *q, *k, *v;               // rows of num_qk_heads x D, the same, num_heads x v_dim
  int64_t q_stride, k_stride, v_stride;
  const float *decay, *log2_decay;         // per head, or per row and head
  const float *v_scale, *skip;             // b per row and head, skip per head, or NULL
  float *state, *out, *workspace;          // state fp32 [slots, heads, D, v_dim]
  const int32_t *query_start_loc, *context_lens, *slot_idx;
  int num_seqs, num_heads, num_qk_heads, v_dim;
};

constexpr int kScanRows = 64;              // rows of a chunk
constexpr int kScanMinRows = 8;            // shorter portions go token by token
constexpr float kMinLog2 = -1.0e4f;        // a decay of 0 (or an overflowed step size): finite, so that differences of sums stay numbers

// A workgroup takes as many value columns as there are, 128, 64 or 32 (16 to a wave): what is done once per workgroup, the
// rows' silu and the chunk's weights, is then done once per head.  Where that gives few workgroups, half as wide ones: two
// portions of 150 rows of 28 heads of 128 columns took 23.0 us in 56 workgroups, 21.1 in 112 and 27.6 in 224.  (lanes: the
// workgroups that have rows, per 128 columns or fewer)
inline int scan_waves(int64_t lanes, int v_dim) {
  if (v_dim % 128 == 0 && lanes * (v_dim / 128) > 96) return 8;
  return v_dim % 64 == 0 ? 4 : 2;
}

// A sequence's chunks follow each other in one workgroup per (head, value slice).  Where that leaves most of the chip idle,
// the portions are cut into segments that run side by side: every segment but the last is summarised from a zero state (its
// state and the sum of its log2 decays), the summaries become the states in front of the segments, and every segment runs from
// its state.  The summaries read the keys and values a second time, so fewer than three segments do not
// pay.  What counts is the work there is (long_portions), not the sequences: single rows and short portions leave the chip to
// a long prompt beside them.  8192 rows of 28 heads of 128 columns beside 63 single rows: lightning 194 us (705 with the
// sequences counted), plain decays 159 (565); 6000 rows beside six portions of 700: 218 (495) and 157 (392).
// As many segments as run at the same time, eight waves to a compute unit: one prompt of 8192 rows of 28 heads of 128
// columns took 138 us (lightning, the keys in one part) and 120 (plain decays) in 256 workgroups of eight waves, 152 and 136 in 512, 175 and 156
// in 1024; of 64 columns 131 us in 512 workgroups of four, 189 in 256, 147 in 1024.  At least 64 rows each (192 / 64, us): 28 heads
// of 128 x 128, one portion of 400 rows 37.4 / 26.7, of 1000 42.2 / 35.0; 16 heads of 64 x 128, one of 577 19.3 / 15.3,
// two of 450 with 128 rows of state 42.4 / 26.3.  Not beside many short portions, which fill what one segment leaves idle and wait
// for the summaries otherwise: 28 heads of 128 x 128, one of 300 beside 32 single rows 29.5 / 27.5, beside 63 30.5 / 36.7;
// 32 heads of 64 columns, one of 520 beside 63 37.0 / 25.8.
//
// The segments of the portions of more than `rows` rows are numbered one behind the other (segment_at); there are no more than
// one per `rows` rows of the step and one per such portion.  What has no rows comes behind what has: a workgroup that ends at
// once in front of others leaves its compute unit idle while those share one (16 heads: 90 -> 145 us).
//
// Up to kMostUnchained segments every one works out the state in front of it for itself, from the summaries before it, which saves a
// launch (6 to 9 us) for at most ten reads of 64 KB: 16 heads of 128 columns, five portions of 700 rows in four segments 41 -> 31 us, of
// 64 columns three of 2000 64 -> 57; with 16 segments level.
// More of them take the chain's launch and more states to and fro, which single rows and short portions wait for unless the chip is
// through with a segment at once: in segments of one chunk, or alone (at least 192 rows each otherwise, but for the first ten).  2048
// rows of 16 heads of 128 x 128, plain decays: alone 32.2 us in 16 segments, 36.0 in 8; beside 63 single rows 47.3 and 38.2; 7 heads,
// lightning, beside 63 37.6 in 32 of one chunk, 45.5 in 8.  Where segments of 64 columns take two places on every compute unit: 32 heads alone
// 39.1 in 16, 35.0 in 8; 16 heads, beside 63 37.8 in 32 of one chunk, 32.9 in 8, lightning 41.4 and 44.1, beside 100 45.6 and 43.9.
constexpr int kMostUnchained = 10, kSegmentRows = 64, kManySegmentRows = 192, kManyColumns = 131072, kSomeColumns = 49152;
struct ScanSegments {
  int rows = 0x7fffffff, count = 0;        // rows of a segment; bound on the segments' numbers
  bool chained = false;                    // whether a launch of its own turns the summaries into the states in front of the segments
  int64_t lanes = 0;                       // (segment, head) pairs that run side by side
};
// Columns of a segment's workgroup, and how many of them run at the same time.
inline int scan_columns(int v_dim) { return v_dim % 128 == 0 ? 128 : v_dim % 64 == 0 ? 64 : 32; }
inline int64_t scan_slots(int v_dim) { return 256 * (128 / scan_columns(v_dim)); }
inline int64_t scan_slices(int num_heads, int v_dim) { return num_heads * std::max<int64_t>(v_dim / scan_columns(v_dim), 1); }
// Segments of a step of `portions` long ones: how many of a head's fit on the chip beside the others.
inline int64_t scan_segments_wanted(int64_t portions, int num_heads, int v_dim, int max_query_len) {
  return std::min<int64_t>(scan_slots(v_dim) / (portions * scan_slices(num_heads, v_dim)), max_query_len / kSegmentRows);
}
// Whether segments of a few chunks pay: a portion's chunks one behind the other, against those of a segment twice (summary and rows, which a
// segment's eight staging waves halve), a launch more, and the states' way through memory, which goes with the places that the
// segments take (and the short portions beside them, a sixteenth of one each) and is shorter where all of a head's are on one die
// (heads in eights).  A chunk with silu takes half as long again.  Rounded to chunks there may be two segments left of three: never.
// Us, cut / whole, plain decays: 28 heads of 128 x 128, three portions of 200 rows 23.0 / 18.8 (two segments), one of 256 18.6 / 17.2, two 23.2 / 18.4, three
// of 260 25.4 / 22.7, one 17.4 / 20.2, three of 500 29.8 / 33.2; 16 heads, two of 256 16.4 / 17.5; lightning, 28 heads, one of 256 21.0 /
// 23.7, two 25.3 / 24.7.  Columns in 64s or fewer, two and more workgroups on a compute unit: 56 heads, one of 256 15.5 / 17.4, three of 400 34.3 / 30.4;
// 32 heads, three of 260 19.5 / 21.2; 28 heads of 64 x 64, five of 450 25.3 / 24.1.  192 rows with nothing to stage are level or slower: 12.4 / 10.9.
inline bool scan_segments_pay(int64_t places, int pieces, int num_heads, int v_dim, int max_query_len, int rows, bool silu) {
  const int64_t slots = scan_slots(v_dim), chunks = (max_query_len + kScanRows - 1) / kScanRows, each = rows / kScanRows;
  if (pieces < 3 || (!silu && chunks < 4)) return false;
  if (v_dim % 128 != 0) return 5 * (chunks - 2 * each) * slots > 7 * (3 * places - slots);
  return 2 * (chunks - each) * slots > (silu ? 1 : 3) * slots + (num_heads % 8 == 0 ? 5 : 7) * places;
}
inline ScanSegments scan_segments(int num_tokens, int num_seqs, int num_heads, int v_dim, int max_query_len, bool silu) {
  const int64_t portions = long_portions(num_tokens, num_seqs, max_query_len), columns = static_cast<int64_t>(num_seqs) * num_heads * v_dim;
  const int64_t fit = scan_segments_wanted(portions, num_heads, v_dim, max_query_len);
  const bool many = columns > kManyColumns;
  const int64_t want = many ? std::min<int64_t>(fit, max_query_len / kManySegmentRows) : fit;
  ScanSegments sg;
  sg.lanes = portions * num_heads;
  if (want < 3) return sg;
  auto rows_of = [=](int64_t pieces) { return static_cast<int>((max_query_len + pieces - 1) / pieces + kScanRows - 1) / kScanRows * kScanRows; };
  int rows = rows_of(want);
  auto pieces = [&] { return (max_query_len + rows - 1) / rows; };
  if (!many) {
    const int64_t slots = scan_slots(v_dim), slices = scan_slices(num_heads, v_dim);
    const bool crowded = v_dim % 128 != 0 && 8 * portions * slices * pieces() > 7 * slots;
    const bool beside = columns > (silu ? 2 : 1) * kSomeColumns;
    if (pieces() > kMostUnchained && (rows > kScanRows ? crowded || beside : crowded && beside))
      rows = rows_of(std::max<int64_t>(kMostUnchained, std::min<int64_t>(fit, max_query_len / kManySegmentRows)));
    if (!scan_segments_pay(portions * slices * pieces() + (num_seqs - portions) * slices / 16, pieces(), num_heads, v_dim, max_query_len, rows, silu)) return sg;
  }
  const int64_t cuts = (std::min<int64_t>(num_tokens, static_cast<int64_t>(num_seqs) * max_query_len) - 1) / rows;
  const int64_t count = cuts + std::min<int64_t>(num_seqs, cuts);
  if (num_seqs + count > 65535) return sg;
  sg.rows = rows, sg.count = static_cast<int>(count), sg.lanes *= pieces(), sg.chained = pieces() > kMostUnchained;
  return sg;
}
// The workspace: per segment and head its summary, then the state in front of it; the segments' sums of log2 decays.
inline size_t scan_segment_bytes(int64_t count, int num_heads, int head_dim, int v_dim) {
  return static_cast<size_t>(count) * num_heads * (static_cast<size_t>(head_dim) * v_dim + 1) * sizeof(float);
}
// Enough for any number of tokens, and for fewer sequences and shorter portions too.  With p long portions of m rows at most
// in segments of at least m / w rows there are no more than (p m + num_seqs) w / m cuts: p w is at most what one portion would
// be cut into, w / m at most 1 / 64.
inline size_t scan_workspace_bytes(int num_seqs, int num_heads, int head_dim, int v_dim, int max_query_len) {
  if (num_seqs <= 0 || num_heads <= 0 || head_dim <= 0 || v_dim <= 0 || scan_segments_wanted(1, num_heads, v_dim, max_query_len) < 3) return 0;
  const int64_t cuts = scan_segments_wanted(1, num_heads, v_dim, 0x7fffffff) + num_seqs / kSegmentRows + 1;
  return scan_segment_bytes(cuts + std::min<int64_t>(num_seqs, cuts), num_heads, head_dim, v_dim);
}

// a chunk's rows at byte offsets below 2^31
inline bool scan_offsets_fit(int64_t row_stride, int num_heads, int v_dim) {
  return row_stride >= 0 && row_stride < (1 << 23) && static_cast<int64_t>(num_heads) * v_dim < (1 << 22);
}

typedef float f32x4s __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4s scan_mfma(bf16x8 a, bf16x8 b, f32x4s c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// the hardware's exponential and reciprocal (about 1 ulp each): the input is bf16
__device__ __forceinline__ float silu_fast(float x) { return x * __builtin_amdgcn_rcpf(1.f + __expf(-x)); }

// Two floats as hi + lo bf16 parts (16 bits of mantissa together).
__device__ __forceinline__ void split_pair(float x, float y, uint32_t& hi, uint32_t& lo) {
  hi = pack_bf16x2(x, y);
  lo = pack_bf16x2(x - lo_bf(hi), y - hi_bf(hi));
}
__device__ __forceinline__ bf16x8 frag_of(bf16x4 a, bf16x4 b) { return bf16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]}; }

// Rows behind a wave-uniform address, at byte offsets below 2^31: what a lane has no row for is read as zeros and not
// written, without a branch (around branches the compiler waits for every load AND store in flight).
struct RowBuffer {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ explicit RowBuffer(const void* base) : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0x7fffffff, 0x00020000)) {}
  __device__ __forceinline__ u32x4 load(bool valid, int offset) const {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, valid ? offset : INT32_MIN, 0, 0));
  }
  __device__ __forceinline__ float load1(bool valid, int offset) const {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, valid ? offset : INT32_MIN, 0, 0));
  }
  __device__ __forceinline__ void store(bool valid, int offset, f32x4s x) const {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), r, valid ? offset : INT32_MIN, 0, 0);
  }
};

// Segment `number` of the step (wave-uniform): its sequence (-1: there is no such segment), that one's rows, and which of its
// segments.
__device__ __forceinline__ PieceAt segment_at(const ChunkScanArgs& a, int seg_rows, int number) {
  return piece_at(a.query_start_loc, a.num_seqs, number, [=](int rows) { return rows > seg_rows ? (rows - 1) / seg_rows + 1 : 0; });
}

// 16 columns of a state, by a wave.
template <int D>
__device__ __forceinline__ void copy_columns(const float* from, float* to, int64_t v_dim, int lane) {
  float x[D / 4];
#pragma unroll
  for (int u = 0; u < D / 4; ++u) x[u] = from[(4 * u + lane / 16) * v_dim + lane % 16];
#pragma unroll
  for (int u = 0; u < D / 4; ++u) to[(4 * u + lane / 16) * v_dim + lane % 16] = x[u];
}
// A lane's rows d0 + 16 db + r of a state's column n (NULL: zeros).
template <int DB>
__device__ __forceinline__ void load_state(f32x4s (&S)[DB], const float* from, int d0, int v_dim, int n) {
  const RowBuffer b(from);
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[db][r] = b.load1(from != nullptr, 4 * ((16 * db + d0 + r) * v_dim + n));
}
// The same of the state in front of a segment: the state in front of the portion (in the last segment's place, if there is one), then
// from segment to segment 2^(its sum of log2 decays) of it and the segment's summary.
template <int DB>
__device__ __forceinline__ void segment_state(f32x4s (&S)[DB], const ChunkScanArgs& a, const PieceAt& seg, int seg_rows, int segments, int number, int h,
                                              int64_t per_head, bool carry, int col0, int d0, int v_dim, int n) {
  const int64_t step = a.num_heads * per_head, first = static_cast<int64_t>(number - seg.index) * a.num_heads + h;
  const float *p = a.workspace + first * per_head + col0, *totals = a.workspace + segments * step + first;
  load_state(S, carry ? p + (seg.rows - 1) / seg_rows * step : nullptr, d0, v_dim, n);
  for (int i = 0; i < seg.index; ++i, p += step) {
    f32x4s summary[DB];
    load_state(summary, p, d0, v_dim, n);
    const float decay = __builtin_amdgcn_exp2f(totals[i * a.num_heads]);
#pragma unroll
    for (int db = 0; db < DB; ++db) S[db] = decay * S[db] + summary[db];
  }
}

// A portion too short for a chunk, row by row in fp32 by the 64 NW threads of a workgroup: a thread holds 4 value columns of the
// rows d0, d0 + 16, ... of the state (16-byte loads, all in flight together), the 16 partial outputs of a column meet in LDS.  The
// next row is on its way while one is worked on.  LDS for two rows each: queries and keys, 2 D floats a row, and partial outputs, 256 NW floats a row.
template <int D, int NW, bool Silu>
__device__ __forceinline__ void scan_single_rows(const ChunkScanArgs& a, int h, int s, int r0, int rows, int col0, float* s_row, float* s_part) {
  constexpr int NT = 64 * NW, C4 = 4 * NW, U = D / 16, kEach = (2 * D + NT - 1) / NT;
  const int c4 = threadIdx.x % C4, d0 = threadIdx.x / C4, H = a.num_heads, Dv = a.v_dim, g = h / (H / a.num_qk_heads);
  const int slot = a.slot_idx[s];
  float* st = slot >= 0 ? a.state + (static_cast<int64_t>(slot) * H + h) * D * Dv + col0 : nullptr;
  const uint32_t at = d0 * Dv + 4 * c4;
  const bool carry = st != nullptr && a.context_lens[s] > 0;
  const float constant = a.decay ? a.decay[h] : 1.f, skip = a.skip ? a.skip[h] : 0.f;
  auto act = [](float x) __attribute__((always_inline)) { return Silu ? x / (1.f + expf(-x)) : x; };
  uint16_t qk[kEach];
  u32x2 vraw;
  float decay, b;
  auto fetch = [&](int64_t t) __attribute__((always_inline)) {
    const uint16_t *q = a.q + t * a.q_stride + static_cast<int64_t>(g) * D, *k = a.k + t * a.k_stride + static_cast<int64_t>(g) * D;
#pragma unroll
    for (int j = 0; j < kEach; ++j) {
      const int d = threadIdx.x + NT * j;
      if (d < 2 * D) qk[j] = d < D ? q[d] : k[d - D];
    }
    vraw = *reinterpret_cast<const u32x2*>(a.v + t * a.v_stride + static_cast<int64_t>(h) * Dv + col0 + 4 * c4);
    decay = a.log2_decay ? __builtin_amdgcn_exp2f(a.log2_decay[t * H + h]) : constant;
    b = a.v_scale ? a.v_scale[t * H + h] : 1.f;
  };
  f32x4s S[U];
#pragma unroll
  for (int u = 0; u < U; ++u) S[u] = carry ? *reinterpret_cast<const f32x4s*>(st + static_cast<int64_t>(16 * u) * Dv + at) : f32x4s{0.f, 0.f, 0.f, 0.f};
  fetch(r0);
  for (int i = 0; i < rows; ++i) {
    float *row = s_row + (i & 1) * 2 * D, *part = s_part + (i & 1) * 256 * NW;
#pragma unroll
    for (int j = 0; j < kEach; ++j) {
      const int d = threadIdx.x + NT * j;
      if (d < 2 * D) row[d] = act(bf2f(qk[j]));
    }
    float v[4] = {act(lo_bf(vraw[0])), act(hi_bf(vraw[0])), act(lo_bf(vraw[1])), act(hi_bf(vraw[1]))};
    const float row_decay = decay, row_b = b;
    __syncthreads();
    if (i + 1 < rows) fetch(r0 + i + 1);
    f32x4s acc = f32x4s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = d0 == 0 ? skip * v[e] : 0.f, v[e] *= row_b;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float qd = row[d0 + 16 * u], kd = row[D + d0 + 16 * u];
#pragma unroll
      for (int e = 0; e < 4; ++e) S[u][e] = fmaf(row_decay, S[u][e], kd * v[e]), acc[e] = fmaf(S[u][e], qd, acc[e]);
    }
    *reinterpret_cast<f32x4s*>(part + d0 * 16 * NW + 4 * c4) = acc;
    __syncthreads();
    for (int c = threadIdx.x; c < 16 * NW; c += NT) {
      float o = 0.f;
#pragma unroll
      for (int d = 0; d < 16; ++d) o += part[d * 16 * NW + c];
      a.out[(static_cast<int64_t>(r0 + i) * H + h) * Dv + col0 + c] = o;
    }
  }
  if (st != nullptr) {
#pragma unroll
    for (int u = 0; u < U; ++u) *reinterpret_cast<f32x4s*>(st + static_cast<int64_t>(16 * u) * Dv + at) = S[u];
  }
}

// Portions of 1 to max_rows rows in a launch of their own.  grid = (heads, value columns in slices of 16 NW, sequences).
template <int D, int NW, bool Silu>
__global__ __launch_bounds__(64 * NW) void scan_short_kernel(ChunkScanArgs a, int max_rows) {
  __shared__ __attribute__((aligned(16))) float s_row[2 * 2 * D], s_part[2 * 256 * NW];
  const int s = blockIdx.z, r0 = a.query_start_loc[s], rows = a.query_start_loc[s + 1] - r0;
  if (rows <= 0 || rows > max_rows) return;
  scan_single_rows<D, NW, Silu>(a, blockIdx.x, s, r0, rows, blockIdx.y * 16 * NW, s_row, s_part);
}

// grid = (heads, value columns in slices of 16 NW, segments + sequences (Summarise: segments)); NW waves.  A workgroup takes a
// segment of a portion that has several, or a portion that has one.
//
// Every wave owns 16 value columns of the state, fp32 in registers as the matrix instructions leave it (a lane holds runs of
// four d of one column): that is also the layout in which the next chunk's product with the queries wants it, so the state
// never goes through LDS.  The rows of a chunk go through their silu once per workgroup and lie in LDS as rows; what a product
// needs transposed is read transposed.  The decays of the state's update go onto the values (a wave splits its own 16 columns
// into hi + lo bf16 parts) and not onto the keys; the chunk's own weights are computed once per workgroup, a block of 16 rows
// x 32 keys per wave, and handed over in LDS as fragments.  What enters a product from fp32 goes in as hi + lo parts, two
// products, so that it keeps 16 bits of mantissa; so do the keys behind their silu in the state's update (three products: the
// values, rounded to bf16 as in the outputs, carry the decays).
// Bound by vector arithmetic between the barriers of a chunk: silu, splits, scales.  One prompt of 8192 rows of 28 heads with 64 value
// columns and decays per row 316 -> 131 us; before, 4 waves to 32 value columns, each such workgroup with its own staging, weights
// and an image of the state in LDS.  (Eight waves: heads of 32 only; the others by chunk_scan_piped_kernel.)
template <int D, int NW, bool Silu, bool Summarise, bool Chained>
__global__ __launch_bounds__(64 * NW, Summarise ? 4 : 2) void chunk_scan_kernel(ChunkScanArgs a, int seg_rows, int segments, bool short_too) {
  constexpr int NT = 64 * NW, KC = D / 8, VC = 2 * NW, KP = 2 * D, VP = 32 * NW, SD = D / 32, DB = D / 16;
  constexpr int KPT = (kScanRows * KC + NT - 1) / NT, VPT = 2;
  typedef ChunkOrder<KC> KOrder;
  typedef ChunkOrder<VC> VOrder;
  __shared__ __attribute__((aligned(16))) char s_k[kScanRows * KP], s_v[kScanRows * VP];
  __shared__ __attribute__((aligned(16))) char s_q[Summarise ? 16 : kScanRows * KP], s_klo[Silu ? kScanRows * KP : 16];
  __shared__ __attribute__((aligned(16))) u32x4 s_p[Summarise ? 1 : 6][2][64];
  __shared__ __attribute__((aligned(16))) float s_cum[kScanRows], s_b[kScanRows], s_w[kScanRows];
  const int h = blockIdx.x, vs = blockIdx.y, number = blockIdx.z;
  const bool whole = number >= segments;
  PieceAt seg;
  if (!whole) {
    seg = segment_at(a, seg_rows, number);
    if (seg.seq < 0) return;
  } else {
    seg.seq = number - segments, seg.index = 0;
    seg.row0 = a.query_start_loc[seg.seq], seg.rows = a.query_start_loc[seg.seq + 1] - seg.row0;
  }
  const int s = seg.seq, r0 = seg.row0, rows_all = seg.rows;
  if (rows_all <= 0) return;                           // (a sequence without rows: its slot may be anything)
  if constexpr (!Summarise) {
    static_assert(sizeof(s_k) >= 16 * D && sizeof(s_v) >= 2048 * NW, "the scratch of single rows");
    if (rows_all < kScanMinRows) {                     // (a segment has more)
      if (short_too) scan_single_rows<D, NW, Silu>(a, h, s, r0, rows_all, vs * 16 * NW, reinterpret_cast<float*>(s_k), reinterpret_cast<float*>(s_v));
      return;
    }
  }
  if (rows_all < kScanMinRows || (whole && rows_all > seg_rows)) return;
  const int r_lo = whole ? 0 : seg.index * seg_rows, rows = r_lo + min(rows_all - r_lo, seg_rows);        // (end of this workgroup's rows)
  const bool last = rows == rows_all;
  const bool copies = Summarise && last;               // nothing comes behind the last segment: its place holds the state in front of the portion
  if (copies && Chained) return;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = a.num_heads, Dv = a.v_dim, g = h / (H / a.num_qk_heads), col0 = vs * 16 * NW + 16 * wave;
  const int slot = a.slot_idx[s];
  float* st = slot >= 0 ? a.state + (static_cast<int64_t>(slot) * H + h) * D * Dv + col0 : nullptr;
  const float l2_const = a.decay ? fmaxf(a.decay[h] > 0.f ? log2f(a.decay[h]) : -INFINITY, kMinLog2) : 0.f;
  const float skip = a.skip ? a.skip[h] : 0.f;
  // a segment's place in the workspace: its summary (Summarise writes it), then the state in front of it; the segments' sums
  // of log2 decays lie behind all the states
  const int64_t place = static_cast<int64_t>(number) * H + h;
  float* wsp = whole ? nullptr : a.workspace + place * D * Dv + col0;
  const bool carry = st != nullptr && a.context_lens[s] > 0;
  const float* init = Summarise ? nullptr : whole ? (carry ? st : nullptr) : wsp;
  if (copies) {
    if (carry && threadIdx.x < NT) copy_columns<D>(st, wsp, Dv, lane);
    return;
  }
  float seg_total = 0.f;

  const uint16_t* qp = a.q + static_cast<int64_t>(g) * D;
  const uint16_t* kp = a.k + static_cast<int64_t>(g) * D;
  const uint16_t* vp = a.v + static_cast<int64_t>(h) * Dv + vs * 16 * NW;
  // a chunk's rows as they come from memory, a chunk ahead: this thread's 16-byte chunks of the keys, queries and values, and
  // (first wave) row `lane`'s log2 decay and input weight
  u32x4 rk[KPT], rq[Summarise ? 1 : KPT], rv[VPT];
  float rl = 0.f, rb = 0.f;
  auto fetch = [&](int c0) {
    const int nrow = min(kScanRows, rows - c0);
    const int64_t t0 = r0 + c0;
    const RowBuffer kr(kp + t0 * a.k_stride), qr(qp + t0 * a.q_stride), vr(vp + t0 * a.v_stride);
#pragma unroll
    for (int u = 0; u < KPT; ++u) {
      const int idx = tid + NT * u, j = idx / KC, ch = idx % KC;
      rk[u] = kr.load(j < nrow, 2 * (j * static_cast<int>(a.k_stride) + 8 * ch));
      if constexpr (!Summarise) rq[u] = qr.load(j < nrow, 2 * (j * static_cast<int>(a.q_stride) + 8 * ch));
    }
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
      const int idx = tid + NT * u, j = idx / VC, ch = idx % VC;
      rv[u] = vr.load(j < nrow, 2 * (j * static_cast<int>(a.v_stride) + 8 * ch));
    }
    const int at = 4 * lane * H;
    if (a.log2_decay || a.v_scale) {
      rl = RowBuffer(a.log2_decay + t0 * H + h).load1(a.log2_decay && lane < nrow, at);
      rb = RowBuffer(a.v_scale + t0 * H + h).load1(a.v_scale && lane < nrow, at);
    }
  };
  auto silu8 = [](u32x4 raw, u32x4& hi, u32x4& lo) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t x, y;
      split_pair(silu_fast(lo_bf(raw[e])), silu_fast(hi_bf(raw[e])), x, y);
      hi[e] = x, lo[e] = y;
    }
  };
  // (rows past the portion were fetched as zeros, and silu(0) = 0: a whole chunk has no look at its rows)
  auto stage_as = [&](int nrow, auto full) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < KPT; ++u) {
      const int idx = tid + NT * u, j = idx / KC, ch = idx % KC;
      if (kScanRows * KC % NT != 0 && j >= kScanRows) break;
      const int at = j * KP + 16 * (ch ^ KOrder::twist(j));
      u32x4 x = rk[u], lo;
      if constexpr (Silu) {
        lo = u32x4{0u, 0u, 0u, 0u};
        if (decltype(full)::value || j < nrow) silu8(rk[u], x, lo);
        st16(s_klo + at, lo);
      }
      st16(s_k + at, x);
      if constexpr (!Summarise) {
        x = rq[u];
        if (Silu && (decltype(full)::value || j < nrow)) silu8(rq[u], x, lo);
        st16(s_q + at, x);
      }
    }
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
      const int idx = tid + NT * u, j = idx / VC, ch = idx % VC, at = j * VP + 16 * (ch ^ VOrder::twist(j));
      u32x4 x = rv[u], lo;
      if (Silu && (decltype(full)::value || j < nrow)) silu8(rv[u], x, lo);
      st16(s_v + at, x);
    }
    if (wave == 0) {
      // running sums of the chunk's log2 decays (rows past the portion add 0)
      float cum;
      if (a.log2_decay) {
        cum = lane_sums(fmaxf(rl, kMinLog2));          // (rows past the portion: 0)
      } else {
        cum = static_cast<float>(min(lane + 1, nrow)) * l2_const;
      }
      const float total = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cum), 63));
      s_cum[lane] = cum;
      const float b = a.v_scale ? rb : 1.f;
      s_b[lane] = b;
      const float left = Silu ? static_cast<float>(nrow - 1 - lane) * l2_const : total - cum;
      s_w[lane] = lane < nrow ? __builtin_amdgcn_exp2f(left) * b : 0.f;
    }
  };
  auto stage = [&](int nrow) __attribute__((always_inline)) {
    if (Silu && nrow < kScanRows) stage_as(nrow, std::false_type{});
    else stage_as(nrow, std::true_type{});
  };
  // LDS offsets of this lane's fragments: rows n (16 bytes of a row, or two times 8 for the product with the state), and the
  // transposed reads of 4 keys x 16 columns
  const int kt = KOrder::twist(n), Rt = 4 * g4 + (n >> 2), kT = KOrder::twist(Rt), vT = VOrder::twist(Rt);
  auto row_frag = [&](const char* img, int block, int sd) { return __builtin_bit_cast(bf16x8, ld16(img + (16 * block + n) * KP + 16 * ((4 * sd + g4) ^ kt))); };
  auto row_frag_halves = [&](const char* img, int block, int sd) {
    const char* row = img + (16 * block + n) * KP + 8 * (g4 & 1);
    const u32x2 x = *reinterpret_cast<const u32x2*>(row + 16 * ((4 * sd + (g4 >> 1)) ^ kt));
    const u32x2 y = *reinterpret_cast<const u32x2*>(row + 16 * ((4 * sd + 2 + (g4 >> 1)) ^ kt));
    return __builtin_bit_cast(bf16x8, (u32x4{x[0], x[1], y[0], y[1]}));
  };
  // keys 32 kk + 4 g4 + e for e < 4, 32 kk + 16 + 4 g4 + e - 4 after, of column 16 db + n / of this wave's value column n
  auto key_frag = [&](const char* img, int db, int kk) {
    const char* p = img + (32 * kk + Rt) * KP + 16 * ((2 * db + ((n & 3) >> 1)) ^ kT) + 8 * (n & 1);
    return frag_of(read_transposed(p), read_transposed(p + 16 * KP));
  };
  auto value_frag = [&](const char* img, int kk) {
    const char* p = img + (32 * kk + Rt) * VP + 16 * ((2 * wave + ((n & 3) >> 1)) ^ vT) + 8 * (n & 1);
    return frag_of(read_transposed(p), read_transposed(p + 16 * VP));
  };

  fetch(r_lo);
  f32x4s S[DB];                                        // S[16 db + 4 g4 + r][col0 + n]
  if (Summarise || Chained || whole) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[db][r] = init ? init[static_cast<int64_t>(16 * db + 4 * g4 + r) * Dv + n] : 0.f;
  } else {
    segment_state(S, a, seg, seg_rows, segments, number, h, D * Dv, carry, col0, 4 * g4, Dv, n);
  }
  stage(min(kScanRows, rows - r_lo));
  fetch(r_lo + kScanRows);
  for (int c0 = r_lo; c0 < rows; c0 += kScanRows) {
    const int nrow = min(kScanRows, rows - c0);
    __syncthreads();
    const float total = s_cum[kScanRows - 1];
    seg_total += total;
    bf16x8 vf[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) vf[kk] = value_frag(s_v, kk);
    if constexpr (!Summarise) {
      // weights of the chunk's own rows, as hi + lo fragments: rows 16 ib + n, keys 32 kk ..
      for (int job = wave; job < 8; job += NW) {
        const int ib = job >> 1, kk = job & 1;
        if (2 * kk > ib) continue;
        const int i = 16 * ib + n;
        const float cum_i = s_cum[i];
        u32x4 hi, lo;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int jb = 2 * kk + t;
          f32x4s sc = f32x4s{0.f, 0.f, 0.f, 0.f};
          if (jb <= ib) {
#pragma unroll
            for (int sd = 0; sd < SD; ++sd) sc = scan_mfma(row_frag(s_k, jb, sd), row_frag(s_q, ib, sd), sc);
          }
          f32x4s span, bj;                             // log2 of the decay between row j and row i; j's input weight
          if constexpr (Silu) {
#pragma unroll
            for (int r = 0; r < 4; ++r) span[r] = static_cast<float>(i - 16 * jb - 4 * g4 - r) * l2_const, bj[r] = 1.f;
          } else {
            span = cum_i - *reinterpret_cast<const f32x4s*>(s_cum + 16 * jb + 4 * g4);
            bj = *reinterpret_cast<const f32x4s*>(s_b + 16 * jb + 4 * g4);
          }
          float p[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) p[r] = 16 * jb + 4 * g4 + r <= i ? sc[r] * __builtin_amdgcn_exp2f(span[r]) * bj[r] : 0.f;
          uint32_t x, y;
          split_pair(p[0], p[1], x, y), hi[2 * t] = x, lo[2 * t] = y;
          split_pair(p[2], p[3], x, y), hi[2 * t + 1] = x, lo[2 * t + 1] = y;
        }
        const int at = ib < 2 ? ib : 2 * ib - 2 + kk;
        s_p[at][0][lane] = hi;
        s_p[at][1][lane] = lo;
      }
      // the state before the chunk
      f32x4s o[4];
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) o[ib] = f32x4s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int sd = 0; sd < SD; ++sd) {
        u32x4 sf[2];                                   // its d 32 sd + 4 g4 + e for e < 4, 32 sd + 16 + 4 g4 + e - 4 after, hi and lo
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          uint32_t x, y;
          split_pair(S[2 * sd + (e >> 1)][2 * (e & 1)], S[2 * sd + (e >> 1)][2 * (e & 1) + 1], x, y);
          sf[0][e] = x, sf[1][e] = y;
        }
        bf16x8 qf[4];
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) qf[ib] = row_frag_halves(s_q, ib, sd);
#pragma unroll
        for (int part = 0; part < 2; ++part)
#pragma unroll
          for (int ib = 0; ib < 4; ++ib) o[ib] = scan_mfma(__builtin_bit_cast(bf16x8, sf[part]), qf[ib], o[ib]);
      }
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) o[ib] *= __builtin_amdgcn_exp2f(s_cum[16 * ib + n]);
      if (skip != 0.f) {
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) {
          const u32x2 vi = *reinterpret_cast<const u32x2*>(s_v + (16 * ib + n) * VP + 16 * ((2 * wave + (g4 >> 1)) ^ VOrder::twist(n)) + 8 * (g4 & 1));
          o[ib][0] = fmaf(skip, lo_bf(vi[0]), o[ib][0]), o[ib][1] = fmaf(skip, hi_bf(vi[0]), o[ib][1]);
          o[ib][2] = fmaf(skip, lo_bf(vi[1]), o[ib][2]), o[ib][3] = fmaf(skip, hi_bf(vi[1]), o[ib][3]);
        }
      }
      __syncthreads();
#pragma unroll
      for (int part = 0; part < 2; ++part)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int ib = 2 * kk; ib < 4; ++ib) {
            const int at = ib < 2 ? ib : 2 * ib - 2 + kk;
            o[ib] = scan_mfma(vf[kk], __builtin_bit_cast(bf16x8, s_p[at][part][lane]), o[ib]);
          }
      const RowBuffer to(a.out + (static_cast<int64_t>(r0 + c0) * H + h) * Dv + col0);
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) to.store(16 * ib + n < nrow, 4 * ((16 * ib + n) * H * Dv + 4 * g4), o[ib]);
    }
    // the state after the chunk
    u32x4 wv[2][2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const u32x4 x = __builtin_bit_cast(u32x4, vf[kk]);
      const f32x4s w0 = *reinterpret_cast<const f32x4s*>(s_w + 32 * kk + 4 * g4), w1 = *reinterpret_cast<const f32x4s*>(s_w + 32 * kk + 16 + 4 * g4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float wa = e < 2 ? w0[2 * e] : w1[2 * e - 4], wb = e < 2 ? w0[2 * e + 1] : w1[2 * e - 3];
        uint32_t hi, lo;
        split_pair(lo_bf(x[e]) * wa, hi_bf(x[e]) * wb, hi, lo);
        wv[kk][0][e] = hi, wv[kk][1][e] = lo;
      }
    }
    const float chunk_decay = __builtin_amdgcn_exp2f(total);
    // fragments a block ahead of their products, where there are registers for them (a read in front of every product: lightning
    // over 512 rows of 28 heads 52 us, so 47)
    constexpr int kAhead = Summarise ? 0 : 1;
    bf16x8 kf[1 + kAhead][Silu ? 2 : 1][2];
    auto read_keys = [&](int db) __attribute__((always_inline)) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        kf[db & kAhead][0][kk] = key_frag(s_k, db, kk);
        if constexpr (Silu) kf[db & kAhead][1][kk] = key_frag(s_klo, db, kk);
      }
    };
    if (kAhead) read_keys(0);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      if (db + kAhead < DB) read_keys(db + kAhead);
      if (kAhead) __builtin_amdgcn_sched_barrier(0);
      f32x4s acc = S[db] * chunk_decay;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        acc = scan_mfma(kf[db & kAhead][0][kk], __builtin_bit_cast(bf16x8, wv[kk][0]), acc);
        acc = scan_mfma(kf[db & kAhead][0][kk], __builtin_bit_cast(bf16x8, wv[kk][1]), acc);
        if constexpr (Silu) acc = scan_mfma(kf[db & kAhead][1][kk], __builtin_bit_cast(bf16x8, wv[kk][0]), acc);
      }
      S[db] = acc;
    }
    __syncthreads();                                   // every wave is done with this chunk's rows
    if (c0 + kScanRows < rows) {
      stage(min(kScanRows, rows - c0 - kScanRows));
      fetch(c0 + 2 * kScanRows);                       // (no row past the segment is read)
    }
  }
  float* to = Summarise ? wsp : (last ? st : nullptr);
  if (to != nullptr) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 4; ++r) to[static_cast<int64_t>(16 * db + 4 * g4 + r) * Dv + n] = S[db][r];
  }
  if (Summarise && vs == 0 && tid == 0) a.workspace[static_cast<int64_t>(segments) * H * D * Dv + place] = seg_total;
}

// The same with 128 columns to a workgroup and heads of 64 and 128, by eight waves that multiply and eight that stage: the rows of the
// next chunk go through their silu and into the other image of two while this one's products run, and so do the own weights, which
// the multiplying waves need last.  A wave issues a vector instruction every five cycles or so however simple it is, and a SIMD
// takes one in under three: two waves on a SIMD that do both, one behind the other, leave half of it idle (the kernel above: 12400 cycles a
// chunk; with the staging dealt among the products of the same waves 12000; so 8600), and 128 registers hold either half.
// Two barriers a chunk (one in Summarise): behind the first the own weights and the next keys beside the state times the queries,
// behind the second the next queries and values beside the weights times the values and the state's update.
// Bound by vector instructions (54 % of the time, the matrix pipe 21 %; silu and splits of 24576 values a chunk are most of them) and by
// waits at the barriers (38 %).  28 heads of 128 x 128, lightning: one prompt of 8192 rows 149 -> 133 us, four of 2000 179 -> 142, six of 1365
// 128 -> 106; plain decays: one of 8192 118 -> 103.
template <int D, bool Silu, bool Summarise, bool Chained>
__global__ __launch_bounds__(1024, 4) void chunk_scan_piped_kernel(ChunkScanArgs a, int seg_rows, int segments, bool short_too) {
  constexpr int NW = 8, NT = 64 * NW, KC = D / 8, VC = 2 * NW, KP = 2 * D, VP = 32 * NW, SD = D / 32, DB = D / 16;
  constexpr int KPT = kScanRows * KC / NT, VPT = 2, kKeyImage = kScanRows * KP, kValueImage = kScanRows * VP;
  static_assert(kScanRows * KC % NT == 0, "every thread stages whole chunks of 16 bytes");
  typedef ChunkOrder<KC> KOrder;
  typedef ChunkOrder<VC> VOrder;
  __shared__ __attribute__((aligned(16))) char s_k[2 * kKeyImage], s_v[2 * kValueImage];
  __shared__ __attribute__((aligned(16))) char s_q[Summarise ? 16 : 2 * kKeyImage], s_klo[Silu ? 2 * kKeyImage : 16];
  __shared__ __attribute__((aligned(16))) u32x4 s_p[Summarise ? 1 : 6][2][64];
  __shared__ __attribute__((aligned(16))) float s_cum[2][kScanRows], s_b[2][kScanRows], s_w[2][kScanRows];
  const int h = blockIdx.x, vs = blockIdx.y, number = blockIdx.z;
  const bool whole = number >= segments;
  PieceAt seg;
  if (!whole) {
    seg = segment_at(a, seg_rows, number);
    if (seg.seq < 0) return;
  } else {
    seg.seq = number - segments, seg.index = 0;
    seg.row0 = a.query_start_loc[seg.seq], seg.rows = a.query_start_loc[seg.seq + 1] - seg.row0;
  }
  const int s = seg.seq, r0 = seg.row0, rows_all = seg.rows;
  if (rows_all <= 0) return;                           // (a sequence without rows: its slot may be anything)
  if constexpr (!Summarise) {
    static_assert(sizeof(s_k) >= 16 * D && sizeof(s_v) >= 2048 * NW, "the scratch of single rows");
    if (rows_all < kScanMinRows) {                     // (a segment has more)
      if (short_too && threadIdx.x < NT) scan_single_rows<D, NW, Silu>(a, h, s, r0, rows_all, vs * 16 * NW, reinterpret_cast<float*>(s_k), reinterpret_cast<float*>(s_v));
      return;
    }
  }
  if (rows_all < kScanMinRows || (whole && rows_all > seg_rows)) return;
  const int r_lo = whole ? 0 : seg.index * seg_rows, rows = r_lo + min(rows_all - r_lo, seg_rows);        // (end of this workgroup's rows)
  const bool last = rows == rows_all;
  const bool copies = Summarise && last;               // nothing comes behind the last segment: its place holds the state in front of the portion
  if (copies && Chained) return;
  const int tid = threadIdx.x % NT, lane = tid & 63, n = lane & 15, g4 = lane >> 4;
  const int all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = all % NW;
  const bool stager = all >= NW;
  const int H = a.num_heads, Dv = a.v_dim, g = h / (H / a.num_qk_heads), col0 = vs * 16 * NW + 16 * wave;
  const int slot = a.slot_idx[s];
  float* st = slot >= 0 ? a.state + (static_cast<int64_t>(slot) * H + h) * D * Dv + col0 : nullptr;
  const float l2_const = a.decay ? fmaxf(a.decay[h] > 0.f ? log2f(a.decay[h]) : -INFINITY, kMinLog2) : 0.f;
  const float skip = a.skip ? a.skip[h] : 0.f;
  // (places in the workspace: as above)
  const int64_t place = static_cast<int64_t>(number) * H + h;
  float* wsp = whole ? nullptr : a.workspace + place * D * Dv + col0;
  const bool carry = st != nullptr && a.context_lens[s] > 0;
  const float* init = Summarise ? nullptr : whole ? (carry ? st : nullptr) : wsp;
  if (copies) {
    if (carry && threadIdx.x < NT) copy_columns<D>(st, wsp, Dv, lane);
    return;
  }
  float seg_total = 0.f;

  const uint16_t* qp = a.q + static_cast<int64_t>(g) * D;
  const uint16_t* kp = a.k + static_cast<int64_t>(g) * D;
  const uint16_t* vp = a.v + static_cast<int64_t>(h) * Dv + vs * 16 * NW;
  u32x4 rk[KPT], rq[Summarise ? 1 : KPT], rv[VPT];
  float rl = 0.f, rb = 0.f;
  auto fetch_rows = [&](auto& to, const uint16_t* base, int64_t stride, auto chunks, int c0) __attribute__((always_inline)) {
    constexpr int kChunks = decltype(chunks)::value;
    const int nrow = min(kScanRows, rows - c0);
    const RowBuffer r(base + (r0 + c0) * stride);
#pragma unroll
    for (int u = 0; u < static_cast<int>(sizeof(to) / sizeof(to[0])); ++u) {
      const int idx = tid + NT * u, j = idx / kChunks, ch = idx % kChunks;
      to[u] = r.load(j < nrow, 2 * (j * static_cast<int>(stride) + 8 * ch));
    }
  };
  auto fetch_keys = [&](int c0) __attribute__((always_inline)) {
    fetch_rows(rk, kp, a.k_stride, Const<KC>{}, c0);
    const int nrow = min(kScanRows, rows - c0), at = 4 * lane * H;
    const int64_t t0 = r0 + c0;
    if (a.log2_decay || a.v_scale) {
      rl = RowBuffer(a.log2_decay + t0 * H + h).load1(a.log2_decay && lane < nrow, at);
      rb = RowBuffer(a.v_scale + t0 * H + h).load1(a.v_scale && lane < nrow, at);
    }
  };
  auto fetch_queries = [&](int c0) __attribute__((always_inline)) {
    if constexpr (!Summarise) fetch_rows(rq, qp, a.q_stride, Const<KC>{}, c0);
  };
  auto fetch_values = [&](int c0) __attribute__((always_inline)) { fetch_rows(rv, vp, a.v_stride, Const<VC>{}, c0); };
  // Half `i` of a 16-byte chunk of this thread's keys, queries or values into image `to`: four values side by side, stored with the
  // second half.  (Rows past the portion were fetched as zeros, and silu(0) = 0.)
  u32x4 half_hi, half_lo;
  auto half = [&](const u32x4& raw, int i) __attribute__((always_inline)) {
    float x[4], y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = e & 1 ? hi_bf(raw[2 * i + e / 2]) : lo_bf(raw[2 * i + e / 2]);
    if constexpr (Silu) {                              // (silu_fast, step by step)
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = -1.4426950408889634f * x[e];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = __builtin_amdgcn_exp2f(y[e]);
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = 1.f + y[e];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = __builtin_amdgcn_rcpf(y[e]);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] *= y[e];
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      uint32_t hi = raw[2 * i + e], lo = 0;
      if constexpr (Silu) split_pair(x[2 * e], x[2 * e + 1], hi, lo);
      half_hi[2 * i + e] = hi, half_lo[2 * i + e] = lo;
    }
  };
  auto key_half = [&](int i, int to) __attribute__((always_inline)) {
    half(rk[i / 2], i % 2);
    if (i % 2 == 0) return;
    const int idx = tid + NT * (i / 2), j = idx / KC, ch = idx % KC, at = to * kKeyImage + j * KP + 16 * (ch ^ KOrder::twist(j));
    st16(s_k + at, half_hi);
    if constexpr (Silu) st16(s_klo + at, half_lo);
  };
  auto query_half = [&](int i, int to) __attribute__((always_inline)) {
    if constexpr (!Summarise) {
      half(rq[i / 2], i % 2);
      if (i % 2 == 0) return;
      const int idx = tid + NT * (i / 2), j = idx / KC, ch = idx % KC;
      st16(s_q + to * kKeyImage + j * KP + 16 * (ch ^ KOrder::twist(j)), half_hi);
    }
  };
  auto value_half = [&](int i, int to) __attribute__((always_inline)) {
    half(rv[i / 2], i % 2);
    if (i % 2 == 0) return;
    const int idx = tid + NT * (i / 2), j = idx / VC, ch = idx % VC;
    st16(s_v + to * kValueImage + j * VP + 16 * (ch ^ VOrder::twist(j)), half_hi);
  };
  constexpr int kKeyHalves = 2 * KPT, kValueHalves = 2 * VPT;
  // running sums of a chunk's log2 decays (rows past the portion add 0), by the first of the staging waves
  auto stage_decays = [&](int nrow, int to) __attribute__((always_inline)) {
    if (wave != 0) return;
    const float cum = a.log2_decay ? lane_sums(fmaxf(rl, kMinLog2)) : static_cast<float>(min(lane + 1, nrow)) * l2_const;
    const float total = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cum), 63));
    s_cum[to][lane] = cum;
    const float b = a.v_scale ? rb : 1.f;
    s_b[to][lane] = b;
    const float left = Silu ? static_cast<float>(nrow - 1 - lane) * l2_const : total - cum;
    s_w[to][lane] = lane < nrow ? __builtin_amdgcn_exp2f(left) * b : 0.f;
  };
  // LDS offsets of this lane's fragments: as above
  const int kt = KOrder::twist(n), Rt = 4 * g4 + (n >> 2), kT = KOrder::twist(Rt), vT = VOrder::twist(Rt);
  auto row_frag = [&](const char* img, int block, int sd) { return __builtin_bit_cast(bf16x8, ld16(img + (16 * block + n) * KP + 16 * ((4 * sd + g4) ^ kt))); };
  auto row_frag_halves = [&](const char* img, int block, int sd) {
    const char* row = img + (16 * block + n) * KP + 8 * (g4 & 1);
    const u32x2 x = *reinterpret_cast<const u32x2*>(row + 16 * ((4 * sd + (g4 >> 1)) ^ kt));
    const u32x2 y = *reinterpret_cast<const u32x2*>(row + 16 * ((4 * sd + 2 + (g4 >> 1)) ^ kt));
    return __builtin_bit_cast(bf16x8, (u32x4{x[0], x[1], y[0], y[1]}));
  };
  auto key_frag = [&](const char* img, int db, int kk) {
    const char* p = img + (32 * kk + Rt) * KP + 16 * ((2 * db + ((n & 3) >> 1)) ^ kT) + 8 * (n & 1);
    return frag_of(read_transposed(p), read_transposed(p + 16 * KP));
  };
  auto value_frag = [&](const char* img, int kk) {
    const char* p = img + (32 * kk + Rt) * VP + 16 * ((2 * wave + ((n & 3) >> 1)) ^ vT) + 8 * (n & 1);
    return frag_of(read_transposed(p), read_transposed(p + 16 * VP));
  };

  // ---- the staging waves
  // A block of the own weights of the chunk in image `cur` as hi + lo fragments: rows 16 ib + n, keys 32 wk ..
  auto own_weights = [&](int cur) __attribute__((always_inline)) {
    const int ib = wave >> 1, wk = wave & 1, i = 16 * ib + n;
    if (2 * wk > ib) return;
    const char *kimg = s_k + cur * kKeyImage, *qimg = s_q + cur * kKeyImage;
    bf16x8 own_q[SD], own_k[SD][2];
#pragma unroll
    for (int sd = 0; sd < SD; ++sd) {
      own_q[sd] = row_frag(qimg, ib, sd);
#pragma unroll
      for (int t = 0; t < 2; ++t) own_k[sd][t] = row_frag(kimg, 2 * wk + t, sd);       // (block 2 wk + 1 may lie behind the rows: masked)
    }
    const float cum_i = s_cum[cur][i];
    f32x4s sc[2], cum_j[2], b_j[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      sc[t] = f32x4s{0.f, 0.f, 0.f, 0.f};
      if constexpr (!Silu) {
        const int j = 16 * (2 * wk + t) + 4 * g4;
        cum_j[t] = *reinterpret_cast<const f32x4s*>(s_cum[cur] + j), b_j[t] = *reinterpret_cast<const f32x4s*>(s_b[cur] + j);
      }
    }
    __builtin_amdgcn_sched_barrier(0);                 // (all on their way: left to itself the compiler waits for each)
#pragma unroll
    for (int sd = 0; sd < SD; ++sd)
#pragma unroll
      for (int t = 0; t < 2; ++t) sc[t] = scan_mfma(own_k[sd][t], own_q[sd], sc[t]);
    u32x4 hi, lo;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      float p[2];
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        const int t = x >> 1, r = 2 * (x & 1) + y, j = 16 * (2 * wk + t) + 4 * g4 + r;
        float span, bj = 1.f;                          // log2 of the decay between row j and row i; j's input weight
        if constexpr (Silu) span = static_cast<float>(i - j) * l2_const;
        else span = cum_i - cum_j[t][r], bj = b_j[t][r];
        p[y] = j <= i ? sc[t][r] * __builtin_amdgcn_exp2f(span) * bj : 0.f;
      }
      uint32_t a, b;
      split_pair(p[0], p[1], a, b);
      hi[x] = a, lo[x] = b;
    }
    const int at = ib < 2 ? ib : 2 * ib - 2 + wk;
    s_p[at][0][lane] = hi;
    s_p[at][1][lane] = lo;
  };

  // ---- the multiplying waves
  f32x4s S[DB], o[4];                                  // S[16 db + 4 g4 + r][col0 + n]
  bf16x8 vf[2];
  u32x4 wv[2][2];                                      // the values with the decays up to the chunk's end, hi and lo
  // the state before the chunk times the queries
  auto state_times_queries = [&](int cur) __attribute__((always_inline)) {
    const char* qimg = s_q + cur * kKeyImage;
#pragma unroll
    for (int x = 0; x < 4; ++x) o[x] = f32x4s{0.f, 0.f, 0.f, 0.f};
    float cum[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) cum[x] = s_cum[cur][16 * x + n];
    bf16x8 qf[6];                                      // of two blocks of rows a step of 32 d ahead
    u32x4 sf[2][2];                                    // the state's d 32 sd + 4 g4 + e for e < 4, 32 sd + 16 + 4 g4 + e - 4 after, hi and lo
    auto read_queries = [&](int sd, int x) __attribute__((always_inline)) { qf[x < 2 ? x + 4 * (sd & 1) : x] = row_frag_halves(qimg, x, sd); };
    auto split_state = [&](int sd, int e) __attribute__((always_inline)) {
      uint32_t x, y;
      split_pair(S[2 * sd + (e >> 1)][2 * (e & 1)], S[2 * sd + (e >> 1)][2 * (e & 1) + 1], x, y);
      sf[sd & 1][0][e] = x, sf[sd & 1][1][e] = y;
    };
    read_queries(0, 0), read_queries(0, 1);
#pragma unroll
    for (int e = 0; e < 4; ++e) split_state(0, e);
    __builtin_amdgcn_sched_barrier(0);
    unrolled<8 * SD>([&](auto at) __attribute__((always_inline)) {
      constexpr int step = decltype(at)::value, sd = step / 8, x = step % 8 < 4 ? step % 2 : 2 + step % 2, part = step / 2 % 2;
      if constexpr (step % 8 == 0) read_queries(sd, 2), read_queries(sd, 3);
      if constexpr (step % 8 == 4 && sd + 1 < SD) read_queries(sd + 1, 0), read_queries(sd + 1, 1);
      o[x] = scan_mfma(__builtin_bit_cast(bf16x8, sf[sd & 1][part]), qf[x < 2 ? x + 4 * (sd & 1) : x], o[x]);
      if constexpr (sd + 1 < SD && step % 2 == 0) split_state(sd + 1, step % 8 / 2);
      __builtin_amdgcn_sched_barrier(0);
    });
#pragma unroll
    for (int x = 0; x < 4; ++x) o[x] *= __builtin_amdgcn_exp2f(cum[x]);
    if (skip != 0.f) {
      const char* vimg = s_v + cur * kValueImage;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const u32x2 vi = *reinterpret_cast<const u32x2*>(vimg + (16 * x + n) * VP + 16 * ((2 * wave + (g4 >> 1)) ^ VOrder::twist(n)) + 8 * (g4 & 1));
        o[x][0] = fmaf(skip, lo_bf(vi[0]), o[x][0]), o[x][1] = fmaf(skip, hi_bf(vi[0]), o[x][1]);
        o[x][2] = fmaf(skip, lo_bf(vi[1]), o[x][2]), o[x][3] = fmaf(skip, hi_bf(vi[1]), o[x][3]);
      }
    }
  };
  auto read_values = [&](int cur) __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) vf[kk] = value_frag(s_v + cur * kValueImage, kk);
  };
  auto weigh_values = [&](int cur) __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const u32x4 x = __builtin_bit_cast(u32x4, vf[kk]);
      const f32x4s w0 = *reinterpret_cast<const f32x4s*>(s_w[cur] + 32 * kk + 4 * g4), w1 = *reinterpret_cast<const f32x4s*>(s_w[cur] + 32 * kk + 16 + 4 * g4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float wa = e < 2 ? w0[2 * e] : w1[2 * e - 4], wb = e < 2 ? w0[2 * e + 1] : w1[2 * e - 3];
        uint32_t hi, lo;
        split_pair(lo_bf(x[e]) * wa, hi_bf(x[e]) * wb, hi, lo);
        wv[kk][0][e] = hi, wv[kk][1][e] = lo;
      }
    }
  };
  // the own weights times the values
  auto finish_rows = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
    for (int part = 0; part < 2; ++part) {
      u32x4 pf[6];
#pragma unroll
      for (int at = 0; at < 6; ++at) pf[at] = s_p[at][part][lane];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int x = 2 * kk; x < 4; ++x) o[x] = scan_mfma(vf[kk], __builtin_bit_cast(bf16x8, pf[x < 2 ? x : 2 * x - 2 + kk]), o[x]);
    }
    const int nrow = min(kScanRows, rows - c0);
    const RowBuffer to(a.out + (static_cast<int64_t>(r0 + c0) * H + h) * Dv + col0);
#pragma unroll
    for (int x = 0; x < 4; ++x) to.store(16 * x + n < nrow, 4 * ((16 * x + n) * H * Dv + 4 * g4), o[x]);
  };
  // the state after the chunk
  auto update_state = [&](int cur, float total) __attribute__((always_inline)) {
    const char *kimg = s_k + cur * kKeyImage, *klo = s_klo + (Silu ? cur * kKeyImage : 0);
    const float chunk_decay = __builtin_amdgcn_exp2f(total);
    bf16x8 kf[2][Silu ? 2 : 1];                        // fragments of 32 keys and 16 d, one set ahead of its products
    auto read_keys = [&](int at) __attribute__((always_inline)) {
      kf[at & 1][0] = key_frag(kimg, at / 2, at & 1);
      if constexpr (Silu) kf[at & 1][1] = key_frag(klo, at / 2, at & 1);
    };
    read_keys(0);
#pragma unroll
    for (int at = 0; at < 2 * DB; ++at) {
      const int db = at / 2, kk = at & 1;
      if (at + 1 < 2 * DB) read_keys(at + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (kk == 0) S[db] *= chunk_decay;
      S[db] = scan_mfma(kf[kk][0], __builtin_bit_cast(bf16x8, wv[kk][0]), S[db]);
      S[db] = scan_mfma(kf[kk][0], __builtin_bit_cast(bf16x8, wv[kk][1]), S[db]);
      if constexpr (Silu) S[db] = scan_mfma(kf[kk][1], __builtin_bit_cast(bf16x8, wv[kk][0]), S[db]);
    }
  };

  // (a loop for either kind of waves, with the same barriers: in one loop the registers of both would be alive at once)
  if (stager) {
    fetch_keys(r_lo), fetch_queries(r_lo), fetch_values(r_lo);
#pragma unroll
    for (int i = 0; i < kKeyHalves; ++i) key_half(i, 0);
#pragma unroll
    for (int i = 0; i < kKeyHalves; ++i) query_half(i, 0);
#pragma unroll
    for (int i = 0; i < kValueHalves; ++i) value_half(i, 0);
    stage_decays(min(kScanRows, rows - r_lo), 0);
    fetch_keys(r_lo + kScanRows), fetch_queries(r_lo + kScanRows), fetch_values(r_lo + kScanRows);      // (no row past the segment is read)
    for (int c0 = r_lo, cur = 0; c0 < rows; c0 += kScanRows, cur ^= 1) {
      const bool more = c0 + kScanRows < rows;
      const int next = cur ^ 1;
      __syncthreads();                                 // the chunk is there, and nobody reads the other image
      if constexpr (!Summarise) own_weights(cur);
      if (more) {
#pragma unroll
        for (int i = 0; i < kKeyHalves; ++i) key_half(i, next);
        stage_decays(min(kScanRows, rows - c0 - kScanRows), next);
        fetch_keys(c0 + 2 * kScanRows);
      }
      if constexpr (!Summarise) __syncthreads();       // the own weights are there
      if (more) {
#pragma unroll
        for (int i = 0; i < kKeyHalves; ++i) query_half(i, next);
        fetch_queries(c0 + 2 * kScanRows);
#pragma unroll
        for (int i = 0; i < kValueHalves; ++i) value_half(i, next);
        fetch_values(c0 + 2 * kScanRows);
      }
    }
    return;
  }
  if (Summarise || Chained || whole) load_state(S, init, 4 * g4, Dv, n);
  else segment_state(S, a, seg, seg_rows, segments, number, h, D * Dv, carry, col0, 4 * g4, Dv, n);
  for (int c0 = r_lo, cur = 0; c0 < rows; c0 += kScanRows, cur ^= 1) {
    __syncthreads();
    const float total = s_cum[cur][kScanRows - 1];
    seg_total += total;
    if constexpr (!Summarise) state_times_queries(cur);
    read_values(cur);
    if constexpr (!Summarise) {
      __syncthreads();
      finish_rows(c0);
    }
    weigh_values(cur);
    update_state(cur, total);
  }
  float* to = Summarise ? wsp : (last ? st : nullptr);
  if (to != nullptr) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 4; ++r) to[static_cast<int64_t>(16 * db + 4 * g4 + r) * Dv + n] = S[db][r];
  }
  if (Summarise && vs == 0 && tid == 0) a.workspace[static_cast<int64_t>(segments) * H * D * Dv + place] = seg_total;
}

// The segments' summaries (each segment's state had it started from zero) become the states in front of the segments:
// run = carried state; per segment: place <- run, run <- 2^(segment's sum of log2 decays) run + summary.  Four elements per
// thread.  grid = (heads, segments, parts per segment): a portion's workgroups deal the parts of 1024 elements among them.
__global__ __launch_bounds__(256) void chunk_scan_chain_kernel(ChunkScanArgs a, int head_dim, int seg_rows, int segments) {
  const int h = blockIdx.x, H = a.num_heads, per_head = head_dim * a.v_dim;
  const PieceAt seg = segment_at(a, seg_rows, blockIdx.y);
  const int s = seg.seq;
  if (s < 0) return;
  const int slot = a.slot_idx[s], segs = (seg.rows - 1) / seg_rows + 1;
  const int64_t step = static_cast<int64_t>(H) * per_head, first = static_cast<int64_t>(blockIdx.y - seg.index) * H + h;
  const float* totals = a.workspace + segments * step + first;
  const bool carry = slot >= 0 && a.context_lens[s] > 0;
  for (int part = seg.index + segs * blockIdx.z; 1024 * part < per_head; part += segs * gridDim.z) {
    const int idx = 1024 * part + 4 * threadIdx.x;
    if (idx >= per_head) return;
    f32x4s run = f32x4s{0.f, 0.f, 0.f, 0.f};
    if (carry) run = *reinterpret_cast<const f32x4s*>(a.state + (static_cast<int64_t>(slot) * H + h) * per_head + idx);
    float* p = a.workspace + first * per_head + idx;
    for (int seg0 = 0; seg0 < segs; seg0 += 8) {         // eight summaries in flight together (the last ones may lie past the end: read again)
      f32x4s summary[8];
      float decay[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int at = min(seg0 + u, segs - 1);
        summary[u] = *reinterpret_cast<const f32x4s*>(p + at * step);
        decay[u] = totals[at * H];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (seg0 + u < segs) {
          *reinterpret_cast<f32x4s*>(p + (seg0 + u) * step) = run;
          run = __builtin_amdgcn_exp2f(decay[u]) * run + summary[u];     // (behind the last segment: not used)
        }
    }
  }
}

template <int D, int NW, bool Silu>
void launch_chunk_scan_as(const ChunkScanArgs& a, ScanSegments sg, bool short_too, hipStream_t st) {
  const dim3 block(64 * NW);
  const unsigned slices = a.v_dim / (16 * NW);
  auto scan = [&](auto summarise, unsigned pieces, bool shorts) {
    constexpr bool Summarise = decltype(summarise)::value;
    const dim3 grid(a.num_heads, slices, pieces);
    auto launch = [&](auto chained) {
      constexpr bool Chained = decltype(chained)::value;
      if constexpr (NW == 8 && D >= 64) hipLaunchKernelGGL((chunk_scan_piped_kernel<D, Silu, Summarise, Chained>), grid, dim3(1024), 0, st, a, sg.rows, sg.count, shorts);
      else hipLaunchKernelGGL((chunk_scan_kernel<D, NW, Silu, Summarise, Chained>), grid, block, 0, st, a, sg.rows, sg.count, shorts);
    };
    if (sg.count > 0 && !sg.chained) launch(std::false_type{});
    else launch(std::true_type{});
  };
  if (sg.count > 0) {
    scan(std::true_type{}, sg.count, false);
    if (sg.chained) hipLaunchKernelGGL(chunk_scan_chain_kernel, dim3(a.num_heads, sg.count, (D * a.v_dim + 3071) / 3072), dim3(256), 0, st, a, D, sg.rows, sg.count);
  }
  scan(std::false_type{}, sg.count + a.num_seqs, short_too);
}

// Portions too short for a chunk run in the chunks' launch, where they cost no launch (about 4 us) and fill what a long portion
// leaves idle.  A workgroup of that launch has a compute unit to itself, though, and eight waves of its sixteen (heads of 64) do nothing for a
// short portion.  So those of states of 64 x 128 have a launch of their own where there are
// more (head, short portion) pairs than kManyShort and the chunks fill half of the chip by themselves, or three times as many: 28 heads, lightning, 2048 rows beside
// 255 single ones 110 -> 87 us, 40 portions of 40 beside 200 92 -> 72, ten of 300 beside 250 104 -> 87, but four of 600 beside 60 38 (48 apart);
// 300 beside 255 is level.  Portions of one chunk that seem to fill the chip may be many short ones of several rows, which gain more: a quarter as
// many pairs (60 of 7 rows beside 40 of 64 96 -> 75).  (Sixteen waves moved the line: 2048 beside 127 would gain apart by now, 68 and 58, four of 600
// beside 200 77 and 67.)  States of 128 rows are level.
//
// Where no portion has a chunk, theirs is the only launch, and its occupancy hides a row's round trips: 28 heads of 128 x 128, 64
// portions of 7 rows 102 -> 58 us, 20 43 -> 25; of 64 x 128, 64 portions of 7 rows 77 -> 40 (a thread per value column, before: 156, 80,
// 55).
constexpr int kManyShort = 3584;
// Single rows whose states do not fit the chip's last-level cache (256 MB) pass through memory fastest with 64 KB a compute unit on
// their way: unused LDS keeps more workgroups away.  28 heads of 128 x 128, 512 single rows 363 -> 315 us; states of 268 MB are faster
// without (81 against 88 us).
constexpr int64_t kManyStateBytes = 384ll << 20;
inline unsigned spare_lds(int head_dim, int used) {
  const int together = 256 / head_dim;     // workgroups of 64 value columns
  return 163840 / (together + 1) + 1024 - used;
}

// A step's rows, of portions of up to max_query_len rows (below kScanMinRows: every portion goes row by row, however long).
template <bool Silu>
void launch_chunk_scan(const ChunkScanArgs& a, int num_tokens, int head_dim, int max_query_len, ScanSegments sg, hipStream_t st) {
  const int nw = scan_waves(sg.lanes, a.v_dim);
  const bool chunks = max_query_len >= kScanMinRows;
  const int64_t shorts = static_cast<int64_t>(a.num_heads) * (chunks ? a.num_seqs - long_portions(num_tokens, a.num_seqs, max_query_len) : a.num_seqs);
  const bool filled = sg.lanes * (a.v_dim / (16 * nw)) >= 128;
  const int most = !filled ? 3 * kManyShort : max_query_len <= kScanRows ? kManyShort / 4 : kManyShort;
  const bool apart = !chunks || (head_dim <= 64 && nw == 8 && shorts > most);
  const bool single = !chunks && num_tokens - a.num_seqs <= a.num_seqs / 4;
  auto launch = [&](auto d) {
    constexpr int D = decltype(d)::value;
    auto launch_short = [&](auto w) {
      constexpr int NW = decltype(w)::value, used = 16 * D + 2048 * NW;
      const unsigned spare = single && shorts * D * a.v_dim * 4 > kManyStateBytes && NW == 4 ? spare_lds(D, used) : 0;
      hipLaunchKernelGGL((scan_short_kernel<D, NW, Silu>), dim3(a.num_heads, a.v_dim / (16 * NW), a.num_seqs), dim3(64 * NW), spare, st, a,
                         chunks ? kScanMinRows - 1 : 0x7fffffff);
    };
    if (apart) {
      if (a.v_dim % 64 == 0) launch_short(std::integral_constant<int, 4>{});
      else launch_short(std::integral_constant<int, 2>{});
    }
    if (!chunks) return;
    if (nw == 8) launch_chunk_scan_as<D, 8, Silu>(a, sg, !apart, st);
    else if (nw == 4) launch_chunk_scan_as<D, 4, Silu>(a, sg, !apart, st);
    else launch_chunk_scan_as<D, 2, Silu>(a, sg, !apart, st);
  };
  if (head_dim == 32) launch(std::integral_constant<int, 32>{});
  else if (head_dim == 64) launch(std::integral_constant<int, 64>{});
  else launch(std::integral_constant<int, 128>{});
}

}  // namespace
}  // namespace hymeta
