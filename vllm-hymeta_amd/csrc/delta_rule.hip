// Gated delta rule: linear attention whose state forgets by a scalar per head and token and is corrected towards each
// token's value before it is read:
//   S <- a_t S;   u_t = beta_t (v_t - S^T k_t);   S <- S + k_t u_t^T;   o_t = S^T q_t
// with unit-length queries and keys, the state fp32 and carried per sequence.  Beside the decayed scan (decay_scan.hip),
// whose state only adds what a token brings.
#include "act_types.h"
#include "row_copy.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace hymeta {

namespace {

constexpr float kMinLog2 = -1.0e4f;         // a decay of 0 (or an overflowed step size): finite, so that differences of sums stay numbers

template <typename A>
__device__ __forceinline__ float exp2_act(float x) {
  return A::kDtype == HYMETA_F32 ? exp2f(x) : __builtin_amdgcn_exp2f(x);
}

// Token by token.  grid = (heads, sequences, value columns in runs of 256); a thread owns one value column c and keeps
// that column of the state, S[:, c], in registers; q_t and k_t go through LDS, their lengths come out of the same loop.
template <typename A, int DMAX>
__global__ __launch_bounds__(256) void delta_rule_rows_kernel(hymeta_delta_rule_args a, int min_rows, int max_rows) {
  typedef typename A::elem elem;
  __shared__ __attribute__((aligned(16))) float s_q[2][DMAX], s_k[2][DMAX];
  const int h = blockIdx.x, s = blockIdx.y;
  const int c = blockIdx.z * 256 + threadIdx.x;
  const int H = a.num_heads, D = a.head_dim, Dv = a.v_dim;
  const int g = h / (H / a.num_qk_heads);
  const int r0 = a.query_start_loc[s], r1 = a.query_start_loc[s + 1];
  if (r1 - r0 < min_rows || r1 - r0 > max_rows) return;
  const int slot = a.slot_idx[s];
  const bool live = c < Dv;
  float* st = (slot >= 0) ? a.state + ((static_cast<int64_t>(slot) * H + h) * D) * Dv : nullptr;
  float S[DMAX];
  const bool carry = st != nullptr && a.context_lens[s] > 0 && live;
#pragma unroll
  for (int d = 0; d < DMAX; ++d) S[d] = (carry && d < D) ? st[static_cast<int64_t>(d) * Dv + c] : 0.f;
  float* out = static_cast<float*>(a.out);
  for (int t = r0; t < r1; ++t) {
    const elem* q = static_cast<const elem*>(a.q) + static_cast<int64_t>(t) * a.q_stride_t + static_cast<int64_t>(g) * D;
    const elem* k = static_cast<const elem*>(a.k) + static_cast<int64_t>(t) * a.k_stride_t + static_cast<int64_t>(g) * D;
    const int buf = (t - r0) & 1;
    for (int d = threadIdx.x; d < DMAX; d += blockDim.x) {
      s_q[buf][d] = d < D ? A::ld(q + d) : 0.f;
      s_k[buf][d] = d < D ? A::ld(k + d) : 0.f;
    }
    const float v = live ? A::ld(static_cast<const elem*>(a.v) + static_cast<int64_t>(t) * a.v_stride_t + static_cast<int64_t>(h) * Dv + c) : 0.f;
    const float decay = exp2_act<A>(fmaxf(a.log2_decay[static_cast<int64_t>(t) * H + h], kMinLog2));
    const float beta = sigmoid_exact(A::ld(static_cast<const elem*>(a.beta_logit) + static_cast<int64_t>(t) * a.beta_stride_t + h));
    __syncthreads();           // one barrier per token: the next token fills the other buffer
    float dot = 0.f, kk = 0.f, qq = 0.f;
#pragma unroll
    for (int d = 0; d < DMAX; ++d) {           // (columns past D hold zeros)
      const float kd = s_k[buf][d], qd = s_q[buf][d];
      dot = fmaf(S[d], kd, dot);
      kk = fmaf(kd, kd, kk);
      qq = fmaf(qd, qd, qq);
    }
    const float ik = 1.f / sqrtf(kk + a.unit_eps), iq = a.q_scale / sqrtf(qq + a.unit_eps);
    const float u = beta * (v - decay * (dot * ik)) * ik;
    float o = 0.f;
#pragma unroll
    for (int d = 0; d < DMAX; ++d) {
      S[d] = fmaf(decay, S[d], s_k[buf][d] * u);
      o = fmaf(S[d], s_q[buf][d], o);
    }
    if (live) out[static_cast<int64_t>(t) * H * Dv + static_cast<int64_t>(h) * Dv + c] = o * iq;
  }
  if (st != nullptr && live) {
#pragma unroll
    for (int d = 0; d < DMAX; ++d)
      if (d < D) st[static_cast<int64_t>(d) * Dv + c] = S[d];
  }
}

// Sequences with one row (decode).  grid = (heads, sequences), 256 threads over the state in fours of value columns: a
// thread takes the columns 4 c4 .. 4 c4 + 3 of the rows d0, d0 + dstep, ... of S and keeps them in registers (16-byte loads,
// all in flight together).  S^T k and S^T q of the OLD state are reduced over the row groups in one go; what the token's own
// write adds to the output is u (k . q), so the state is read once and written once with one reduction between.  Norm: the
// head's output row goes through its RMS norm, weight and silu gate in the same launch.
constexpr int kStepMaxD = 256, kStepRows = 16;
template <typename A, bool Norm>
__global__ __launch_bounds__(256) void delta_rule_step_kernel(hymeta_delta_rule_args a) {
  __shared__ float s_q[kStepMaxD], s_k[kStepMaxD];
  __shared__ __attribute__((aligned(16))) float s_a[256 * 4], s_c[256 * 4], s_u[1024];
  __shared__ float red[4];
  const int h = blockIdx.x, s = blockIdx.y, t = a.query_start_loc[s];
  if (a.query_start_loc[s + 1] - t != 1) return;
  typedef typename A::elem elem;
  const int H = a.num_heads, D = a.head_dim, Dv = a.v_dim, Dv4 = Dv / 4;
  const int g = h / (H / a.num_qk_heads);
  const int c4 = threadIdx.x % Dv4, d0 = threadIdx.x / Dv4, dstep = 256 / Dv4, lane = threadIdx.x & 63;
  const int slot = a.slot_idx[s];
  float* st = slot >= 0 ? a.state + ((static_cast<int64_t>(slot) * H + h) * D) * Dv : nullptr;
  const bool carry = st != nullptr && a.context_lens[s] > 0;
  const uint32_t lane_at = d0 * Dv + 4 * c4;                      // (rows of S further on: a wave-uniform step)
  f32x4 S[kStepRows];
#pragma unroll
  for (int u = 0; u < kStepRows; ++u) {
    const int d = d0 + u * dstep;
    S[u] = (carry && d < D) ? *reinterpret_cast<const f32x4*>(st + u * dstep * Dv + lane_at) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const elem* q = static_cast<const elem*>(a.q) + static_cast<int64_t>(t) * a.q_stride_t + static_cast<int64_t>(g) * D;
  const elem* k = static_cast<const elem*>(a.k) + static_cast<int64_t>(t) * a.k_stride_t + static_cast<int64_t>(g) * D;
  const float decay = exp2_act<A>(fmaxf(a.log2_decay[static_cast<int64_t>(t) * H + h], kMinLog2));
  const float beta = sigmoid_exact(A::ld(static_cast<const elem*>(a.beta_logit) + static_cast<int64_t>(t) * a.beta_stride_t + h));
  // every wave sums the lengths and the product for itself
  float kk = 0.f, qq = 0.f, kq = 0.f;
  for (int d = lane; d < D; d += 64) {
    const float kd = A::ld(k + d), qd = A::ld(q + d);
    if (threadIdx.x < 64) s_k[d] = kd, s_q[d] = qd;
    kk = fmaf(kd, kd, kk);
    qq = fmaf(qd, qd, qq);
    kq = fmaf(kd, qd, kq);
  }
  kk = wave_sum(kk), qq = wave_sum(qq), kq = wave_sum(kq);
  const float ik = 1.f / sqrtf(kk + a.unit_eps), iq = a.q_scale / sqrtf(qq + a.unit_eps);
  __syncthreads();
  f32x4 pa = f32x4{0.f, 0.f, 0.f, 0.f}, pc = pa;
#pragma unroll
  for (int u = 0; u < kStepRows; ++u) {
    const int d = d0 + u * dstep;
    if (d >= D) continue;
    const float kd = s_k[d], qd = s_q[d];
#pragma unroll
    for (int e = 0; e < 4; ++e) pa[e] = fmaf(S[u][e], kd, pa[e]), pc[e] = fmaf(S[u][e], qd, pc[e]);
  }
  *reinterpret_cast<f32x4*>(&s_a[threadIdx.x * 4]) = pa;        // [d0][4 c4 + e]
  *reinterpret_cast<f32x4*>(&s_c[threadIdx.x * 4]) = pc;
  __syncthreads();
  float o[4] = {0.f, 0.f, 0.f, 0.f}, ss = 0.f;                  // columns threadIdx.x, + 256, ...
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = threadIdx.x + 256 * i;
    if (c >= Dv) continue;
    float da = 0.f, dc = 0.f;
    for (int gg = 0; gg < dstep; ++gg) da += s_a[gg * Dv + c], dc += s_c[gg * Dv + c];
    const float v = A::ld(static_cast<const elem*>(a.v) + static_cast<int64_t>(t) * a.v_stride_t + static_cast<int64_t>(h) * Dv + c);
    const float u = beta * (v - decay * (da * ik)) * ik;        // (with the key's length: what multiplies the raw key)
    s_u[c] = u;
    o[i] = iq * fmaf(u, kq, decay * dc);
    ss = fmaf(o[i], o[i], ss);
  }
  __syncthreads();
  if (st != nullptr) {
    const f32x4 u4 = *reinterpret_cast<const f32x4*>(&s_u[4 * c4]);
#pragma unroll
    for (int u = 0; u < kStepRows; ++u) {
      const int d = d0 + u * dstep;
      if (d >= D) continue;
      const float kd = s_k[d];
#pragma unroll
      for (int e = 0; e < 4; ++e) S[u][e] = fmaf(decay, S[u][e], kd * u4[e]);
      *reinterpret_cast<f32x4*>(st + u * dstep * Dv + lane_at) = S[u];
    }
  }
  const int64_t at = (static_cast<int64_t>(t) * H + h) * Dv;
  if constexpr (Norm) {
    ss = block_sum<4>(ss, red);
    const float inv = 1.f / sqrtf(ss / static_cast<float>(Dv) + a.norm_eps);
    const elem* gate = static_cast<const elem*>(a.gate) + static_cast<int64_t>(t) * a.gate_stride_t + static_cast<int64_t>(h) * Dv;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = threadIdx.x + 256 * i;
      if (c >= Dv) continue;
      const float gv = A::ld(gate + c);
      A::st(static_cast<elem*>(a.out) + at + c, o[i] * inv * a.norm_weight[c] * gv * sigmoid_exact(gv));
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = threadIdx.x + 256 * i;
      if (c < Dv) static_cast<float*>(a.out)[at + c] = o[i];
    }
  }
}

// A portion too short for a chunk, row by row in fp32 by NT threads over 4 C4 value columns of one head: a thread holds 4 columns of
// U rows of the state.  S^T k and S^T q of the state in front of a row are reduced together, over a wave's lanes and,
// in LDS, over the waves, whose sums every thread adds up for itself; the next row is on its way while one is worked on.  Two
// barriers a row, or none with one wave.
template <int D, int NT>
struct ShortScratch {
  __attribute__((aligned(16))) float dots[2][NT / 64][2][64];        // [row parity][wave][k, q][column]
  __attribute__((aligned(16))) float q[2][D], k[2][D];
};
template <int D, int C4, int NT>
__device__ __forceinline__ void delta_short_rows(const hymeta_delta_rule_args& a, int tid, int h, int s, int r0, int rows, int col0, ShortScratch<D, NT>& m) {
  typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
  constexpr int kGroups = NT / C4, U = D / kGroups, kEach = (D + 63) / 64, kWaves = NT / 64;
  static_assert(D % kGroups == 0 && 4 * C4 <= 64, "the state deals evenly over the threads");
  // (rows side by side where a thread has many: their queries and keys come four to a read)
  constexpr int kFirst = NT < 256 ? U : 1, kNext = NT < 256 ? 1 : kGroups;
  const int c4 = tid % C4, d0 = tid / C4 * kFirst, lane = tid & 63, wave = tid >> 6;
  const int H = a.num_heads, Dv = a.v_dim, g = h / (H / a.num_qk_heads);
  const int slot = a.slot_idx[s];
  float* st = slot >= 0 ? a.state + (static_cast<int64_t>(slot) * H + h) * D * Dv + col0 : nullptr;
  const bool carry = st != nullptr && a.context_lens[s] > 0;
  const uint32_t at = d0 * Dv + 4 * c4;
  f32x4 S[U];
#pragma unroll
  for (int u = 0; u < U; ++u) S[u] = carry ? *reinterpret_cast<const f32x4*>(st + u * kNext * Dv + at) : f32x4{0.f, 0.f, 0.f, 0.f};
  uint16_t kr[kEach], qr[kEach], vr[4], br;
  float l2;
  auto fetch = [&](int64_t t) __attribute__((always_inline)) {
    const uint16_t* q = static_cast<const uint16_t*>(a.q) + t * a.q_stride_t + static_cast<int64_t>(g) * D;
    const uint16_t* k = static_cast<const uint16_t*>(a.k) + t * a.k_stride_t + static_cast<int64_t>(g) * D;
    const uint16_t* v = static_cast<const uint16_t*>(a.v) + t * a.v_stride_t + static_cast<int64_t>(h) * Dv + col0 + 4 * c4;
#pragma unroll
    for (int j = 0; j < kEach; ++j) {
      const int d = min(lane + 64 * j, D - 1);
      kr[j] = k[d], qr[j] = q[d];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) vr[e] = v[e];
    l2 = a.log2_decay[t * H + h];
    br = static_cast<const uint16_t*>(a.beta_logit)[t * a.beta_stride_t + h];
  };
  fetch(r0);
  for (int i = 0; i < rows; ++i) {
    const int at_row = i & 1;
    float kk = 0.f, qq = 0.f, kq = 0.f, v[4];
#pragma unroll
    for (int j = 0; j < kEach; ++j) {
      const int d = lane + 64 * j;
      const bool in = D % 64 == 0 || d < D;
      const float kd = in ? bf2f(kr[j]) : 0.f, qd = in ? bf2f(qr[j]) : 0.f;
      if (wave == 0 && in) m.k[at_row][d] = kd, m.q[at_row][d] = qd;
      kk = fmaf(kd, kd, kk), qq = fmaf(qd, qd, qq), kq = fmaf(kd, qd, kq);
    }
    kk = wave_sum(kk), qq = wave_sum(qq), kq = wave_sum(kq);         // (every wave for itself)
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = bf2f(vr[e]);
    const float decay = __builtin_amdgcn_exp2f(fmaxf(l2, kMinLog2)), beta = sigmoid_exact(bf2f(br));
    const float ik = 1.f / sqrtf(kk + a.unit_eps), iq = a.q_scale / sqrtf(qq + a.unit_eps);
    __syncthreads();                                                 // the row's queries and keys are there
    if (i + 1 < rows) fetch(r0 + i + 1);
    float kd[U];
    f32x4 pa = f32x4{0.f, 0.f, 0.f, 0.f}, pc = pa;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      kd[u] = m.k[at_row][d0 + u * kNext];
      const float qd = m.q[at_row][d0 + u * kNext];
#pragma unroll
      for (int e = 0; e < 4; ++e) pa[e] = fmaf(S[u][e], kd[u], pa[e]), pc[e] = fmaf(S[u][e], qd, pc[e]);
    }
#pragma unroll
    for (int x = C4; x < 64; x <<= 1)
#pragma unroll
      for (int e = 0; e < 4; ++e) pa[e] += __shfl_xor(pa[e], x, 64), pc[e] += __shfl_xor(pc[e], x, 64);
    if constexpr (kWaves > 1) {
      if (lane < C4) {
        *reinterpret_cast<f32x4*>(&m.dots[at_row][wave][0][4 * c4]) = pa;
        *reinterpret_cast<f32x4*>(&m.dots[at_row][wave][1][4 * c4]) = pc;
      }
      __syncthreads();
      pa = pc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int x = 0; x < kWaves; ++x) pa += *reinterpret_cast<const f32x4*>(&m.dots[at_row][x][0][4 * c4]);
      if (d0 == 0) {
#pragma unroll
        for (int x = 0; x < kWaves; ++x) pc += *reinterpret_cast<const f32x4*>(&m.dots[at_row][x][1][4 * c4]);
      }
    }
    f32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = beta * (v[e] - decay * (pa[e] * ik)) * ik;       // (with the key's length: what multiplies the raw key)
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) S[u][e] = fmaf(decay, S[u][e], kd[u] * w[e]);
    if (d0 == 0) {
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = iq * fmaf(w[e], kq, decay * pc[e]);
      *reinterpret_cast<f32x4_any*>(static_cast<float*>(a.out) + (static_cast<int64_t>(r0 + i) * H + h) * Dv + col0 + 4 * c4) = o;
    }
  }
  if (st != nullptr) {
#pragma unroll
    for (int u = 0; u < U; ++u) *reinterpret_cast<f32x4*>(st + u * kNext * Dv + at) = S[u];
  }
}

// Portions of 1 to max_rows rows in a launch of their own.  grid = (heads, value columns in slices of 4 C4, sequences).
template <int D, int C4, int NT>
__global__ __launch_bounds__(NT) void delta_short_kernel(hymeta_delta_rule_args a, int max_rows) {
  __shared__ ShortScratch<D, NT> m;
  const int s = blockIdx.z, r0 = a.query_start_loc[s], rows = a.query_start_loc[s + 1] - r0;
  if (rows <= 0 || rows > max_rows) return;
  delta_short_rows<D, C4, NT>(a, threadIdx.x, blockIdx.x, s, r0, rows, blockIdx.y * 4 * C4, m);
}

// ------------------------------------------------------------------------------------------------
// bf16 portions in chunks of 64 rows on the matrix cores.  With S the state before the chunk, i and j rows of it, c_i the
// running sums of its log2 decays (c the whole chunk's), k' and q' the unit vectors:
//   (I + A) U = diag(beta) V - diag(beta_i 2^(c_i)) K' S,     A_ij = beta_i 2^(c_i - c_j) (k'_i . k'_j)   for j < i, else 0
//   O = diag(2^(c_i)) Q' S + P U,                             P_ij = 2^(c_i - c_j) (q'_i . k'_j)          for j <= i, else 0
//   S_new = 2^c S + sum_j 2^(c - c_j) k'_j u_j^T
// T = (I + A)^-1 and P depend on the chunk alone: a first launch computes them for all chunks and heads side by side; a
// second one carries the state through a sequence's chunks.  The keys and queries enter every product as the bf16 rows they
// are, their lengths as fp32 factors of the rows around the product; what enters a product from fp32 (T, P, the state, U
// and the right-hand side) goes in as hi + lo bf16 parts, so that it keeps 16 bits of mantissa.
//
// Chunks are numbered so that no count has to be known ahead: chunk c of sequence s is number
// query_start_loc[s] / 64 + s + c, at most num_tokens / 64 + num_seqs of them.
// ------------------------------------------------------------------------------------------------
typedef float f32x4v __attribute__((ext_vector_type(4)));
constexpr int kChunk = HYMETA_DELTA_CHUNK;
// Workgroups with slices of 32 value columns up to which the second launch runs slices of 16 whose waves share a chunk's rows
// (delta_chunk_narrow_kernel), about 2 us a chunk against 2.6 where a wave takes all rows of its columns: one prompt of 8192
// rows with 28 heads of 128 x 128 (112 workgroups) 327 us against 388, with 16 heads 216 against 345, of 96 x 96 190 against 319, of 32 x 32
// 157 against 248.  They also double the
// workgroups of the sequences without a chunk, which end at once but take about 0.65 ns each to come and go, and save about 0.6
// us a chunk of 64 rows: not where those are more than 10 per row of the longest portion.
// Workgroups with slices of 64 columns up to which the other kernel takes those: its images leave room for one workgroup on a
// compute unit, where four waves take 2.6 us a chunk and eight (slices of 128) 4.4.  28 heads: three portions of 2700 (168)
// 177 us, 301 before; five of 1801 (280, in slices of 128) 182, 280 before (154 with some sequences'
// slices of 64: delta_chunk_mixed_kernel).
// All count the portions that the step's rows are worth (long_portions): single rows leave the chip to a long prompt.
constexpr int kFewGroups = 128, kIdleGroupsPerRow = 10, kManyGroups = 256;
// Whether portions too short for a chunk have a launch of their own and do not run in the chunks' first one, where they cost no
// launch (about 4 us) and stand beside the chunks' work, but go through a head's value columns 64 at a time with the registers of
// that kernel.  `shorts`: the (head, short portion) pairs that there may be.  Us in the first launch / in their own:
//   28 heads of 128 x 128: 40 rows beside 15 single ones (420 pairs) 24.6 / 27.9, beside 63 56.7 / 55.0, beside 127 105 / 92; 2048
//   beside 63 127 / 131, beside 255 330 / 294; 16 heads, 2048 beside 255 (4080) 184 / 196: with few rows in chunks from 1000 pairs on,
//   else from 4096.
//   28 heads of 64 x 128: 40 beside 63 29.7 / 36.8, beside 255 85 / 97, 2048 beside 255 179 / 176: single rows stay.
//   60 portions of 7 rows beside 40: 64 x 128 79 / 52, 128 x 128 98 / 80: where the longest fits a chunk and the others have two rows
//   each, apart.
//   Three or four times through the columns, four portions of 600 beside three of 5: 8 heads of 128 x 256 72 / 55, 16 of 32 x 96 55 / 49;
//   where none are to be expected, the launch is saved: 16 heads of 96 x 96, 64 rows 18.9 -> 16.0.
inline bool short_apart(const hymeta_delta_rule_args& a, int64_t shorts) {
  const int passes = a.v_dim / (a.v_dim % 64 == 0 ? 64 : 32);
  if (shorts == 0) return false;
  if (passes > 2 || (a.head_dim > 64 && shorts > 4096)) return true;
  const int64_t chunks = static_cast<int64_t>(a.num_heads) * (a.num_tokens / kChunk);
  if (a.head_dim > 64 && shorts > 1000 && 10 * chunks < shorts) return true;
  return shorts > 256 && a.max_query_len <= kChunk && a.num_tokens - a.max_query_len >= 2 * (a.num_seqs - 1);
}
constexpr int kChunkMinRows = 8;            // shorter portions go token by token
constexpr int kMat = kChunk * kChunk;
// Where the second launch reads 64 x 64 matrices (or the chunk's keys) as matrix operands, they lie in the operand's own
// order: per 16 rows and 32 columns the 64 lanes' 8 elements one after the other, so that a wave's load is 1 KB in a row.
__device__ __forceinline__ int operand_at(int row, int col, int cols) {       // (col in whole fours)
  return ((row >> 4) * (cols >> 5) + (col >> 5)) * 512 + (((col >> 3) & 3) * 16 + (row & 15)) * 8 + (col & 7);
}
// a chunk's and head's place in the workspace: T hi, T lo, P hi, P lo (bf16, operand order), then per row beta,
// beta 2^(c_i) / |k|, q_scale 2^(c_i) / |q|, 2^(c - c_j) / |k|, then 2^c
struct ChunkPlace {
  uint16_t t[2][kMat], p[2][kMat];
  float beta[kChunk], rhs[kChunk], read[kChunk], write[kChunk];
  float total, pad[3];
};
static_assert(sizeof(ChunkPlace) % 16 == 0, "16-byte loads of every place");

__device__ __forceinline__ f32x4v mfma16(bf16x8 a, bf16x8 b, f32x4v c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ bf16x8 frag(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// Inclusive sums over a wave's lanes in double precision (lane_sums, a word at a time).
__device__ __forceinline__ double lane_sums64(double x) {
  auto add = [&](auto ctrl, auto rows_mask) {
    const uint64_t bits = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(bits), decltype(ctrl)::value, decltype(rows_mask)::value, 0xf, false);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(bits >> 32), decltype(ctrl)::value, decltype(rows_mask)::value, 0xf, false);
    x += __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
  };
  add(Const<0x111>{}, Const<0xf>{}), add(Const<0x112>{}, Const<0xf>{}), add(Const<0x114>{}, Const<0xf>{}), add(Const<0x118>{}, Const<0xf>{});
  add(Const<0x142>{}, Const<0xa>{}), add(Const<0x143>{}, Const<0xc>{});
  return x;
}

// four fp32 values as hi + lo bf16 parts
__device__ __forceinline__ void split4(const float* v, u32x2& hi, u32x2& lo) {
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    hi[u] = pack_bf16x2(v[2 * u], v[2 * u + 1]);
    lo[u] = pack_bf16x2(v[2 * u] - lo_bf(hi[u]), v[2 * u + 1] - hi_bf(hi[u]));
  }
}

// Workspace: the chunks' places ([chunk][head]), then (narrow slices) per chunk and query / key head the chunk's keys [64][D],
// queries [64][D] and transposed keys [D][64], bf16 in operand order.
__host__ __device__ inline size_t rows_at(int64_t chunks, int heads) { return static_cast<size_t>(chunks) * heads * sizeof(ChunkPlace); }

// grid = (chunk numbers, heads), 4 waves with 16 rows of the chunk each.
// Bound by vector instructions and the latency of its phases: A stays in the registers that the elimination multiplies it from, and only
// a wave's diagonal block passes through LDS, to the wave itself, so that six workgroups are on a compute unit (four with all of A in
// LDS); the sequence is found in one round trip.  28 heads, five portions of 1801 rows 53 -> 46 us.
// Short: portions shorter than kChunkMinRows go row by row here, all of a head's value columns in turn, at the price of registers.
template <int D, bool Pack, bool Short>
__global__ __launch_bounds__(256, Pack ? 3 : Short ? 4 : 6) void delta_chunk_solve_kernel(hymeta_delta_rule_args a, int64_t chunks) {
  constexpr int PK = D + 8, PF = kChunk + 4, PD = 20;
  // (the keys and T share their place where nothing asks for the keys again: six workgroups to a compute unit)
  constexpr int kKeyBytes = kChunk * PK * 2, kMatrixBytes = kChunk * PF * 4;
  __shared__ __attribute__((aligned(16))) char s_keys[Pack ? kKeyBytes + kMatrixBytes : kKeyBytes > kMatrixBytes ? kKeyBytes : kMatrixBytes];
  uint16_t* sk = reinterpret_cast<uint16_t*>(s_keys);
  float* sT = reinterpret_cast<float*>(s_keys + (Pack ? kKeyBytes : 0));
  __shared__ __attribute__((aligned(16))) float s_diag[4][16 * PD];                // a wave's diagonal block of A
  __shared__ float s_hi[kChunk], s_lo[kChunk], s_beta[kChunk], s_ik[kChunk], s_iq[kChunk];
  // the sequence: the last one whose first number is not past this one, by 64 probes a round trip, each time `step` apart (64 at a time
  // one behind the other: 2048 rows beside 1023 single ones 498 -> 469 us, beside 2047 972 -> 830)
  const int number = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  int s = 0, r0 = 0, rows = 0;
  for (int end = a.num_seqs;;) {
    const int step = (end - s + 63) / 64, probe = s + lane * step, start = a.query_start_loc[min(probe, a.num_seqs)];
    const int upto = __popcll(__ballot(probe < end && start / kChunk + probe <= number));
    if (upto == 0) return;
    s += (upto - 1) * step;
    if (step == 1) {
      r0 = __builtin_amdgcn_readlane(start, upto - 1);
      rows = (upto < 64 ? __builtin_amdgcn_readlane(start, upto) : a.query_start_loc[s + 1]) - r0;
      break;
    }
    end = min(s + step, end);
  }
  const int c0 = (number - (r0 / kChunk + s)) * kChunk;
  if (c0 >= rows) return;
  if (rows < kChunkMinRows) {
    if constexpr (Short) {
      static_assert(sizeof(ShortScratch<D, 256>) <= sizeof(s_keys), "the scratch lies where the keys would");
      ShortScratch<D, 256>& m = *reinterpret_cast<ShortScratch<D, 256>*>(s_keys);
      if (a.v_dim % 64 == 0) {
        for (int col0 = 0; col0 < a.v_dim; col0 += 64) delta_short_rows<D, 16, 256>(a, tid, blockIdx.y, s, r0, rows, col0, m), __syncthreads();
      } else {
        for (int col0 = 0; col0 < a.v_dim; col0 += 32) delta_short_rows<D, 8, 256>(a, tid, blockIdx.y, s, r0, rows, col0, m), __syncthreads();
      }
    }
    return;
  }
  const int nrow = min(kChunk, rows - c0), h = blockIdx.y, H = a.num_heads, group = H / a.num_qk_heads, g = h / group;
  const int64_t t0 = r0 + c0;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15, g4 = lane >> 4;
  const int i = 16 * wave + n;                          // this lane's row of the chunk
  ChunkPlace* place = static_cast<ChunkPlace*>(a.workspace) + static_cast<int64_t>(number) * H + h;
  u32x4 kf[D / 32], qf[D / 32];
  {
    const uint16_t* kr = static_cast<const uint16_t*>(a.k) + (t0 + i) * a.k_stride_t + static_cast<int64_t>(g) * D + 8 * g4;
    const uint16_t* qr = static_cast<const uint16_t*>(a.q) + (t0 + i) * a.q_stride_t + static_cast<int64_t>(g) * D + 8 * g4;
#pragma unroll
    for (int sd = 0; sd < D / 32; ++sd) {
      kf[sd] = qf[sd] = u32x4{0u, 0u, 0u, 0u};
      if (i < nrow) kf[sd] = ld16g(kr + 32 * sd), qf[sd] = ld16g(qr + 32 * sd);
    }
  }
  if (wave == 0) {
    // running sums in double precision, kept as two floats: a difference of two sums is exact to its own rounding however
    // large the sums are
    const bool on = lane < nrow;
    const double cum = lane_sums64(on ? static_cast<double>(fmaxf(a.log2_decay[(t0 + lane) * H + h], kMinLog2)) : 0.0);
    s_hi[lane] = static_cast<float>(cum);
    s_lo[lane] = static_cast<float>(cum - static_cast<double>(s_hi[lane]));
    s_beta[lane] = on ? sigmoid_exact(bf2f(static_cast<const uint16_t*>(a.beta_logit)[(t0 + lane) * a.beta_stride_t + h])) : 0.f;
  }
  float kk = 0.f, qq = 0.f;
#pragma unroll
  for (int sd = 0; sd < D / 32; ++sd) {
    st16(&sk[i * PK + 32 * sd + 8 * g4], kf[sd]);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      kk = fmaf(lo_bf(kf[sd][u]), lo_bf(kf[sd][u]), fmaf(hi_bf(kf[sd][u]), hi_bf(kf[sd][u]), kk));
      qq = fmaf(lo_bf(qf[sd][u]), lo_bf(qf[sd][u]), fmaf(hi_bf(qf[sd][u]), hi_bf(qf[sd][u]), qq));
    }
  }
  kk += __shfl_xor(kk, 16, 64), kk += __shfl_xor(kk, 32, 64);
  qq += __shfl_xor(qq, 16, 64), qq += __shfl_xor(qq, 32, 64);
  if (g4 == 0) {
    s_ik[i] = 1.f / sqrtf(kk + a.unit_eps);
    s_iq[i] = a.q_scale / sqrtf(qq + a.unit_eps);
  }
  __syncthreads();
  // A and P in blocks of 16 x 16, transposed products: a lane gets four consecutive j of its row i
  const float ch = s_hi[i], cl = s_lo[i], bk = s_beta[i] * s_ik[i], iq = s_iq[i];
  f32x4v A[4];                                          // this lane's row, columns 16 jb + 4 g4 + r
#pragma unroll
  for (int jb = 0; jb < 4; ++jb) {
    float pv[4] = {0.f, 0.f, 0.f, 0.f};
    A[jb] = f32x4v{0.f, 0.f, 0.f, 0.f};
    if (jb <= wave) {
      f32x4v xk = f32x4v{0.f, 0.f, 0.f, 0.f}, xq = xk;
#pragma unroll
      for (int sd = 0; sd < D / 32; ++sd) {
        const bf16x8 kj = frag(ld16(&sk[(16 * jb + n) * PK + 32 * sd + 8 * g4]));
        xk = mfma16(kj, frag(kf[sd]), xk);
        xq = mfma16(kj, frag(qf[sd]), xq);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = 16 * jb + 4 * g4 + r;
        if (j > i) continue;
        const float w = __builtin_amdgcn_exp2f((ch - s_hi[j]) + (cl - s_lo[j])) * s_ik[j];
        if (j < i) A[jb][r] = bk * w * xk[r];
        pv[r] = iq * w * xq[r];
      }
      if (jb == wave) *reinterpret_cast<f32x4v*>(&s_diag[wave][n * PD + 4 * g4]) = A[jb];
    }
    u32x2 hi, lo;
    split4(pv, hi, lo);
    if (!Pack && wave < 2 && jb >= 2) continue;         // (rows up to 31, columns from 32 on: narrow slices alone multiply these zeros)
    *reinterpret_cast<u32x2*>(&place->p[0][operand_at(i, 16 * jb + 4 * g4, kChunk)]) = hi;
    *reinterpret_cast<u32x2*>(&place->p[1][operand_at(i, 16 * jb + 4 * g4, kChunk)]) = lo;
  }
  // T: the diagonal blocks by forward substitution, a column per lane (the four groups of lanes do the same), each by the wave
  // that has it
  {
    const float* diag = s_diag[wave];
    float x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      f32x4v row[4];
#pragma unroll
      for (int j = 0; j < (r + 3) / 4; ++j) row[j] = *reinterpret_cast<const f32x4v*>(&diag[r * PD + 4 * j]);
      float v = r == n ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < r; ++j) v = fmaf(-row[j >> 2][j & 3], x[j], v);
      x[r] = v;
      asm volatile("" : "+v"(x[r]));                    // (here, not behind the barrier with all of A's rows in registers)
    }
    __syncthreads();                                    // nobody reads the keys where T comes to lie
    if (g4 == 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) sT[(16 * wave + r) * PF + 16 * wave + n] = x[r];
    }
  }
  __syncthreads();
  // ... then the blocks below them, a diagonal at a time: T_ij = -T_ii sum_{j <= l < i} A_il T_lj, in fp32 on the matrix
  // cores (step e of a product takes the inner indices 4 g4 + e, so that the first product's result is the second's operand
  // as it lies in the registers)
#pragma unroll
  for (int below = 1; below < 4; ++below) {
    if (wave >= below) {
      const int jb = wave - below;
      f32x4v m = f32x4v{0.f, 0.f, 0.f, 0.f}, x = m;
#pragma unroll
      for (int lb = 0; lb < 3; ++lb) {
        if (lb < jb || lb >= wave) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) m = __builtin_amdgcn_mfma_f32_16x16x4f32(A[lb][e], sT[(16 * lb + 4 * g4 + e) * PF + 16 * jb + n], m, 0, 0, 0);
      }
      const f32x4v ti = *reinterpret_cast<const f32x4v*>(&sT[i * PF + 16 * wave + 4 * g4]);
#pragma unroll
      for (int e = 0; e < 4; ++e) x = __builtin_amdgcn_mfma_f32_16x16x4f32(ti[e], m[e], x, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) sT[(16 * wave + 4 * g4 + r) * PF + 16 * jb + n] = -x[r];
    }
    __syncthreads();
  }
  {
    const int row = tid >> 2, jb = tid & 3, rb = row >> 4;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (!Pack && rb < 2 && jb >= 2) break;
      float v[4] = {0.f, 0.f, 0.f, 0.f};
      if (jb <= rb) {
        const f32x4v tv = *reinterpret_cast<const f32x4v*>(&sT[row * PF + 16 * jb + 4 * u]);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = tv[e];
      }
      u32x2 hi, lo;
      split4(v, hi, lo);
      *reinterpret_cast<u32x2*>(&place->t[0][operand_at(row, 16 * jb + 4 * u, kChunk)]) = hi;
      *reinterpret_cast<u32x2*>(&place->t[1][operand_at(row, 16 * jb + 4 * u, kChunk)]) = lo;
    }
  }
  if (Pack && h % group == 0) {
    uint16_t* kr = reinterpret_cast<uint16_t*>(static_cast<char*>(a.workspace) + rows_at(chunks, H)) +
                   (static_cast<int64_t>(number) * a.num_qk_heads + g) * 3 * D * kChunk;
    uint16_t *qr = kr + D * kChunk, *kt = qr + D * kChunk;
#pragma unroll
    for (int sd = 0; sd < D / 32; ++sd) {
      st16(kr + operand_at(i, 32 * sd + 8 * g4, D), kf[sd]);
      st16(qr + operand_at(i, 32 * sd + 8 * g4, D), qf[sd]);
    }
    for (int idx = tid; idx < D * (kChunk / 8); idx += 256) {
      const int d = idx % D, tc = idx / D;
      u32x4 w;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        w[u] = static_cast<uint32_t>(sk[(8 * tc + 2 * u) * PK + d]) | (static_cast<uint32_t>(sk[(8 * tc + 2 * u + 1) * PK + d]) << 16);
      st16(kt + operand_at(d, 8 * tc, kChunk), w);
    }
  }
  if (wave == 0) {
    const float th = s_hi[kChunk - 1], tl = s_lo[kChunk - 1];          // (rows past the portion add 0)
    const float here = __builtin_amdgcn_exp2f(s_hi[lane] + s_lo[lane]);
    place->beta[lane] = s_beta[lane];
    place->rhs[lane] = s_beta[lane] * s_ik[lane] * here;
    place->read[lane] = s_iq[lane] * here;
    place->write[lane] = lane < nrow ? s_ik[lane] * __builtin_amdgcn_exp2f((th - s_hi[lane]) + (tl - s_lo[lane])) : 0.f;
    if (lane == 0) place->total = __builtin_amdgcn_exp2f(th + tl);
  }
}

// grid = (heads, sequences, value columns in slices of 16), 4 waves.  The state slice stays fp32 in registers in blocks of
// 16 x 16 dealt over the waves (a lane holds 4 consecutive rows d of one column); its bf16 parts, the right-hand side and
// U pass through LDS with the reduced index consecutive; everything a chunk brings comes from memory in the matrix
// operands' own layout, loaded two chunks ahead (the loads of two chunks are in flight, each in registers of its own).  Rows past the portion read its last row (beta, and with it what they would
// write, is 0 there), and the last chunk fetches itself once more, so that no load stands under a condition.
template <int D>
__global__ __launch_bounds__(256) void delta_chunk_narrow_kernel(hymeta_delta_rule_args a, int64_t chunks) {
  constexpr int SV = 16, PK = D + 8, PT = kChunk + 8, DB = D / 16, NBW = (DB + 3) / 4;
  // (what is left over of the deal, with heads of 32 and 96: the last block again, whose owner alone writes it)
  auto block_of = [](int wave, int ib) __attribute__((always_inline)) { return DB % 4 == 0 ? wave + 4 * ib : min(wave + 4 * ib, DB - 1); };
  auto owned = [](int wave, int ib) __attribute__((always_inline)) { return DB % 4 == 0 || wave + 4 * ib < DB; };
  __shared__ __attribute__((aligned(16))) uint16_t sst[2][SV * PK];                                      // state, [c][d]
  __shared__ __attribute__((aligned(16))) uint16_t srt[2][SV * PT], su[2][SV * PT], sw[2][SV * PT];      // [c][row]
  const int h = blockIdx.x, s = blockIdx.y, vs = blockIdx.z;
  const int r0 = a.query_start_loc[s], rows = a.query_start_loc[s + 1] - r0;
  if (rows < kChunkMinRows) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, g4 = lane >> 4;
  const int H = a.num_heads, G = a.num_qk_heads, Dv = a.v_dim, g = h / (H / G);
  const int slot = a.slot_idx[s];
  float* st = slot >= 0 ? a.state + ((static_cast<int64_t>(slot) * H + h) * D) * Dv + vs * SV : nullptr;
  const bool carry = st != nullptr && a.context_lens[s] > 0;
  f32x4v S[NBW];
#pragma unroll
  for (int ib = 0; ib < NBW; ++ib) {
    const int db = block_of(wave, ib);
#pragma unroll
    for (int r = 0; r < 4; ++r) S[ib][r] = carry ? st[static_cast<int64_t>(16 * db + 4 * g4 + r) * Dv + n] : 0.f;
  }
  auto state_to_lds = [&]() {
#pragma unroll
    for (int ib = 0; ib < NBW; ++ib) {
      if (!owned(wave, ib)) continue;
      const int db = block_of(wave, ib);
      const float v[4] = {S[ib][0], S[ib][1], S[ib][2], S[ib][3]};
      u32x2 hi, lo;
      split4(v, hi, lo);
      *reinterpret_cast<u32x2*>(&sst[0][n * PK + 16 * db + 4 * g4]) = hi;
      *reinterpret_cast<u32x2*>(&sst[1][n * PK + 16 * db + 4 * g4]) = lo;
    }
  };
  state_to_lds();
  const uint16_t* vp = static_cast<const uint16_t*>(a.v) + static_cast<int64_t>(h) * Dv + vs * SV + n;
  const int64_t first = r0 / kChunk + s;
  const ChunkPlace* places = static_cast<const ChunkPlace*>(a.workspace) + first * H + h;
  const uint16_t* packed = reinterpret_cast<const uint16_t*>(static_cast<const char*>(a.workspace) + rows_at(chunks, H)) +
                           (first * G + g) * 3 * D * kChunk + 8 * lane;          // keys, queries, transposed keys of the chunks
  const int iq = 16 * wave + 4 * g4;        // the first of the four rows of this lane's results
  // what a chunk brings: row fragments of the keys, queries, T and P, the transposed keys of this wave's state blocks, values
  struct Chunk {
    u32x4 kf[D / 32], qf[D / 32], tf[2][2], pf[2][2], wf[NBW][2];
    uint16_t vv[4];
    f32x4v beta, rhs, read, write;
    float total;
  };
  auto fetch_rows = [&](Chunk& m, int c) {
    const int last = rows - 1 - c * kChunk;
    const int64_t t0 = r0 + static_cast<int64_t>(c) * kChunk;
    const uint16_t* kr = packed + static_cast<int64_t>(c) * G * 3 * D * kChunk + wave * (D / 32) * 512;
#pragma unroll
    for (int sd = 0; sd < D / 32; ++sd) m.kf[sd] = ld16g(kr + 512 * sd), m.qf[sd] = ld16g(kr + D * kChunk + 512 * sd);
#pragma unroll
    for (int r = 0; r < 4; ++r) m.vv[r] = vp[(t0 + min(iq + r, last)) * a.v_stride_t];
  };
  auto fetch_t = [&](Chunk& m, int c) {
    const ChunkPlace* p = places + static_cast<int64_t>(c) * H;
#pragma unroll
    for (int part = 0; part < 2; ++part)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) m.tf[part][kk] = ld16g(&p->t[part][(2 * wave + kk) * 512 + 8 * lane]);
    m.beta = *reinterpret_cast<const f32x4v*>(&p->beta[iq]);
    m.rhs = *reinterpret_cast<const f32x4v*>(&p->rhs[iq]);
    m.read = *reinterpret_cast<const f32x4v*>(&p->read[iq]);
    m.write = *reinterpret_cast<const f32x4v*>(&p->write[iq]);
  };
  auto fetch_p = [&](Chunk& m, int c) {
    const ChunkPlace* p = places + static_cast<int64_t>(c) * H;
#pragma unroll
    for (int part = 0; part < 2; ++part)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) m.pf[part][kk] = ld16g(&p->p[part][(2 * wave + kk) * 512 + 8 * lane]);
  };
  auto fetch_transposed = [&](Chunk& m, int c) {
    const uint16_t* kt = packed + (static_cast<int64_t>(c) * G * 3 + 2) * D * kChunk;
    m.total = places[static_cast<int64_t>(c) * H].total;
#pragma unroll
    for (int ib = 0; ib < NBW; ++ib) {
      const int db = block_of(wave, ib);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) m.wf[ib][kk] = ld16g(kt + (2 * db + kk) * 512);
    }
  };
  float* out = static_cast<float*>(a.out) + static_cast<int64_t>(r0) * H * Dv + static_cast<int64_t>(h) * Dv + vs * SV + n;
  const int num = (rows + kChunk - 1) / kChunk;
  auto advance = [&](Chunk& m, int c, auto full) {         // full: a whole chunk (every row is the portion's)
    const int next = min(c + 2, num - 1);
    __syncthreads();                        // the state's parts are in place
    f32x4v x, y;
    {
      x = y = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int sd = 0; sd < D / 32; ++sd) {
        const bf16x8 sh = frag(ld16(&sst[0][n * PK + 32 * sd + 8 * g4]));
        const bf16x8 sl = frag(ld16(&sst[1][n * PK + 32 * sd + 8 * g4]));
        x = mfma16(frag(m.kf[sd]), sh, x);
        y = mfma16(frag(m.qf[sd]), sh, y);
        x = mfma16(frag(m.kf[sd]), sl, x);
        y = mfma16(frag(m.qf[sd]), sl, y);
      }
    }
    {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = m.beta[r] * bf2f(m.vv[r]) - m.rhs[r] * x[r];
        y[r] *= m.read[r];
      }
      u32x2 hi, lo;
      split4(v, hi, lo);
      *reinterpret_cast<u32x2*>(&srt[0][n * PT + iq]) = hi;
      *reinterpret_cast<u32x2*>(&srt[1][n * PT + iq]) = lo;
    }
    fetch_rows(m, next);
    __syncthreads();
    {
      f32x4v u = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const bf16x8 rh = frag(ld16(&srt[0][n * PT + 32 * kk + 8 * g4]));
        const bf16x8 rl = frag(ld16(&srt[1][n * PT + 32 * kk + 8 * g4]));
        u = mfma16(frag(m.tf[0][kk]), rh, u);
        u = mfma16(frag(m.tf[0][kk]), rl, u);
        u = mfma16(frag(m.tf[1][kk]), rh, u);
      }
      float v[4] = {u[0], u[1], u[2], u[3]};
      u32x2 hi, lo;
      split4(v, hi, lo);
      *reinterpret_cast<u32x2*>(&su[0][n * PT + iq]) = hi;
      *reinterpret_cast<u32x2*>(&su[1][n * PT + iq]) = lo;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] *= m.write[r];
      split4(v, hi, lo);
      *reinterpret_cast<u32x2*>(&sw[0][n * PT + iq]) = hi;
      *reinterpret_cast<u32x2*>(&sw[1][n * PT + iq]) = lo;
    }
    fetch_t(m, next);
    __syncthreads();
#pragma unroll
    for (int ib = 0; ib < NBW; ++ib) {
      f32x4v acc = S[ib] * m.total;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        acc = mfma16(frag(m.wf[ib][kk]), frag(ld16(&sw[0][n * PT + 32 * kk + 8 * g4])), acc);
        acc = mfma16(frag(m.wf[ib][kk]), frag(ld16(&sw[1][n * PT + 32 * kk + 8 * g4])), acc);
      }
      S[ib] = acc;
    }
    fetch_transposed(m, next);
    state_to_lds();                         // (its last readers passed the barrier before)
    {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const bf16x8 uh = frag(ld16(&su[0][n * PT + 32 * kk + 8 * g4]));
        const bf16x8 ul = frag(ld16(&su[1][n * PT + 32 * kk + 8 * g4]));
        y = mfma16(frag(m.pf[0][kk]), uh, y);
        y = mfma16(frag(m.pf[0][kk]), ul, y);
        y = mfma16(frag(m.pf[1][kk]), uh, y);
      }
    }
    fetch_p(m, next);
    const int live = rows - c * kChunk - iq;            // rows of this lane's four that are the portion's
    float* to = out + (static_cast<int64_t>(c) * kChunk + iq) * H * Dv;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (decltype(full)::value || r < live) {
        to[static_cast<int64_t>(r) * H * Dv ] = y[r];
      }
  };
  Chunk even, odd;
  auto fetch = [&](Chunk& m, int c) {
    fetch_rows(m, c);
    fetch_t(m, c);
    fetch_transposed(m, c);
    fetch_p(m, c);
  };
  fetch(even, 0);
  fetch(odd, min(1, num - 1));
  // (the loop's body has no branch: loads under one, or a chunk that might not run, would make the waits in front of the
  // matrix products wait for the loads of the chunks behind as well)
  int c = 0;
  for (; c + 2 < num; c += 2) {
    advance(even, c, std::true_type{});
    advance(odd, c + 1, std::true_type{});
  }
  advance(even, c, std::false_type{});
  if (c + 1 < num) advance(odd, c + 1, std::false_type{});
  if (st != nullptr) {
#pragma unroll
    for (int ib = 0; ib < NBW; ++ib) {
      if (!owned(wave, ib)) continue;
      const int db = block_of(wave, ib);
#pragma unroll
      for (int r = 0; r < 4; ++r) st[static_cast<int64_t>(16 * db + 4 * g4 + r) * Dv + n] = S[ib][r];
    }
  }
}

// grid = (heads, sequences, value columns in slices of 16 NW), NW waves of 16 columns.  Every step of a chunk keeps to
// its columns, so a wave runs alone from barrier to barrier: the state, the right-hand side and U are accumulators (a lane
// holds four consecutive rows of a column), and a pair of such blocks IS the operand of the next product.  Which row of 32 a
// block's row m stands for is free: block 0 of a pair takes 8 (m / 4) + m % 4, block 1 the ones 4 further on, so that a lane's
// eight values of a pair are consecutive and the other operand is the plain one, a 16-byte read.  What a chunk brings is copied
// to LDS a chunk ahead, once for all columns, the keys' and queries' rows as they lie in memory; transposed keys are read
// transposed.  A chunk's outputs are stored in the next one, so that the wait for the copies does not wait for stores just
// issued.
// Bound by what a wave can issue: 132 matrix and 450 vector instructions a chunk of 64 rows x 128 keys, on a SIMD with one wave
// or two.  Left to itself the compiler reads a fragment in front of its product and waits (3.9 us a chunk with four waves), so
// the step is laid out by hand: fragments six ahead, vector work and copies dealt between the products.  LDS is busy about 60 %
// of the time with eight waves, as each reads the chunk's 72 KB; waves of 32 columns would halve that, but their state and
// operands do not fit 256 registers (5.5 us a chunk instead of 4.4).  Earlier forms: operands packed by the first launch, in
// halves of 8 bytes, no fragment ahead: 6.7 us.
//
// LDS: blocks of 16 rows x 32 columns, 1 KB, in operand order but for the rows: chunk (16 bytes) ch of the block's row m lies
// at 16 ch + (m ^ 4 ch), so that the transposed reads of 4 rows x 4 chunks spread over the banks too.
template <int D, int NW>
struct WideImage {                                          // keys, queries | T hi, lo, P hi, lo | beta, rhs, read, write | values
  static constexpr bool kDirect = NW == 2;                  // values of any alignment, read by the lanes that want them
  static constexpr int kRowsBytes = kChunk * D * 2, kMatBytes = 6 * 1024, kMatsAt = 2 * kRowsBytes, kScaleAt = kMatsAt + 4 * kMatBytes, kValuesAt = kScaleAt + 1024;
  static constexpr int kBytes = kValuesAt + (kDirect ? 0 : kChunk * 32 * NW);
};
// Columns 16 NW vs .. of head h of sequence s, by NW waves (short_too: portions shorter than kChunkMinRows as well, row by row).
template <int D, int NW>
__device__ __forceinline__ void delta_chunk_wide(const hymeta_delta_rule_args& a, int h, int s, int vs, char* lds, bool short_too) {
  typedef WideImage<D, NW> Image;
  constexpr bool Direct = Image::kDirect;
  constexpr int SD = D / 32, DB = D / 16, VC = 2 * NW, kRowsBytes = Image::kRowsBytes, kMatBytes = Image::kMatBytes;
  constexpr int kMatsAt = Image::kMatsAt, kScaleAt = Image::kScaleAt, kValuesAt = Image::kValuesAt, kImage = Image::kBytes;
  static_assert(NW == 2 || NW == 4 || NW == 8, "the copies deal evenly over the waves");
  typedef ChunkOrder<VC> VOrder;
  typedef f32x4v f32x4_any __attribute__((aligned(4)));
  const int r0 = a.query_start_loc[s], rows = a.query_start_loc[s + 1] - r0;
  if (rows < kChunkMinRows) {
    constexpr int NT = NW == 2 ? 128 : 256, kCols = NW == 2 ? 32 : 64;          // (eight waves: 64 columns by four each)
    if (!short_too || rows <= 0) return;
    ShortScratch<D, NT>* m = reinterpret_cast<ShortScratch<D, NT>*>(lds);
    const int part = threadIdx.x / NT;
    delta_short_rows<D, kCols / 4, NT>(a, threadIdx.x % NT, h, s, r0, rows, vs * 16 * NW + part * kCols, m[part]);
    return;
  }
  const int lane = threadIdx.x & 63, n = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = a.num_heads, Dv = a.v_dim, g = h / (H / a.num_qk_heads), col0 = (vs * NW + wave) * 16;
  const ChunkPlace* places = static_cast<const ChunkPlace*>(a.workspace) + static_cast<int64_t>(r0 / kChunk + s) * H + h;
  const int num = (rows + kChunk - 1) / kChunk;
  auto row_of = [](int ib, int m) __attribute__((always_inline)) { return 32 * (ib >> 1) + 4 * (ib & 1) + 8 * (m >> 2) + (m & 3); };
  // ---- copies: number i of a wave's; chunk c's rows past the portion's last one read that again
  constexpr int kRowCopies = 8 * SD / NW, kMatCopies = 24 / NW, kCopies = kRowCopies + kMatCopies + (Direct ? 0 : 2) + 1;
  const int ch = lane >> 4, m = (lane & 15) ^ (4 * ch);     // this lane's place in a block: row m, chunk ch
  const uint32_t mat_lane = (m >> 3) * 2048 + (8 * ((m >> 2) & 1) + (m & 3)) * 16 + ch * 256;
  const int k_stride = static_cast<int>(a.k_stride_t), q_stride = static_cast<int>(a.q_stride_t), v_stride = static_cast<int>(a.v_stride_t);
  struct Source { const char *k, *q, *v, *place; int last; };
  auto source = [&](int c) __attribute__((always_inline)) {
    const int64_t t0 = r0 + static_cast<int64_t>(c) * kChunk;
    return Source{reinterpret_cast<const char*>(static_cast<const uint16_t*>(a.k) + t0 * a.k_stride_t + static_cast<int64_t>(g) * D),
                  reinterpret_cast<const char*>(static_cast<const uint16_t*>(a.q) + t0 * a.q_stride_t + static_cast<int64_t>(g) * D),
                  reinterpret_cast<const char*>(static_cast<const uint16_t*>(a.v) + t0 * a.v_stride_t + static_cast<int64_t>(h) * Dv + vs * 8 * VC),
                  reinterpret_cast<const char*>(places + static_cast<int64_t>(c) * H), rows - 1 - c * kChunk};
  };
  auto copy = [&](const Source& from, char* image, int i) __attribute__((always_inline)) {
    if (i < kRowCopies) {                                   // 16 rows x 32 columns of the keys or the queries
      const int sd = i % SD, block = wave + NW * (i / SD), ib = block & 3, row = min(row_of(ib, m), from.last);
      const bool keys = block < 4;
      copy16_to_lds((keys ? from.k : from.q) + 64 * sd, 2 * (__umul24(row, keys ? k_stride : q_stride) + 8 * ch), image + (keys ? 0 : kRowsBytes) + 1024 * (ib * SD + sd));
    } else if (i < kRowCopies + kMatCopies) {               // a lower triangular matrix's blocks of 16 x 32 that are not all zero
      const int j = kMatCopies * wave + i - kRowCopies, which = j / 6, b = j % 6, ib = b < 2 ? b : b / 2 + 1, kk = b < 2 ? 0 : b & 1;
      copy16_to_lds(from.place + 8192 * which + 4096 * (ib >> 1) + 64 * (ib & 1) + 1024 * kk, mat_lane, image + kMatsAt + 1024 * j);
    } else if (i < kCopies - 1) {                           // rows of the slice's values
      const int j = wave + NW * (i - kRowCopies - kMatCopies), row = (64 * j + lane) / VC;
      copy16_to_lds(from.v, 2 * __umul24(min(row, from.last), v_stride) + 16 * ((lane % VC) ^ VOrder::twist(row)), image + kValuesAt + 1024 * j);
    } else if (wave == 0) {
      copy16_to_lds(from.place + 32768, 16 * lane, image + kScaleAt);
    }
  };
  uint32_t vv[4][4];                                        // Direct: values of rows row_of(ib, 4 g4 + r)
  float total = 0.f;
  auto fetch = [&](const Source& from) __attribute__((always_inline)) {
    if constexpr (Direct) {
#pragma unroll
      for (int ib = 0; ib < 4; ++ib)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          vv[ib][r] = reinterpret_cast<const uint16_t*>(from.v)[__umul24(min(row_of(ib, 4 * g4 + r), from.last), v_stride) + 16 * wave + n];
    }
    total = reinterpret_cast<const ChunkPlace*>(from.place)->total;
  };
  {
    const Source from = source(0);
#pragma unroll
    for (int i = 0; i < kCopies; ++i) copy(from, lds, i);
    fetch(from);
  }
  const int slot_ = a.slot_idx[s];
  float* st = slot_ >= 0 ? a.state + (static_cast<int64_t>(slot_) * H + h) * D * Dv + col0 + n : nullptr;
  const bool carry = st != nullptr && a.context_lens[s] > 0;
  f32x4v S[DB];                                             // rows d row_of(db, 4 g4 + r) of its pair's 32, column n
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[db][r] = carry ? st[static_cast<int64_t>(row_of(db, 4 * g4 + r)) * Dv] : 0.f;
  const int place_of = 16 * (16 * g4 + (n ^ (4 * g4)));     // this lane's 16 bytes of an operand block
  auto operand = [&](const char* block) __attribute__((always_inline)) { return ld16(block + place_of); };
  // transposed keys: rows 32 kk + 8 g4 + e of the chunk (positions 4 g4 .. of the blocks 2 kk, 2 kk + 1), column n of block db
  const int across = 16 * (16 * (n & 3) + ((4 * g4 + (n >> 2)) ^ (4 * (n & 3))));
  auto transposed = [&](const char* keys, int db, int kk) __attribute__((always_inline)) {
    const char* p = keys + 1024 * (2 * kk * SD + (db >> 1)) + 8 * (db & 1) + across;
    const u32x2 x = __builtin_bit_cast(u32x2, read_transposed(p)), y = __builtin_bit_cast(u32x2, read_transposed(p + 1024 * SD));
    return u32x4{x[0], x[1], y[0], y[1]};
  };
  // values: rows row_of(ib, 4 g4 + r), r < 4, of column n, in pairs
  auto value_at = [&](const char* values, int ib) __attribute__((always_inline)) {
    const int row = row_of(ib, 4 * g4 + (n >> 2)), chunk = 2 * wave + ((n >> 1) & 1);
    return __builtin_bit_cast(u32x2, read_transposed(values + row * 16 * VC + 16 * (chunk ^ VOrder::twist(row)) + 8 * (n & 1)));
  };
  f32x4v x[4], y[4];                        // right-hand side, then U; the outputs: columns 4 g4 + r of row row_of(ib, n)
  bf16x8 sh[SD], sl[SD], hi[2], lo[2], wh[2], wl[2];
  // four values as half of an operand's parts (block ib of pairs)
  auto split_half = [&](const f32x4v& v, int ib, bf16x8& to_hi, bf16x8& to_lo) __attribute__((always_inline)) {
    const float p[4] = {v[0], v[1], v[2], v[3]};
    u32x2 ph, pl;
    split4(p, ph, pl);
    u32x4 h4 = __builtin_bit_cast(u32x4, to_hi), l4 = __builtin_bit_cast(u32x4, to_lo);
    h4[2 * (ib & 1)] = ph[0], h4[2 * (ib & 1) + 1] = ph[1], l4[2 * (ib & 1)] = pl[0], l4[2 * (ib & 1) + 1] = pl[1];
    to_hi = frag(h4), to_lo = frag(l4);
  };
  auto split_state = [&](int i) __attribute__((always_inline)) { split_half(S[i], i, sh[i / 2], sl[i / 2]); };
#pragma unroll
  for (int i = 0; i < DB; ++i) split_state(i);
  const int64_t row_floats = static_cast<int64_t>(H) * Dv;
  float* out = static_cast<float*>(a.out) + static_cast<int64_t>(r0) * row_floats + static_cast<int64_t>(h) * Dv + col0 + 4 * g4;
  auto store = [&](int c, int ib, int live) __attribute__((always_inline)) {
    const int row = row_of(ib, n);
    float* to = out + static_cast<int64_t>(c) * kChunk * row_floats + __umul24(row, static_cast<int>(row_floats));
    if (row < live) *reinterpret_cast<f32x4_any*>(to) = y[ib];
  };
  for (int c = 0; c < num; ++c) {
    const char* image = lds + (c & 1) * kImage;
    char* next = lds + ((c + 1) & 1) * kImage;
    const Source from = source(min(c + 1, num - 1));        // (the last chunk fetches itself once more: no copy under a condition)
    copies_landed_barrier();                 // this chunk's image is there, the other's readers are done
    // what the compiler still counts as in flight has landed: it is used here, in front of the next copies, which it would
    // otherwise wait for as well
    float decay = total;
    asm volatile("" : "+v"(decay));
    if constexpr (Direct) {
#pragma unroll
      for (int ib = 0; ib < 4; ++ib)
#pragma unroll
        for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(vv[ib][r]));
    }
    const char *keys = image, *queries = image + kRowsBytes, *mats = image + kMatsAt;
    // beta, rhs, write of this lane's rows of block ib
    auto scale = [&](int which, int ib) __attribute__((always_inline)) {
      return *reinterpret_cast<const f32x4v*>(image + kScaleAt + 4 * (kChunk * which + 32 * (ib >> 1) + 4 * (ib & 1) + 8 * g4));
    };
    // Fragments in the order of their use, four to a slot, read kAhead of them ahead: keys (slots of 32 columns), half of the
    // queries, T, the other queries, transposed keys, P.
    constexpr int kQa = SD / 2, kT = SD + kQa, kQb = kT + 3, kK = kQb + SD - kQa, kP = kK + SD, kSlots = kP + 3, kAhead = 6;
    u32x4 fr[4 * kSlots + kAhead];
    auto read = [&](int f) __attribute__((always_inline)) {
      const int slot = f / 4, i = f % 4;
      auto matrix = [&](int which, int pair) __attribute__((always_inline)) {       // blocks (0, 0) (1, 0), (2, 0) (3, 0), (2, 1) (3, 1): hi, then lo
        const int ib = (pair == 0 ? 0 : 2) + (i & 1), kk = pair == 2;
        return operand(mats + kMatBytes * (2 * which + (i >> 1)) + 1024 * (ib < 2 ? ib : 2 * ib - 2 + kk));
      };
      if (slot < SD) fr[f] = operand(keys + 1024 * (i * SD + slot));
      else if (slot < kT) fr[f] = operand(queries + 1024 * (i * SD + slot - SD));
      else if (slot < kQb) fr[f] = matrix(0, slot - kT);
      else if (slot < kK) fr[f] = operand(queries + 1024 * (i * SD + slot - kQb + kQa));
      else if (slot < kP) fr[f] = transposed(keys, 2 * (slot - kK) + (i & 1), i >> 1);
      else if (slot < kSlots) fr[f] = matrix(1, slot - kP);
    };
    // pieces of other work of `count`, dealt evenly over the steps [0, of) of a phase
    auto pieces = [&](int step, int of, int count, auto&& piece) __attribute__((always_inline)) {
#pragma unroll
      for (int i = step * count / of; i < (step + 1) * count / of; ++i) piece(i);
    };
    // the next chunk's copies, dealt over the steps (products) up to the middle of the state's update: issued side by side they
    // hold the wave up (25 cycles of the compute unit's address path each)
    auto copies = [&](int step) __attribute__((always_inline)) {
      pieces(step, 20 * SD + 18, kCopies, [&](int i) __attribute__((always_inline)) { if (i < kCopies) copy(from, next, i); });
    };
    f32x4v beta[4], rhs[4], write[4];
    u32x2 value[4];
    float reads[4];
#pragma unroll
    for (int f = 0; f < kAhead; ++f) read(f);
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) x[ib] = f32x4v{0.f, 0.f, 0.f, 0.f};
    auto right_hand_side = [&](int b) __attribute__((always_inline)) {
      const float v[4] = {lo_bf(value[b][0]), hi_bf(value[b][0]), lo_bf(value[b][1]), hi_bf(value[b][1])};
#pragma unroll
      for (int r = 0; r < 4; ++r) x[b][r] = beta[b][r] * v[r] - rhs[b][r] * x[b][r];
      split_half(x[b], b, hi[b >> 1], lo[b >> 1]);
    };
    __builtin_amdgcn_sched_barrier(0);
    unrolled<kSlots>([&](auto number) __attribute__((always_inline)) {
      constexpr int slot = decltype(number)::value;
#pragma unroll
      for (int f = 4 * slot + kAhead; f < 4 * slot + 4 + kAhead; ++f) read(f);
      const u32x4* fs = fr + 4 * slot;
      if constexpr (slot == SD) {
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) y[ib] = f32x4v{0.f, 0.f, 0.f, 0.f};
        if constexpr (kQa == 0) {                           // (a head of 32: the right-hand side in front of T)
#pragma unroll
          for (int i = 0; i < 4; ++i) right_hand_side(i);
        }
      }
      if constexpr (slot == kT) {
        if constexpr (Direct) fetch(from);
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) x[ib] = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) write[ib] = scale(3, ib), reads[ib] = *reinterpret_cast<const float*>(image + kScaleAt + 4 * (2 * kChunk + row_of(ib, n)));
      }
      if constexpr (slot == SD - 1) {
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) {
          beta[ib] = scale(0, ib), rhs[ib] = scale(1, ib);
          if constexpr (Direct) value[ib] = u32x2{vv[ib][0] | (vv[ib][1] << 16), vv[ib][2] | (vv[ib][3] << 16)};
          else value[ib] = value_at(image + kValuesAt, ib);
        }
      }
      if constexpr (slot < kT || (slot >= kQb && slot < kK)) {        // keys times the state; the state times queries, transposed
        constexpr int sd = slot < SD ? slot : slot < kT ? slot - SD : slot - kQb + kQa;
#pragma unroll
        for (int part = 0; part < 2; ++part)
#pragma unroll
          for (int ib = 0; ib < 4; ++ib) {
            const bf16x8 state = part == 0 ? sh[sd] : sl[sd];
            if constexpr (slot < SD) x[ib] = mfma16(frag(fs[ib]), state, x[ib]);
            else y[ib] = mfma16(state, frag(fs[ib]), y[ib]);
            constexpr int from_step = 8 * (slot < SD ? slot : slot < kT ? slot - SD : slot - kQb);
            const int step = from_step + 4 * part + ib;
            copies((slot < kT ? 0 : 8 * kT + 18) + from_step + (slot >= SD && slot < kT ? 8 * SD : 0) + 4 * part + ib);
            if constexpr (slot < SD) {
              pieces(step, 4 * SD, 4, [&](int i) __attribute__((always_inline)) {
                if (i < 4 && c > 0) store(c - 1, i, kChunk);
              });
            } else if constexpr (slot < kT) pieces(step, 8 * kQa, 4, right_hand_side);
            else {
              pieces(step, 8 * (SD - kQa), 4, [&](int b) __attribute__((always_inline)) { split_half(x[b] * write[b], b, wh[b >> 1], wl[b >> 1]); });
            }
            __builtin_amdgcn_sched_barrier(0);
          }
      } else if constexpr (slot < kQb || slot >= kP) {      // T times the right-hand side; U times P, transposed
        constexpr int pair = slot < kQb ? slot - kT : slot - kP, kk = pair == 2;
#pragma unroll
        for (int part = 0; part < 3; ++part) {
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const int ib = (pair == 0 ? 0 : 2) + i;
            const bf16x8 mat = frag(fs[part == 2 ? 2 + i : i]), other = part == 1 ? lo[kk] : hi[kk];
            if constexpr (slot < kQb) x[ib] = mfma16(mat, other, x[ib]), copies(8 * kT + 6 * pair + 2 * part + i);
            else y[ib] = mfma16(other, mat, y[ib]);
            if constexpr (slot >= kP) pieces(6 * pair + 2 * part + i, 18, DB, split_state);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        if constexpr (slot == kT && !Direct) fetch(from);
      } else {                                              // the state's update, two blocks at a time
        constexpr int db = 2 * (slot - kK);
        f32x4v acc[2] = {S[db] * decay, S[db + 1] * decay};
#pragma unroll
        for (int part = 0; part < 4; ++part)
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            acc[i] = mfma16(frag(fs[2 * (part >> 1) + i]), part & 1 ? wl[part >> 1] : wh[part >> 1], acc[i]);
            copies(8 * 2 * SD + 18 + 8 * (slot - kK) + 2 * part + i);
            pieces(8 * (slot - kK) + 2 * part + i, 8 * SD, 4, [&](int b) __attribute__((always_inline)) {
              split_half(x[b], b, hi[b >> 1], lo[b >> 1]);
              y[b] *= reads[b];
            });
            __builtin_amdgcn_sched_barrier(0);
          }
        S[db] = acc[0], S[db + 1] = acc[1];
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // (the last copies, which nobody waits for, end before the workgroup)
#pragma unroll
  for (int i = 0; i < 4; ++i) store(num - 1, i, rows - (num - 1) * kChunk);
  if (st != nullptr) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 4; ++r) st[static_cast<int64_t>(row_of(db, 4 * g4 + r)) * Dv] = S[db][r];
  }
}

template <int D, int NW>
__global__ __launch_bounds__(64 * NW, NW / 4 > 0 ? NW / 4 : 1) void delta_chunk_wide_kernel(hymeta_delta_rule_args a, bool short_too) {
  __shared__ __attribute__((aligned(16))) char images[2 * WideImage<D, NW>::kBytes];
  delta_chunk_wide<D, NW>(a, blockIdx.x, blockIdx.y, blockIdx.z, images, short_too);
}

// More (head, sequence, 128 columns) than half of the compute units, but not more than there are: `whole` of them, of the shortest
// sequences, by eight waves, which take 4.4 us a chunk, the others by four waves on each of two compute units, 2.6 us a chunk.  A step ends
// with the longest of either, and lengths differ: 28 heads, five portions of 1801 to 1413 rows 128 -> 110 us, six of 1365 to 910 (80
// pairs of 168 whole) 139.5 -> 130 with the launch in front; equal ones are level (five of 1600, 162), and so are portions of up to kMixedRows rows
// (six of 90 27.7 and 28.3).  grid = (whole + 2 (pairs - whole)), 8 waves, of which a half needs 4; at most 64 sequences.
constexpr int kMixedRows = 4 * kChunk;
template <int D>
__global__ __launch_bounds__(512, 2) void delta_chunk_mixed_kernel(hymeta_delta_rule_args a, int whole, bool short_too) {
  __shared__ __attribute__((aligned(16))) char images[2 * WideImage<D, 8>::kBytes];
  const int lane = threadIdx.x & 63, n = a.num_seqs, per_seq = a.num_heads * (a.v_dim / 128), halves = n * per_seq - whole;
  int pair, half = -1;                                      // pairs numbered from the longest sequence's on
  if (static_cast<int>(blockIdx.x) < whole) pair = n * per_seq - 1 - blockIdx.x;
  else {                                                    // a pair's halves eight workgroups apart, on one die: they read the same keys and matrices
    const int j = blockIdx.x - whole, first = j / 16 * 8, side = min(8, halves - first), in = j - 2 * first;
    half = in >= side, pair = first + in - half * side;
  }
  // the sequence of a rank: a lane each
  const int len = lane < n ? a.query_start_loc[lane + 1] - a.query_start_loc[lane] : -1;
  int rank = 0;
  for (int i = 0; i < n; ++i) {
    const int other = __builtin_amdgcn_readlane(len, i);
    rank += other > len || (other == len && i < lane);
  }
  auto uniform = [](int x) __attribute__((always_inline)) { return __builtin_amdgcn_readfirstlane(x); };      // (of a division, which runs in vector registers)
  const int place = uniform(pair / per_seq), s = __builtin_ctzll(__ballot(lane < n && rank == place));
  const int at = pair - place * per_seq, part = uniform(at / a.num_heads), h = at - part * a.num_heads;
  if (half < 0) delta_chunk_wide<D, 8>(a, h, s, part, images, short_too);
  else if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < 4) delta_chunk_wide<D, 4>(a, h, s, 2 * part + half, images, short_too);
}

inline bool chunk_dims(int head_dim, int v_dim, int act_dtype) {
  return act_dtype == HYMETA_BF16 && head_dim >= 32 && head_dim <= 128 && head_dim % 32 == 0 && v_dim % 32 == 0 && v_dim / 16 <= 65535;
}
inline bool chunk_shape(const hymeta_delta_rule_args& a) {
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  // (a chunk's rows at 24-bit products of row and stride)
  const bool offsets = std::max(a.q_stride_t, std::max(a.k_stride_t, a.v_stride_t)) < (1 << 23) && static_cast<int64_t>(a.num_heads) * a.v_dim < (1 << 22);
  return chunk_dims(a.head_dim, a.v_dim, a.act_dtype) && offsets && a.q_stride_t % 8 == 0 && a.k_stride_t % 8 == 0 && aligned(a.q) && aligned(a.k);
}
inline int64_t chunk_numbers(int num_tokens, int num_seqs) { return static_cast<int64_t>(num_tokens) / kChunk + num_seqs; }

inline bool step_shape(const hymeta_delta_rule_args& a) {
  const int dv4 = a.v_dim / 4;
  return a.v_dim % 4 == 0 && dv4 <= 256 && 256 % dv4 == 0 && a.head_dim <= kStepMaxD && static_cast<int64_t>(a.head_dim) * dv4 <= 256 * kStepRows &&
         reinterpret_cast<uintptr_t>(a.state) % 16 == 0;
}

template <typename A>
void launch_rows(const hymeta_delta_rule_args& a, hipStream_t st, int min_rows, int max_rows) {
  const dim3 grid(a.num_heads, a.num_seqs, (a.v_dim + 255) / 256);
  const dim3 block(a.v_dim >= 256 ? 256 : (a.v_dim + 63) / 64 * 64);
  if (a.head_dim <= 32) hipLaunchKernelGGL((delta_rule_rows_kernel<A, 32>), grid, block, 0, st, a, min_rows, max_rows);
  else if (a.head_dim <= 64) hipLaunchKernelGGL((delta_rule_rows_kernel<A, 64>), grid, block, 0, st, a, min_rows, max_rows);
  else if (a.head_dim <= 128) hipLaunchKernelGGL((delta_rule_rows_kernel<A, 128>), grid, block, 0, st, a, min_rows, max_rows);
  else hipLaunchKernelGGL((delta_rule_rows_kernel<A, 256>), grid, block, 0, st, a, min_rows, max_rows);
}

template <int D>
void launch_short(const hymeta_delta_rule_args& a, hipStream_t st, int max_rows) {
  constexpr int NT = D <= 64 ? 64 : 128;
  if (a.v_dim % 64 == 0) hipLaunchKernelGGL((delta_short_kernel<D, 16, NT>), dim3(a.num_heads, a.v_dim / 64, a.num_seqs), dim3(NT), 0, st, a, max_rows);
  else hipLaunchKernelGGL((delta_short_kernel<D, 8, NT>), dim3(a.num_heads, a.v_dim / 32, a.num_seqs), dim3(NT), 0, st, a, max_rows);
}

template <int D>
void launch_chunks(const hymeta_delta_rule_args& a, hipStream_t st, int64_t chunks, bool short_too) {
  const int64_t portions = long_portions(a.num_tokens, a.num_seqs, a.max_query_len), lanes = a.num_heads * portions;
  const int64_t idle = a.num_heads * (a.num_seqs - portions) * (a.v_dim / 32);
  const bool narrow = lanes * (a.v_dim / 32) <= kFewGroups && idle <= static_cast<int64_t>(kIdleGroupsPerRow) * a.max_query_len;
  const dim3 solve(static_cast<unsigned>(chunks), a.num_heads);
  if (narrow) {
    if (short_too) hipLaunchKernelGGL((delta_chunk_solve_kernel<D, true, true>), solve, dim3(256), 0, st, a, chunks);
    else hipLaunchKernelGGL((delta_chunk_solve_kernel<D, true, false>), solve, dim3(256), 0, st, a, chunks);
    hipLaunchKernelGGL(delta_chunk_narrow_kernel<D>, dim3(a.num_heads, a.num_seqs, a.v_dim / 16), dim3(256), 0, st, a, chunks);
    return;
  }
  // Short portions in the first launch take it registers, and with them a third of its workgroups: where none are to be expected, those
  // that there are after all go along in the second (28 heads, portions of 6 to 9 rows 34.6 -> 26.9 us).
  const bool later = short_too && a.num_seqs == portions;
  if (short_too && !later) hipLaunchKernelGGL((delta_chunk_solve_kernel<D, false, true>), solve, dim3(256), 0, st, a, chunks);
  else hipLaunchKernelGGL((delta_chunk_solve_kernel<D, false, false>), solve, dim3(256), 0, st, a, chunks);
  auto launch = [&](auto nw) {
    constexpr int NW = decltype(nw)::value;
    hipLaunchKernelGGL((delta_chunk_wide_kernel<D, NW>), dim3(a.num_heads, a.num_seqs, a.v_dim / (16 * NW)), dim3(64 * NW), 0, st, a, later);
  };
  using std::integral_constant;
  const bool aligned = a.v_stride_t % 8 == 0 && reinterpret_cast<uintptr_t>(a.v) % 16 == 0;      // (values copied to LDS)
  const int64_t pairs = static_cast<int64_t>(a.num_heads) * a.num_seqs * (a.v_dim / 128);
  if (aligned && a.v_dim % 128 == 0 && lanes * (a.v_dim / 64) > kManyGroups) {
    if (pairs < kManyGroups && a.num_seqs <= 64 && a.max_query_len > kMixedRows) {
      const int whole = static_cast<int>(2 * pairs - kManyGroups);
      hipLaunchKernelGGL((delta_chunk_mixed_kernel<D>), dim3(kManyGroups), dim3(512), 0, st, a, whole, later);
    } else {
      launch(integral_constant<int, 8>{});
    }
  }
  else if (aligned && a.v_dim % 64 == 0) launch(integral_constant<int, 4>{});
  else launch(integral_constant<int, 2>{});
}

}  // namespace

}  // namespace hymeta

using namespace hymeta;

extern "C" size_t hymeta_delta_rule_workspace_bytes(int32_t num_tokens, int32_t num_seqs, int32_t num_heads, int32_t num_qk_heads, int32_t head_dim,
                                                    int32_t v_dim, int32_t act_dtype, int32_t max_query_len) {
  if (num_tokens <= 0 || num_seqs <= 0 || num_heads <= 0 || num_qk_heads <= 0 || max_query_len < kChunkMinRows || !chunk_dims(head_dim, v_dim, act_dtype)) return 0;
  const int64_t chunks = chunk_numbers(num_tokens, num_seqs);
  return rows_at(chunks, num_heads) + static_cast<size_t>(chunks) * num_qk_heads * 3 * head_dim * kChunk * 2;
}

extern "C" int hymeta_delta_rule(const hymeta_delta_rule_args* args, hymeta_stream_t stream) {
  if (!args_ok(args)) return HYMETA_ERR_INVALID_ARG;
  const hymeta_delta_rule_args& a = *args;
  if (a.num_tokens < 0 || a.num_seqs < 0 || a.num_heads <= 0 || a.num_qk_heads <= 0 || a.head_dim <= 0 || a.v_dim <= 0) return HYMETA_ERR_INVALID_ARG;
  if (a.num_heads % a.num_qk_heads != 0) return HYMETA_ERR_INVALID_ARG;
  if (!act_dtype_ok(a.act_dtype)) return HYMETA_ERR_UNSUPPORTED;
  if (a.head_dim > 256 || a.num_seqs > 65535 || a.num_heads > 65535 || a.v_dim > 256 * 65535) return HYMETA_ERR_UNSUPPORTED;
  if (a.num_tokens == 0 || a.num_seqs == 0) return HYMETA_OK;
  if (!a.q || !a.k || !a.v || !a.beta_logit || !a.log2_decay || !a.state || !a.out || !a.query_start_loc || !a.context_lens || !a.slot_idx) return HYMETA_ERR_INVALID_ARG;
  const int64_t qk = static_cast<int64_t>(a.num_qk_heads) * a.head_dim, hv = static_cast<int64_t>(a.num_heads) * a.v_dim;
  if (a.q_stride_t < qk || a.k_stride_t < qk || a.v_stride_t < hv || a.beta_stride_t < a.num_heads) return HYMETA_ERR_INVALID_ARG;
  const bool step = step_shape(a);
  if (a.norm_weight) {
    if (!a.gate || a.gate_stride_t < hv) return HYMETA_ERR_INVALID_ARG;
    if (!step || a.max_query_len != 1 || a.num_tokens != a.num_seqs) return HYMETA_ERR_UNSUPPORTED;
  }
  hipStream_t st = begin_launches(stream);
  const bool bf = a.act_dtype == HYMETA_BF16;
  int min_rows = 1, max_rows = 0x7fffffff;
  const bool rows_too = reinterpret_cast<uintptr_t>(a.state) % 16 == 0;          // (the kernels of short portions read the state in fours)
  if (chunk_shape(a) && a.max_query_len >= (rows_too ? 2 : kChunkMinRows)) {
    auto dims = [&](auto&& run) {
      if (a.head_dim == 32) run(std::integral_constant<int, 32>{});
      else if (a.head_dim == 64) run(std::integral_constant<int, 64>{});
      else if (a.head_dim == 96) run(std::integral_constant<int, 96>{});
      else run(std::integral_constant<int, 128>{});
    };
    if (a.max_query_len < kChunkMinRows) {
      dims([&](auto d) { launch_short<decltype(d)::value>(a, st, max_rows); });
      return launch_status();
    }
    const size_t need = hymeta_delta_rule_workspace_bytes(a.num_tokens, a.num_seqs, a.num_heads, a.num_qk_heads, a.head_dim, a.v_dim, a.act_dtype, a.max_query_len);
    if (!a.workspace || a.workspace_bytes < need || reinterpret_cast<uintptr_t>(a.workspace) % 16 != 0) return HYMETA_ERR_WORKSPACE;
    const int64_t shorts = static_cast<int64_t>(a.num_heads) * (a.num_seqs - long_portions(a.num_tokens, a.num_seqs, a.max_query_len));
    const bool apart = rows_too && short_apart(a, shorts);
    dims([&](auto d) {
      if (apart) launch_short<decltype(d)::value>(a, st, kChunkMinRows - 1);
      launch_chunks<decltype(d)::value>(a, st, chunk_numbers(a.num_tokens, a.num_seqs), rows_too && !apart);
    });
    if (rows_too) return launch_status();
    max_rows = kChunkMinRows - 1;
  }
  if (step) {
    const dim3 grid(a.num_heads, a.num_seqs), block(256);
    if (a.norm_weight) {
      if (bf) hipLaunchKernelGGL((delta_rule_step_kernel<ActBf16, true>), grid, block, 0, st, a);
      else hipLaunchKernelGGL((delta_rule_step_kernel<ActF32, true>), grid, block, 0, st, a);
    } else {
      if (bf) hipLaunchKernelGGL((delta_rule_step_kernel<ActBf16, false>), grid, block, 0, st, a);
      else hipLaunchKernelGGL((delta_rule_step_kernel<ActF32, false>), grid, block, 0, st, a);
    }
    min_rows = 2;
  }
  if (a.max_query_len >= min_rows && max_rows >= min_rows) {
    if (bf) launch_rows<ActBf16>(a, st, min_rows, max_rows);
    else launch_rows<ActF32>(a, st, min_rows, max_rows);
  }
  return launch_status();
}
