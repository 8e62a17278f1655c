// Linear attention with a constant decay per head ("lightning attention"): S <- decay S + k v^T, out = S^T q, the state
// fp32 and carried per sequence; and the output norm with its sigmoid gate.
#include <algorithm>
#include <type_traits>

#include "chunk_scan.h"

namespace hymeta {

namespace {

__device__ __forceinline__ float silu_f(float x) { return x / (1.f + expf(-x)); }

// Token by token.  grid = (heads, sequences, value columns in runs of 256); a thread owns one value column c and keeps
// that column of the state, S[:, c], in registers; q_t and k_t go through LDS.
template <typename A, int DMAX>
__global__ __launch_bounds__(256) void lightning_rows_kernel(hymeta_lightning_attention_args a, int min_rows) {
  typedef typename A::elem elem;
  __shared__ float s_q[2][DMAX], s_k[2][DMAX];
  const int h = blockIdx.x, s = blockIdx.y;
  const int c = blockIdx.z * 256 + threadIdx.x;
  const int H = a.num_heads, D = a.head_dim, Dv = a.v_dim;
  const int r0 = a.query_start_loc[s], r1 = a.query_start_loc[s + 1];
  if (r1 - r0 < min_rows) return;          // single rows: the other kernel's
  const int slot = a.slot_idx[s];
  const bool live = c < Dv;
  float* st = (slot >= 0) ? a.state + ((static_cast<int64_t>(slot) * H + h) * D) * Dv : nullptr;
  float S[DMAX];
  const bool carry = st != nullptr && a.context_lens[s] > 0 && live;
#pragma unroll
  for (int d = 0; d < DMAX; ++d) S[d] = (carry && d < D) ? st[static_cast<int64_t>(d) * Dv + c] : 0.f;
  const float decay = a.decay[h];
  const int64_t q_off = static_cast<int64_t>(h) * D, k_off = static_cast<int64_t>(H) * D + q_off;
  const int64_t v_off = 2 * static_cast<int64_t>(H) * D + static_cast<int64_t>(h) * Dv;
  for (int t = r0; t < r1; ++t) {
    const elem* row = static_cast<const elem*>(a.qkv) + static_cast<int64_t>(t) * a.qkv_stride_t;
    const int buf = (t - r0) & 1;
    for (int d = threadIdx.x; d < D; d += blockDim.x) {
      s_q[buf][d] = silu_f(A::ld(row + q_off + d));
      s_k[buf][d] = silu_f(A::ld(row + k_off + d));
    }
    const float v = live ? silu_f(A::ld(row + v_off + c)) : 0.f;
    __syncthreads();           // one barrier per token: the next token fills the other buffer
    float o = 0.f;
#pragma unroll
    for (int d = 0; d < DMAX; ++d) {
      if (d < D) {
        S[d] = fmaf(decay, S[d], s_k[buf][d] * v);
        o = fmaf(S[d], s_q[buf][d], o);
      }
    }
    if (live) a.out[static_cast<int64_t>(t) * H * Dv + static_cast<int64_t>(h) * Dv + c] = o;
  }
  if (st != nullptr && live) {
#pragma unroll
    for (int d = 0; d < DMAX; ++d)
      if (d < D) st[static_cast<int64_t>(d) * Dv + c] = S[d];
  }
}

// Rows of up to kGatedCached columns are read once (a thread keeps its columns in registers).
constexpr int kGatedPerThread = 16, kGatedCached = 256 * kGatedPerThread;

// grid = (rows, groups): a workgroup norms one of the row's equal consecutive parts.
template <typename A, bool Cached>
__global__ __launch_bounds__(256) void gated_rms_norm_kernel(hymeta_gated_rms_norm_args a) {
  typedef typename A::elem elem;
  __shared__ float red[4];
  const int64_t t = blockIdx.x;
  const int width = a.width / gridDim.y, c0 = blockIdx.y * width;
  const float* x = a.x + t * a.width + c0;
  const elem* g = static_cast<const elem*>(a.gate) + t * a.gate_stride_t + c0;
  const float* weight = a.weight ? a.weight + c0 : nullptr;
  elem* out = static_cast<elem*>(a.out) + t * a.width + c0;
  const bool silu = a.gate_act == HYMETA_GATE_SILU, first = a.gate_first != 0;
  auto gate_of = [&](float gv) { const float sg = sigmoid_exact(gv); return silu ? gv * sg : sg; };
  float ss = 0.f;
  if (Cached) {
    float xv[kGatedPerThread], gv[kGatedPerThread];
#pragma unroll
    for (int u = 0; u < kGatedPerThread; ++u) {
      const int c = threadIdx.x + 256 * u;
      xv[u] = c < width ? x[c] : 0.f;
      gv[u] = c < width ? gate_of(A::ld(g + c)) : 0.f;
      if (first) xv[u] *= gv[u], gv[u] = 1.f;
      ss = fmaf(xv[u], xv[u], ss);
    }
    ss = block_sum<4>(ss, red);
    const float inv = 1.f / sqrtf(ss / static_cast<float>(width) + a.eps);
#pragma unroll
    for (int u = 0; u < kGatedPerThread; ++u) {
      const int c = threadIdx.x + 256 * u;
      if (c < width) A::st(out + c, xv[u] * inv * (weight ? weight[c] : 1.f) * gv[u]);
    }
    return;
  }
  for (int c = threadIdx.x; c < width; c += 256) {
    const float v = first ? x[c] * gate_of(A::ld(g + c)) : x[c];
    ss = fmaf(v, v, ss);
  }
  ss = block_sum<4>(ss, red);
  const float inv = 1.f / sqrtf(ss / static_cast<float>(width) + a.eps);
  for (int c = threadIdx.x; c < width; c += 256) {
    const float gv = gate_of(A::ld(g + c));
    A::st(out + c, x[c] * inv * (weight ? weight[c] : 1.f) * gv);
  }
}

// Narrow groups (a head's output): a wave per (row, group), the group's columns in the lanes' registers, no barrier.
constexpr int kGatedWavePerLane = 16, kGatedWaveCols = 64 * kGatedWavePerLane;

template <typename A>
__global__ __launch_bounds__(256) void gated_rms_norm_wave_kernel(hymeta_gated_rms_norm_args a, int groups) {
  typedef typename A::elem elem;
  const int64_t t = blockIdx.x;
  const int lane = threadIdx.x & 63, grp = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (grp >= groups) return;
  const int width = a.width / groups, c0 = grp * width;
  const float* x = a.x + t * a.width + c0;
  const elem* g = static_cast<const elem*>(a.gate) + t * a.gate_stride_t + c0;
  const float* weight = a.weight ? a.weight + c0 : nullptr;
  elem* out = static_cast<elem*>(a.out) + t * a.width + c0;
  const bool silu = a.gate_act == HYMETA_GATE_SILU, first = a.gate_first != 0;
  float xv[kGatedWavePerLane], gv[kGatedWavePerLane];
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < kGatedWavePerLane; ++u) {
    const int c = lane + 64 * u;
    if (64 * u >= width) { xv[u] = 0.f, gv[u] = 0.f; continue; }
    xv[u] = c < width ? x[c] : 0.f;
    const float raw = c < width ? A::ld(g + c) : 0.f;
    const float sg = sigmoid_exact(raw);
    gv[u] = silu ? raw * sg : sg;
    if (first) xv[u] *= gv[u], gv[u] = 1.f;
    ss = fmaf(xv[u], xv[u], ss);
  }
  ss = wave_sum(ss);
  const float inv = 1.f / sqrtf(ss / static_cast<float>(width) + a.eps);
#pragma unroll
  for (int u = 0; u < kGatedWavePerLane; ++u) {
    const int c = lane + 64 * u;
    if (c < width) A::st(out + c, xv[u] * inv * (weight ? weight[c] : 1.f) * gv[u]);
  }
}

static_assert(kScanRows == HYMETA_LIGHTNING_CHUNK, "the chunk of the header");

inline bool chunk_shape(const hymeta_lightning_attention_args& a) {
  return a.act_dtype == HYMETA_BF16 && (a.head_dim == 32 || a.head_dim == 64 || a.head_dim == 128) && a.v_dim % 32 == 0 &&
         a.qkv_stride_t % 8 == 0 && reinterpret_cast<uintptr_t>(a.qkv) % 16 == 0 && reinterpret_cast<uintptr_t>(a.state) % 16 == 0 &&
         reinterpret_cast<uintptr_t>(a.out) % 16 == 0 && a.v_dim / 32 <= 65535 && scan_offsets_fit(a.qkv_stride_t, a.num_heads, a.v_dim);
}

// Sequences with one row (decode).  grid = (heads, sequences), 256 threads over the state in fours of value columns: a
// thread takes the columns 4 c4 .. 4 c4 + 3 of the rows d0, d0 + dstep, ... of S (16-byte loads and stores, four rows in
// flight together), the partial outputs of the dstep row groups meet in LDS.
constexpr int kStepMaxD = 256;
template <typename A>
__global__ __launch_bounds__(256) void lightning_step_kernel(hymeta_lightning_attention_args a) {
  typedef typename A::elem elem;
  __shared__ float s_q[kStepMaxD], s_k[kStepMaxD];
  __shared__ __attribute__((aligned(16))) float s_o[256 * 4];
  const int h = blockIdx.x, s = blockIdx.y;
  const int t = a.query_start_loc[s];
  if (a.query_start_loc[s + 1] - t != 1) return;
  const int H = a.num_heads, D = a.head_dim, Dv = a.v_dim, Dv4 = Dv / 4;
  const int c4 = threadIdx.x % Dv4, d0 = threadIdx.x / Dv4, dstep = 256 / Dv4;
  const int slot = a.slot_idx[s];
  float* st = slot >= 0 ? a.state + ((static_cast<int64_t>(slot) * H + h) * D) * Dv : nullptr;
  const bool carry = st != nullptr && a.context_lens[s] > 0;
  const elem* row = static_cast<const elem*>(a.qkv) + static_cast<int64_t>(t) * a.qkv_stride_t;
  for (int d = threadIdx.x; d < D; d += 256) {
    s_q[d] = silu_f(A::ld(row + static_cast<int64_t>(h) * D + d));
    s_k[d] = silu_f(A::ld(row + static_cast<int64_t>(H + h) * D + d));
  }
  float v[4];
  A::ld4(row + 2 * static_cast<int64_t>(H) * D + static_cast<int64_t>(h) * Dv + 4 * c4, v);
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = silu_f(v[e]);
  const float decay = a.decay[h];
  __syncthreads();
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int db = d0; db < D; db += 4 * dstep) {
    f32x4 S[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int d = db + u * dstep;
      S[u] = (carry && d < D) ? *reinterpret_cast<const f32x4*>(st + static_cast<int64_t>(d) * Dv + 4 * c4) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int d = db + u * dstep;
      if (d >= D) continue;
      const float k = s_k[d], q = s_q[d];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        S[u][e] = fmaf(decay, S[u][e], k * v[e]);
        acc[e] = fmaf(S[u][e], q, acc[e]);
      }
      if (st != nullptr) *reinterpret_cast<f32x4*>(st + static_cast<int64_t>(d) * Dv + 4 * c4) = S[u];
    }
  }
  *reinterpret_cast<f32x4*>(&s_o[threadIdx.x * 4]) = acc;          // [d0][4 c4 + e]
  __syncthreads();
  for (int c = threadIdx.x; c < Dv; c += 256) {
    float o = 0.f;
    for (int g = 0; g < dstep; ++g) o += s_o[(g * Dv4 + c / 4) * 4 + (c & 3)];
    a.out[static_cast<int64_t>(t) * H * Dv + static_cast<int64_t>(h) * Dv + c] = o;
  }
}

inline bool step_shape(const hymeta_lightning_attention_args& a) {
  const int dv4 = a.v_dim / 4;
  const int bytes = a.act_dtype == HYMETA_BF16 ? 2 : 4;
  return a.v_dim % 4 == 0 && dv4 <= 256 && 256 % dv4 == 0 && a.head_dim <= kStepMaxD && reinterpret_cast<uintptr_t>(a.state) % 16 == 0 &&
         reinterpret_cast<uintptr_t>(a.qkv) % (4 * bytes) == 0 && a.qkv_stride_t % 4 == 0 && (2 * a.num_heads * a.head_dim) % 4 == 0;
}

template <typename A>
void launch_rows(const hymeta_lightning_attention_args& a, hipStream_t st, int min_rows) {
  const dim3 grid(a.num_heads, a.num_seqs, (a.v_dim + 255) / 256);
  const dim3 block(a.v_dim >= 256 ? 256 : (a.v_dim + 63) / 64 * 64);
  if (a.head_dim <= 32) hipLaunchKernelGGL((lightning_rows_kernel<A, 32>), grid, block, 0, st, a, min_rows);
  else if (a.head_dim <= 64) hipLaunchKernelGGL((lightning_rows_kernel<A, 64>), grid, block, 0, st, a, min_rows);
  else if (a.head_dim <= 128) hipLaunchKernelGGL((lightning_rows_kernel<A, 128>), grid, block, 0, st, a, min_rows);
  else hipLaunchKernelGGL((lightning_rows_kernel<A, 256>), grid, block, 0, st, a, min_rows);
}

}  // namespace

}  // namespace hymeta

using namespace hymeta;

extern "C" size_t hymeta_lightning_attention_workspace_bytes(int32_t num_seqs, int32_t num_heads, int32_t head_dim, int32_t v_dim,
                                                             int32_t max_query_len) {
  return scan_workspace_bytes(num_seqs, num_heads, head_dim, v_dim, max_query_len);
}

extern "C" int hymeta_lightning_attention(const hymeta_lightning_attention_args* args, hymeta_stream_t stream) {
  if (!args_ok(args)) return HYMETA_ERR_INVALID_ARG;
  const hymeta_lightning_attention_args& a = *args;
  if (a.num_tokens < 0 || a.num_seqs < 0 || a.num_heads <= 0 || a.head_dim <= 0 || a.v_dim <= 0) return HYMETA_ERR_INVALID_ARG;
  if (!act_dtype_ok(a.act_dtype)) return HYMETA_ERR_UNSUPPORTED;
  if (a.head_dim > 256 || a.num_seqs > 65535 || a.v_dim > 256 * 65535) return HYMETA_ERR_UNSUPPORTED;
  if (a.num_tokens == 0 || a.num_seqs == 0) return HYMETA_OK;
  if (!a.qkv || !a.state || !a.decay || !a.out || !a.query_start_loc || !a.context_lens || !a.slot_idx) return HYMETA_ERR_INVALID_ARG;
  if (a.qkv_stride_t < static_cast<int64_t>(a.num_heads) * (2 * a.head_dim + a.v_dim)) return HYMETA_ERR_INVALID_ARG;
  hipStream_t st = begin_launches(stream);
  // (portions shorter than a chunk's least run in the same launch)
  if (chunk_shape(a) && a.max_query_len >= 2) {
    const ScanSegments sg = scan_segments(a.num_tokens, a.num_seqs, a.num_heads, a.v_dim, a.max_query_len, true);
    const size_t need = scan_segment_bytes(sg.count, a.num_heads, a.head_dim, a.v_dim);
    if (need > 0 && (!a.workspace || a.workspace_bytes < need)) return HYMETA_ERR_WORKSPACE;
    const uint16_t* qkv = static_cast<const uint16_t*>(a.qkv);
    const int64_t keys = static_cast<int64_t>(a.num_heads) * a.head_dim;
    const ChunkScanArgs c{qkv, qkv + keys, qkv + 2 * keys, a.qkv_stride_t, a.qkv_stride_t, a.qkv_stride_t, a.decay, nullptr, nullptr, nullptr,
                          a.state, a.out, static_cast<float*>(a.workspace), a.query_start_loc, a.context_lens, a.slot_idx,
                          a.num_seqs, a.num_heads, a.num_heads, a.v_dim};
    launch_chunk_scan<true>(c, a.num_tokens, a.head_dim, a.max_query_len, sg, st);
    return launch_status();
  }
  int min_rows = 1;
  if (step_shape(a)) {
    const dim3 grid(a.num_heads, a.num_seqs);
    if (a.act_dtype == HYMETA_BF16) hipLaunchKernelGGL(lightning_step_kernel<ActBf16>, grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL(lightning_step_kernel<ActF32>, grid, dim3(256), 0, st, a);
    min_rows = 2;
  }
  if (a.max_query_len >= min_rows) {
    if (a.act_dtype == HYMETA_BF16) launch_rows<ActBf16>(a, st, min_rows);
    else launch_rows<ActF32>(a, st, min_rows);
  }
  return launch_status();
}

extern "C" int hymeta_gated_rms_norm(const hymeta_gated_rms_norm_args* args, hymeta_stream_t stream) {
  if (!args_ok(args)) return HYMETA_ERR_INVALID_ARG;
  const hymeta_gated_rms_norm_args& a = *args;
  if (a.num_tokens < 0 || a.width <= 0) return HYMETA_ERR_INVALID_ARG;
  if (!act_dtype_ok(a.act_dtype)) return HYMETA_ERR_UNSUPPORTED;
  if (a.num_tokens == 0) return HYMETA_OK;
  if (!a.x || !a.gate || !a.out || a.gate_stride_t < a.width) return HYMETA_ERR_INVALID_ARG;
  const int groups = a.groups > 1 ? a.groups : 1;
  if (a.width % groups != 0 || groups > 65535) return HYMETA_ERR_INVALID_ARG;
  if (a.gate_act != HYMETA_GATE_SIGMOID && a.gate_act != HYMETA_GATE_SILU) return HYMETA_ERR_UNSUPPORTED;
  hipStream_t st = begin_launches(stream);
  if (groups > 1 && a.width / groups <= kGatedWaveCols) {
    const dim3 grid(a.num_tokens, (groups + 3) / 4);
    if (a.act_dtype == HYMETA_BF16) hipLaunchKernelGGL(gated_rms_norm_wave_kernel<ActBf16>, grid, dim3(256), 0, st, a, groups);
    else hipLaunchKernelGGL(gated_rms_norm_wave_kernel<ActF32>, grid, dim3(256), 0, st, a, groups);
    return launch_status();
  }
  const bool cached = a.width / groups <= kGatedCached;
  if (a.act_dtype == HYMETA_BF16) {
    if (cached) hipLaunchKernelGGL((gated_rms_norm_kernel<ActBf16, true>), dim3(a.num_tokens, groups), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((gated_rms_norm_kernel<ActBf16, false>), dim3(a.num_tokens, groups), dim3(256), 0, st, a);
  } else {
    if (cached) hipLaunchKernelGGL((gated_rms_norm_kernel<ActF32, true>), dim3(a.num_tokens, groups), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((gated_rms_norm_kernel<ActF32, false>), dim3(a.num_tokens, groups), dim3(256), 0, st, a);
  }
  return launch_status();
}
