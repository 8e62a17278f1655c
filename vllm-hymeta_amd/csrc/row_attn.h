// Prompts' portions of the attention over paged rows, keys of up to 192 elements, where the value lies inside the key or is it, one
// key for all heads meets a cap or a bias, or a cap meets a bias (the others: row_pipe.h): included by sink_attn.hip.
#pragma once

#include "row_copy.h"

namespace hymeta {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

constexpr float kLazyMax2 = 8.f;     // the softmax reference may trail a row's maximum by a factor of 2^8

// Grid = the portions' blocks of 128 rows x slices of the keys at most x key/value heads (fastest, so that workgroups without
// rows come last); a row is a (query, head) pair, the heads of a key/value head side by side: they share every key, so that a
// portion of a few tokens fills its blocks and a block's causal edge is one tile.
// Sequences with one row are left to the decode form, but where the step's keys are few (one_launch).
//
// Four waves of 32 rows, keys in tiles of 64 copied to two LDS images without passing registers, the values read transposed
// from the rows as they lie; one barrier per tile; two workgroups on a compute unit, so that one's softmax runs under the
// other's products.  v_mfma_f32_32x32x16 holds the issue port for a quarter of its time, the 16 x 16 form for half, and the
// kernel needs the port for its scores (measured level, with less to read from LDS and fewer registers).  The scores are
// formed relative to the row's running reference, which moves only when a score exceeds it by 2^8 (or at the row's first
// visible key): no maximum across lanes, no subtraction and no pass over the output registers on most tiles.
// Bound by the vector and the matrix pipe in turn, hardly ever busy at once.  8192 rows x 28 heads on a latent of 128 + 64: 1629 ->
// 745 us; key and value in one vector, 4 key/value heads of 128, window of 1024: 357 -> 230.
template <int D, int DV, int Layout>
struct RowShape {
  static constexpr bool Scaled = Layout == HYMETA_KV_SCALED_KEY, Inside = Layout == HYMETA_KV_VALUE_IN_KEY || Scaled, Shared = Layout == HYMETA_KV_SHARED_KEY;
  static constexpr int kKeyChunks = D / 8, kValueChunks = Inside ? 0 : DV / 8, kChunks = kKeyChunks + kValueChunks;
  static constexpr int kPitch = 16 * kChunks, kImage = kTileKeys * kPitch;
  static constexpr int kWaves = 4, kRows = 32 * kWaves;
  static_assert(kRows == kPortionRows, "the merge finds a row's block");
};

// How a score follows from its product, in kernels of their own where a design's every layer asks for it: a branch per row
// block in the middle of a tile keeps the compiler from overlapping what stands on its two sides.  (kLogBias, kCapped: row_pipe.h)
enum ScoreRule { kPlain, kLogBias, kCapped, kAnyRule };

template <int D, int DV, int Layout, int Rule>
__global__ __launch_bounds__(256, 2) void row_prefill_kernel(hymeta_sink_attention_args a, PortionSlices ps) {
  static_assert(Rule == kPlain || Rule == kAnyRule, "the others are row_pipe_kernel's");
  typedef RowShape<D, DV, Layout> S;
  constexpr int kSteps = D / 16, CB = DV / 32;
  __shared__ __attribute__((aligned(16))) char s_rows[2][S::kImage];
  __shared__ __attribute__((aligned(16))) float s_scale[2][S::Scaled ? kTileKeys : 4];
  const int group = a.num_heads / a.num_kv_heads, g = blockIdx.x % a.num_kv_heads, item = blockIdx.x / a.num_kv_heads, split = item % ps.splits;
  const PieceAt block = portion_block(a, item / ps.splits, ps);
  const int s = block.seq, row0 = block.row0, q = block.rows, rows = q * group;
  if (s < 0) return;
  const int r0 = ((rows - 1) / S::kRows - block.index) * S::kRows;        // (the longest rows first)
  const int lane = threadIdx.x & 63, n = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ctx = a.seq_lens[s] - q, w0 = r0 + 32 * wave;
  const BlockKeys keys = block_keys<kTileKeys>(a, ctx + r0 / group, ctx + (min(rows, r0 + S::kRows) - 1) / group);
  const int splits = keys.slices(ps);
  if (split >= splits) return;

  // this lane's row; it holds the row's scores against half of a tile's keys, its partner lane +- 32 the others
  const int r = w0 + n;
  const bool ok = r < rows;
  const int qi = ok ? r / group : 0, h = g * group + (ok ? r % group : 0);
  const int pos = ok ? ctx + qi : -1;
  float ba = a.bias_mode ? -a.bias_a[h] : 0.f;
  if (S::Scaled) ba *= 1.4426950408889634f;
  const float bb = a.bias_mode == HYMETA_BIAS_LOG_DISTANCE ? a.bias_b[h] : 0.f;
  const bool sink = a.sink && splits == 1;            // (of several slices of the keys none has the sink: the merge adds it)
  float m = sink ? (a.sink_logits ? a.sink_logits[h] * 1.4426950408889634f : 0.f) : -INFINITY;
  float l = sink && hh == 0 ? 1.f : 0.f;              // the sink's exp(m - m), counted once per row
  bf16x8 qf[kSteps];
  {
    const uint16_t* qrow = static_cast<const uint16_t*>(a.q) + static_cast<int64_t>(row0 + qi) * a.q_stride_t + static_cast<int64_t>(h) * D;
#pragma unroll
    for (int st = 0; st < kSteps; ++st) qf[st] = ok ? __builtin_bit_cast(bf16x8, ld16g(qrow + 16 * st + 8 * hh)) : bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
  }
  f32x16 o[CB];                                       // O^T: columns 32 cb + 8 i + 4 hh + e of the lane's row, i, e < 4
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[cb][i] = 0.f;
  // positions the block's and the wave's rows span
  const int p_hi = ctx + (min(rows, r0 + S::kRows) - 1) / group;
  const int w_lo = ctx + min(rows - 1, w0) / group, w_hi = ctx + min(rows - 1, w0 + 31) / group;
  const int w_first_lo = first_key(a, w_lo), w_first_hi = first_key(a, w_hi);
  const bool full = w0 + 32 <= rows, any = w0 < rows;
  const int per = (keys.tiles + splits - 1) / splits, t_lo = split * per, t_hi = min(keys.tiles, t_lo + per);
  auto key0 = [&](int t) { return keys.first(t); };

  const ScaledRow lay = scaled_row(a.num_kv_heads, D, 2);
  const int64_t row_elems = S::Scaled ? lay.elems : S::Shared ? D + static_cast<int64_t>(a.num_kv_heads) * DV : static_cast<int64_t>(a.num_kv_heads) * (S::Inside ? D : D + DV);
  const int64_t key_elems = S::Shared ? 0 : static_cast<int64_t>(g) * (S::Inside ? D : D + DV);
  const int32_t* bt = a.block_tables + static_cast<int64_t>(s) * a.block_table_stride;
  const RowCopy<S::kKeyChunks, S::kValueChunks, kTileKeys, S::kWaves> copy(a.kv_cache, 2 * row_elems, 2 * key_elems, 2 * (D + (S::Shared ? g * DV : 0)), a.block_size, bt, wave);
  float rs = 0.f;                                     // (scaled keys) the factor of key threadIdx.x of the next tile
  auto issue = [&](int t, char* image) {
    const int j0 = key0(t);
    if (S::Scaled && threadIdx.x < kTileKeys) {
      const int j = min(j0 + static_cast<int>(threadIdx.x), p_hi);
      const int64_t row = (static_cast<int64_t>(bt[j >> copy.shift]) << copy.shift) + (j & copy.mask);
      rs = reinterpret_cast<const float*>(static_cast<const char*>(a.kv_cache) + row * copy.row_bytes + lay.scale_bytes)[g];
    }
    copy.issue(j0, p_hi, image);
  };
  // LDS offsets of this lane's fragments.  Keys: row n, chunk 2 st + hh.  Values: a tile's 16-key step i takes its keys 8 i + 4 hh
  // + e and 32 keys further on, which are the keys whose weights the lane holds
  constexpr int kValueAt = S::Inside ? 0 : S::kKeyChunks;
  int koff[8], voff[2][CB];
#pragma unroll
  for (int i = 0; i < 8; ++i) koff[i] = n * S::kPitch + 16 * ((2 * i + hh) ^ ChunkOrder<S::kChunks>::twist(n));
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      const int R = 8 * i + 4 * hh + ((lane & 15) >> 2), chunk = kValueAt + 4 * cb + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
      voff[i][cb] = R * S::kPitch + 16 * (chunk ^ ChunkOrder<S::kChunks>::twist(R)) + 8 * (lane & 1);
    }
  const float scale2 = a.scale * 1.4426950408889634f, cap_in = a.softcap > 0.f ? a.scale / a.softcap : 0.f, cap2 = a.softcap * 1.4426950408889634f;

  auto attend = [&](int j0, const char* img, const float* scales) {
    f32x16 sc[2];                                     // keys j0 + 32 t + 8 i + 4 hh + e: element 4 i + e of sc[t]
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) sc[t][i] = 0.f;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int st = 0; st < kSteps; ++st)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        sc[t] = mfma32(__builtin_bit_cast(bf16x8, ld16(img + koff[st & 7] + t * 32 * S::kPitch + (st >> 3) * 256)), qf[st], sc[t]);
    __builtin_amdgcn_s_setprio(0);
    const bool masked = !(full && j0 + kTileKeys - 1 <= w_lo && j0 >= w_first_hi);
    const float ref = m == -INFINITY ? 0.f : m;
    // the scores, in the base-2 domain, less the reference (the logarithm's argument from the exact distance: formed from
    // the tile's it would lose 64 of the coefficient's ulps, on the nearest keys of a steep bias all of itself)
    const float d0 = static_cast<float>(pos - j0 - 4 * hh), slope = fmaf(ba, d0, -ref);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f32x4v f;
        if (S::Scaled) f = *reinterpret_cast<const f32x4v*>(scales + 32 * t + 8 * i + 4 * hh) * scale2;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float x = sc[t][4 * i + e];
          const float away = static_cast<float>(32 * t + 8 * i + e);
          if (S::Scaled) x = fmaf(x, f[e], fmaf(-ba, away, slope));
          else if (Rule == kPlain) x = fmaf(x, scale2, -ref);
          sc[t][4 * i + e] = x;
        }
      }
    if (Rule == kAnyRule) {
      if (a.softcap > 0.f) {
#pragma unroll
        for (int i = 0; i < 32; ++i) sc[i >> 4][i & 15] = fmaf(cap2, tanh_fast(sc[i >> 4][i & 15] * cap_in), -ref);
      } else {
#pragma unroll
        for (int i = 0; i < 32; ++i) sc[i >> 4][i & 15] = fmaf(sc[i >> 4][i & 15], scale2, -ref);
      }
      if (a.bias_mode == HYMETA_BIAS_LOG_DISTANCE) {
#pragma unroll
        for (int i = 0; i < 32; ++i)
          sc[i >> 4][i & 15] = fmaf(ba, __builtin_amdgcn_logf(fmaf(bb, d0 - static_cast<float>(32 * (i >> 4) + 8 * ((i & 15) >> 2) + (i & 3)), 1.f)), sc[i >> 4][i & 15]);
      }
    }
    if (masked) {
      const int first = first_key(a, pos);
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        const int j = j0 + 32 * (i >> 4) + 8 * ((i & 15) >> 2) + 4 * hh + (i & 3);
        sc[i >> 4][i & 15] = (j <= pos && (j >= first || j < a.keep_first)) ? sc[i >> 4][i & 15] : -INFINITY;
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 32; ++i) mx = fmaxf(mx, sc[i >> 4][i & 15]);
    if (__any(mx > kLazyMax2 || (m == -INFINITY && mx > -INFINITY))) {
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const bool unset = m == -INFINITY, up = mx > kLazyMax2 || (unset && mx > -INFINITY);
      const float step = up ? mx : 0.f, corr = up ? (unset ? 0.f : __builtin_amdgcn_exp2f(-mx)) : 1.f;
      if (up) m = ref + mx;
      l *= corr;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) o[cb] *= corr;
#pragma unroll
      for (int i = 0; i < 32; ++i) sc[i >> 4][i & 15] -= step;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {                     // 16 keys: e < 4 of sc[0], then of sc[1]
      u32x4 hi, lo;                                   // the weights' bf16 parts, as the second product's fragment
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p0 = __builtin_amdgcn_exp2f(sc[e >> 1][4 * i + 2 * (e & 1)]), p1 = __builtin_amdgcn_exp2f(sc[e >> 1][4 * i + 2 * (e & 1) + 1]);
        l += p0 + p1;
        hi[e] = pack_bf16x2(p0, p1);
        lo[e] = pack_bf16x2(p0 - lo_bf(hi[e]), p1 - hi_bf(hi[e]));
      }
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        const char* v = img + voff[i & 1][cb] + (i >> 1) * 16 * S::kPitch;
        const bf16x4 v0 = read_transposed(v), v1 = read_transposed(v + 32 * S::kPitch);
        const bf16x8 vf = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
        o[cb] = mfma32(vf, __builtin_bit_cast(bf16x8, hi), o[cb]);
        o[cb] = mfma32(vf, __builtin_bit_cast(bf16x8, lo), o[cb]);
      }
      __builtin_amdgcn_s_setprio(0);
    }
  };

  if (t_lo < t_hi) issue(t_lo, s_rows[t_lo & 1]);
  for (int t = t_lo; t < t_hi; ++t) {
    if (S::Scaled && threadIdx.x < kTileKeys) s_scale[t & 1][threadIdx.x] = rs;
    copies_landed_barrier();                          // tile t is there, and everybody is done with tile t - 1
    if (t + 1 < t_hi) issue(t + 1, s_rows[(t + 1) & 1]);
    const int j0 = key0(t);
    if (any && j0 <= w_hi && !(j0 + kTileKeys - 1 < w_first_lo && j0 >= a.keep_first)) attend(j0, s_rows[t & 1], s_scale[t & 1]);
  }
  l += __shfl_xor(l, 32, 64);
  if (!ok) return;
  const int64_t token = row0 + qi;
  if (splits > 1) {
    float* part = ps.parts + ((token * a.num_heads + h) * ps.splits + split) * partial_row_floats(DV);
    if (hh == 0) part[DV] = m, part[DV + 1] = l;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4v*>(part + 32 * cb + 8 * i + 4 * hh) = f32x4v{o[cb][4 * i], o[cb][4 * i + 1], o[cb][4 * i + 2], o[cb][4 * i + 3]};
    return;
  }
  float inv = l > 0.f ? 1.f / l : 0.f;
  if (a.head_gate) inv *= sigmoid_exact(bf2f(static_cast<const uint16_t*>(a.head_gate)[token * a.head_gate_stride_t + h]));
  uint16_t* out = static_cast<uint16_t*>(a.out) + (token * a.num_heads + h) * DV;
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int col = 32 * cb + 8 * i + 4 * hh;
      f32x4v v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = o[cb][4 * i + e] * inv;
      if (a.elem_gate) {
        float gate[4];
        ActBf16::ld4(static_cast<const uint16_t*>(a.elem_gate) + token * a.elem_gate_stride_t + static_cast<int64_t>(h) * DV + col, gate);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= ActBf16::sigmoid(gate[e]);
      }
      *reinterpret_cast<u32x2*>(out + col) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    }
}

}  // namespace
}  // namespace hymeta
