// Causal paged attention with a distance bias and a sink, for any head size, fp32 or bf16 rows:
// the per-head query / key norm with the paged key / value write, and the attention itself.
//
// Scores, the running maximum, the weights and the weighted sum of the values are fp32 whatever the
// activation type.  The sink is a key of score 0 without a value: the running maximum starts at 0
// and the denominator at exp(0 - 0) = 1, everything else is the ordinary streaming softmax.
//
// Rows of HYMETA_KV_SCALED_KEY hold ONE vector per key/value head that is both: the projected key, which is the value,
// and its inverse root mean square, by which the score of the normed key differs from the score of the stored one (the
// norm's weight rides in the queries).  A page then holds half of what keys and values apart would take.
#include <algorithm>

#include "act_types.h"
#include "row_copy.h"

namespace hymeta {

namespace {

constexpr int kMaxHeadDim = 4096;
constexpr int kMaxVChunks = 8;       // value size <= 512

// grid = tokens; a wave per (token, head) task: query heads, then key heads, then value heads.
template <typename A>
__global__ __launch_bounds__(256) void qk_norm_cache_kernel(hymeta_qk_norm_cache_args a) {
  typedef typename A::elem elem;
  const int64_t t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int H = a.num_heads, G = a.num_kv_heads, D = a.head_dim, Dv = a.v_dim;
  elem* row = static_cast<elem*>(a.qkv) + t * a.qkv_stride_t;
  const int64_t slot = a.slot_mapping ? a.slot_mapping[t] : -1;
  const bool store = slot >= 0 && slot < a.num_blocks * a.block_size;
  elem* cache = static_cast<elem*>(a.kv_cache) + (store ? slot : 0) * G * static_cast<int64_t>(D + Dv);
  for (int task = wave; task < H + 2 * G; task += 4) {
    if (task < H + G) {
      const bool is_q = task < H;
      elem* src = row + static_cast<int64_t>(task) * D;          // q heads, then k heads, contiguous
      const float* w = is_q ? a.q_weight : a.k_weight;
      if (!is_q && !store && w == nullptr) continue;
      float inv = 1.f;
      if (w != nullptr) {
        float ss = 0.f;
        for (int d = lane; d < D; d += 64) {
          const float v = A::ld(src + d);
          ss += v * v;
        }
        ss = wave_sum(ss);
        inv = 1.f / sqrtf(ss / static_cast<float>(D) + a.eps);
      }
      elem* dst = is_q ? src : cache + static_cast<int64_t>(task - H) * (D + Dv);
      if (is_q && w == nullptr) continue;
      if (!is_q && !store) continue;
      for (int d = lane; d < D; d += 64) {
        const float v = A::ld(src + d);
        A::st(dst + d, w ? v * inv * w[d] : v);
      }
    } else if (store) {
      const int g = task - H - G;
      const elem* src = row + static_cast<int64_t>(H + G) * D + static_cast<int64_t>(g) * Dv;
      elem* dst = cache + static_cast<int64_t>(g) * (D + Dv) + D;
      for (int d = lane; d < Dv; d += 64) dst[d] = src[d];
    }
  }
}

// A row of HYMETA_KV_SCALED_KEY: num_kv_heads keys of head_dim elements, then (from the next multiple of 4 bytes on) an
// fp32 scale per key/value head, the whole padded to 16 bytes.
struct ScaledRow {
  int64_t elems;          // elements of the activation type per row
  int64_t scale_bytes;    // where the scales start, in bytes
};
__host__ __device__ inline ScaledRow scaled_row(int num_kv_heads, int head_dim, int elem_bytes) {
  const int64_t at = (static_cast<int64_t>(num_kv_heads) * head_dim * elem_bytes + 3) / 4 * 4;
  return ScaledRow{(at + 4 * static_cast<int64_t>(num_kv_heads) + 15) / 16 * 16 / elem_bytes, at};
}

// grid = tokens.  `Lanes` neighbouring lanes (a power of two) share a head, four elements each (Vec), or the lanes of a wave
// stride over it: query heads (normed, times q_weight, k_weight and the temperature of the row's position, in place), then
// key heads (stored as they are, with their inverse root mean square).
template <typename A, bool Vec>
__global__ __launch_bounds__(256) void scaled_key_cache_kernel(hymeta_scaled_key_cache_args a, int lanes) {
  typedef typename A::elem elem;
  const int64_t t = blockIdx.x;
  const int H = a.num_heads, G = a.num_kv_heads, D = a.head_dim;
  const int sub = threadIdx.x & (lanes - 1), first = threadIdx.x / lanes, step = 256 / lanes;
  elem* row = static_cast<elem*>(a.qk) + t * a.qk_stride_t;
  const int64_t slot = a.slot_mapping ? a.slot_mapping[t] : -1;
  const bool store = slot >= 0 && slot < a.num_blocks * a.block_size;
  const ScaledRow lay = scaled_row(G, D, sizeof(elem));
  elem* cache = store ? static_cast<elem*>(a.kv_cache) + slot * lay.elems : nullptr;
  float temp = 1.f;
  if (a.temp_coef != 0.f) {
    // floor of the exact quotient: a double holds positions and periods exactly, and no quotient of two of them rounds up
    // to the next integer
    const double n = floor((static_cast<double>(a.positions[t]) + 1.0) / a.temp_every) + 1.0;
    temp = 1.f + a.temp_coef * logf(static_cast<float>(n));
  }
  for (int task = first; task < H + G; task += step) {
    const bool is_q = task < H;
    elem* src = row + static_cast<int64_t>(task) * D;
    float ss = 0.f, v[4];
    if (Vec) {
      const bool on = 4 * sub < D;
      if (on) A::ld4(src + 4 * sub, v);
#pragma unroll
      for (int e = 0; e < 4; ++e) ss = on ? fmaf(v[e], v[e], ss) : ss;
    } else {
      for (int d = sub; d < D; d += lanes) {
        const float x = A::ld(src + d);
        ss = fmaf(x, x, ss);
      }
    }
    for (int o = lanes >> 1; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
    const float inv = 1.f / sqrtf(ss / static_cast<float>(D) + a.eps);
    if (is_q) {
      const float f = inv * temp;
      if (Vec) {
        if (4 * sub < D) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] *= f * a.q_weight[4 * sub + e] * a.k_weight[4 * sub + e];
          A::st4(src + 4 * sub, v);
        }
      } else {
        for (int d = sub; d < D; d += lanes) A::st(src + d, A::ld(src + d) * f * a.q_weight[d] * a.k_weight[d]);
      }
    } else if (store) {
      const int g = task - H;
      elem* dst = cache + static_cast<int64_t>(g) * D;
      if (Vec) {
        if (4 * sub < D) A::st4(dst + 4 * sub, v);
      } else {
        for (int d = sub; d < D; d += lanes) dst[d] = src[d];
      }
      if (sub == 0) reinterpret_cast<float*>(reinterpret_cast<char*>(cache) + lay.scale_bytes)[g] = inv;
    }
  }
}

__device__ __forceinline__ float distance_bias(int mode, float a, float b, int dist) {
  if (mode == HYMETA_BIAS_LINEAR_DISTANCE) return a * static_cast<float>(dist);
  return mode == HYMETA_BIAS_LOG_DISTANCE ? a * log1pf(b * static_cast<float>(dist)) : 0.f;
}

// First key a query at position pos sees: `window_left` tokens back, or the start of its chunk of `chunk` tokens (counted from
// the sequence's first token), or the sequence's first.  Never decreases with pos.
__host__ __device__ __forceinline__ bool bounded(const hymeta_sink_attention_args& a) { return a.window_left >= 0 || a.chunk > 0; }
__device__ __forceinline__ int first_key(const hymeta_sink_attention_args& a, int pos) {
  if (a.chunk > 0) return pos / a.chunk * a.chunk;
  return a.window_left >= 0 ? max(0, pos - a.window_left) : 0;
}

// One wave per (query row, head).  Keys in tiles of 64: lane = key for the scores, lane = value channel for the
// weighted sum, the tile's weights and row addresses handed over through LDS.
template <typename A>
__global__ __launch_bounds__(64) void sink_attention_rows_kernel(hymeta_sink_attention_args a) {
  typedef typename A::elem elem;
  __shared__ float s_q[kMaxHeadDim];
  __shared__ float s_p[64];
  __shared__ int64_t s_row[64];
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int D = a.head_dim, Dv = a.v_dim, G = a.num_kv_heads;
  const int g = h / (a.num_heads / G);
  const int s = seq_of_row(a.query_start_loc, a.num_seqs, t);
  const int pos = a.seq_lens[s] - (a.query_start_loc[s + 1] - t);
  if (pos < 0) return;
  const int first = first_key(a, pos);
  const elem* q = static_cast<const elem*>(a.q) + static_cast<int64_t>(t) * a.q_stride_t + static_cast<int64_t>(h) * D;
  for (int d = lane; d < D; d += 64) s_q[d] = A::ld(q + d);
  const int32_t* bt = a.block_tables + static_cast<int64_t>(s) * a.block_table_stride;
  const elem* cache = static_cast<const elem*>(a.kv_cache);
  // where the head's key and value lie in a cache row: a key followed by its value per key/value head; a key whose first Dv
  // elements are the value; or one key for all heads followed by the key/value heads' values
  int64_t row_elems, key_off, val_off;
  const bool scaled = a.kv_layout == HYMETA_KV_SCALED_KEY;
  const ScaledRow lay = scaled_row(G, D, sizeof(elem));
  if (scaled) row_elems = lay.elems, key_off = static_cast<int64_t>(g) * D, val_off = key_off;
  else if (a.kv_layout == HYMETA_KV_SHARED_KEY) row_elems = D + static_cast<int64_t>(G) * Dv, key_off = 0, val_off = D + static_cast<int64_t>(g) * Dv;
  else if (a.kv_layout == HYMETA_KV_VALUE_IN_KEY) row_elems = static_cast<int64_t>(G) * D, key_off = static_cast<int64_t>(g) * D, val_off = key_off;
  else row_elems = static_cast<int64_t>(G) * (D + Dv), key_off = static_cast<int64_t>(g) * (D + Dv), val_off = key_off + D;
  const float ba = a.bias_mode ? a.bias_a[h] : 0.f, bb = a.bias_mode == HYMETA_BIAS_LOG_DISTANCE ? a.bias_b[h] : 0.f;
  // the sink: a key of score sink_logits[h] (0 without) that has no value
  float m = a.sink ? (a.sink_logits ? a.sink_logits[h] : 0.f) : -INFINITY, l = a.sink ? 1.f : 0.f;
  float acc[kMaxVChunks] = {};
  const int nvc = (Dv + 63) / 64;
  __syncthreads();
  // two runs of keys: the kept first ones that lie before the window, then the window
  const int kept = a.window_left >= 0 ? min(a.keep_first, first) : 0;
  for (int run = 0; run < 2; ++run) {
    const int lo = run == 0 ? 0 : first, hi = run == 0 ? kept - 1 : pos;
    for (int j0 = lo; j0 <= hi; j0 += 64) {
      const int j = j0 + lane;
      const bool valid = j <= hi;
      float sc = -INFINITY;
      int64_t roff = 0;
      if (valid) {
        const int64_t blk = bt[j / a.block_size];
        roff = (blk * a.block_size + j % a.block_size) * row_elems;
        const elem* k = cache + roff + key_off;
        float dot = 0.f;
        for (int d = 0; d < D; ++d) dot = fmaf(s_q[d], A::ld(k + d), dot);
        if (scaled) dot *= reinterpret_cast<const float*>(reinterpret_cast<const char*>(cache + roff) + lay.scale_bytes)[g];
        sc = dot * a.scale;
        if (a.softcap > 0.f) sc = a.softcap * tanhf(sc / a.softcap);
        sc -= distance_bias(a.bias_mode, ba, bb, pos - j);
      }
      const float m_new = fmaxf(m, wave_max(sc));
      const float p = valid ? expf(sc - m_new) : 0.f;
      const float corr = expf(m - m_new);            // m = -inf only without a sink before the first tile: corr = 0, l = 0
      l = l * corr + wave_sum(p);
      m = m_new;
      __syncthreads();
      s_p[lane] = p;
      s_row[lane] = roff + val_off;
      __syncthreads();
      const int n = min(64, hi - j0 + 1);
#pragma unroll
      for (int cc = 0; cc < kMaxVChunks; ++cc) {
        if (cc < nvc) {
          const int c = cc * 64 + lane;
          float r = acc[cc] * corr;
          if (c < Dv)
            for (int jj = 0; jj < n; ++jj) r = fmaf(s_p[jj], A::ld(cache + s_row[jj] + c), r);
          acc[cc] = r;
        }
      }
    }
  }
  elem* out = static_cast<elem*>(a.out) + (static_cast<int64_t>(t) * a.num_heads + h) * Dv;
  float inv = l > 0.f ? 1.f / l : 0.f;
  if (a.head_gate) inv *= sigmoid_exact(A::ld(static_cast<const elem*>(a.head_gate) + static_cast<int64_t>(t) * a.head_gate_stride_t + h));
#pragma unroll
  for (int cc = 0; cc < kMaxVChunks; ++cc) {
    const int c = cc * 64 + lane;
    if (cc < nvc && c < Dv) {
      float v = acc[cc] * inv;
      if (a.elem_gate) v *= sigmoid_exact(A::ld(static_cast<const elem*>(a.elem_gate) + static_cast<int64_t>(t) * a.elem_gate_stride_t + static_cast<int64_t>(h) * Dv + c));
      A::st(out + c, v);
    }
  }
}


// ------------------------------------------------------------------------------------------------
// bf16 on the matrix cores.  A wave owns 32 "rows" (two blocks of 16): in a prompt's portion 32 consecutive query
// rows of one head, in a decode step the query heads of one key/value head (they share every key and value row they
// read).  Keys come in tiles of 64 through LDS: the key rows as they lie in the pages, the value rows transposed, so
// that both are read as MFMA operands with 8- and 16-byte LDS loads.
//
//   S^T[key][row] = K[key][:] . Q[row][:]           v_mfma_f32_16x16x32_bf16, A = K fragment, B = Q fragment
//   O^T[c][row]  += V^T[c][key] P^T[key][row]       A = V^T fragment, B = P^T
//
// The transposed forms make the result layout of the first product (a lane holds 4 consecutive keys of one row) the
// B-operand layout of the second, so the weights never leave their registers, and they leave the row statistics in the
// lane that owns the row in both products.  The weights stay fp32-exact through the bf16 matrix product: p = hi + lo
// with hi = bf16(p), lo = bf16(p - hi), two products (relative error of p 2^-17 instead of 2^-9).
// ------------------------------------------------------------------------------------------------
typedef float f32x4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4v mfma16(bf16x8 a, bf16x8 b, f32x4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

constexpr int kTileKeys = 64;
constexpr int kRowsPerWave = 32;

// (decode form) the query heads of a key/value head one launch takes as its rows: first .. first + count of the group;
// count 0: the whole group.  Groups of more than 32 heads run as several launches.
struct HeadSlice {
  int first = 0, count = 0;
};

template <int D, int DV>
struct MfmaSmem {
  static constexpr int kPitchK = D + 8;               // bf16 elements per key row (16-byte reads of 16 rows: no bank conflict)
  static constexpr int kPitchV = kTileKeys + 8;       // bf16 elements per value channel
  uint16_t k[kTileKeys * kPitchK];
  uint16_t vt[DV * kPitchV];
};

// Staging of keys [j0, j0 + 64) of a sequence's key/value head g, in two halves so that the loads of the next tile
// are in flight while the current one is multiplied: `issue` reads 16-byte chunks into registers (keys past `last` read
// as zero), `commit` stores them into LDS.  A key row goes in as it is.  The value rows go in transposed: a thread takes
// the same 8 channels of 4 consecutive keys (4 chunks), which are 8 runs of 4 keys in the transposed image, one 8-byte
// store each.  The 4-key groups of a channel are permuted by the channel's chunk number (XOR), which spreads the stores
// of threads that hold the same keys over the banks; the reader applies the same permutation.
// Layout (enum hymeta_kv_layout).  VALUE_IN_KEY: a head's part of a cache row is its key alone (D elements), whose first DV
// elements are also its value.  SHARED_KEY: a row is one key of D elements for all heads, then num_kv_heads values of DV.
// SCALED_KEY: a head's part is one vector that is key and value (D == DV), read from memory once and stored into both images,
// and the keys' scales go into an array of their own.
template <int D, int DV, int Threads, int Layout>
struct TileStage {
  static constexpr bool VinK = Layout == HYMETA_KV_VALUE_IN_KEY, Shared = Layout == HYMETA_KV_SHARED_KEY;
  static constexpr bool Scaled = Layout == HYMETA_KV_SCALED_KEY;
  static constexpr int kKeyChunksPerRow = D / 8, kValChunksPerRow = DV / 8;
  static constexpr int kKeyChunks = kTileKeys * kKeyChunksPerRow;
  static constexpr int kKeyPerThread = (kKeyChunks + Threads - 1) / Threads;
  static constexpr int kValBlocks = (kTileKeys / 4) * kValChunksPerRow;       // (4 keys) x (8 channels) each
  static constexpr int kHeadElems = (VinK || Scaled) ? D : D + DV, kValueAt = (VinK || Scaled) ? 0 : D;
  static_assert(D % 32 == 0 && DV % 16 == 0 && kValBlocks <= Threads && (!VinK || DV <= D) && (!Scaled || DV == D) && kTileKeys <= Threads,
                "the staging roles fit the workgroup");
  u32x4 rk[Scaled ? 1 : kKeyPerThread];
  u32x4 rv[4];
  float rs = 0.f;               // (SCALED_KEY) the scale of key j0 + threadIdx.x
  int value_at = kValueAt;      // where the value starts in a head's part of a row

  // Pages hold a power of two of rows here (the host sends other sizes to the plain kernel).  A page of 64 rows or more
  // holds a whole tile (tiles start at multiples of 64): its number is one scalar load per tile, not a dependent vector
  // load in front of every row's loads.
  struct Pages {
    const uint16_t* cache;
    const int32_t* bt;
    int64_t row_elems, head_off;
    int shift, mask;
    int64_t tile_base;          // first row of the tile's page, in rows of the cache (pages of >= 64 rows)
    bool whole;
  };

  static __device__ __forceinline__ Pages pages(const hymeta_sink_attention_args& a, const int32_t* bt, int g, int j0) {
    Pages p;
    p.cache = static_cast<const uint16_t*>(a.kv_cache);
    p.bt = bt;
    p.row_elems = Scaled ? scaled_row(a.num_kv_heads, D, 2).elems : Shared ? D + static_cast<int64_t>(a.num_kv_heads) * DV : static_cast<int64_t>(a.num_kv_heads) * kHeadElems;
    p.head_off = Shared ? 0 : static_cast<int64_t>(g) * kHeadElems;
    p.shift = __builtin_ctz(a.block_size);
    p.mask = a.block_size - 1;
    p.whole = a.block_size >= kTileKeys;
    p.tile_base = 0;
    if (p.whole) p.tile_base = (static_cast<int64_t>(__builtin_amdgcn_readfirstlane(bt[j0 >> p.shift])) << p.shift) + (j0 & p.mask);
    return p;
  }

  static __device__ __forceinline__ const uint16_t* row_ptr(const Pages& p, int j0, int j) {
    const int64_t row = p.whole ? p.tile_base + (j - j0) : (static_cast<int64_t>(p.bt[j >> p.shift]) << p.shift) + (j & p.mask);
    return p.cache + row * p.row_elems + p.head_off;
  }

  __device__ __forceinline__ void issue(const hymeta_sink_attention_args& a, const int32_t* bt, int g, int j0, int last) {
    const Pages p = pages(a, bt, g, j0);
    if constexpr (Scaled) {
      const int j = j0 + static_cast<int>(threadIdx.x);
      rs = 0.f;
      if (static_cast<int>(threadIdx.x) < kTileKeys && j <= last)
        rs = reinterpret_cast<const float*>(reinterpret_cast<const char*>(row_ptr(p, j0, j) - p.head_off) + scaled_row(a.num_kv_heads, D, 2).scale_bytes)[g];
    } else {
#pragma unroll
      for (int i = 0; i < kKeyPerThread; ++i) {
        const int idx = i * Threads + threadIdx.x;
        const int j = j0 + idx / kKeyChunksPerRow;
        rk[i] = u32x4{0u, 0u, 0u, 0u};
        if (j <= last && (kKeyChunks % Threads == 0 || idx < kKeyChunks)) rk[i] = ld16g(row_ptr(p, j0, j) + (idx % kKeyChunksPerRow) * 8);
      }
    }
    if (static_cast<int>(threadIdx.x) < kValBlocks) {
      const int ch = threadIdx.x % kValChunksPerRow, grp = threadIdx.x / kValChunksPerRow;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = j0 + 4 * grp + i;
        rv[i] = u32x4{0u, 0u, 0u, 0u};
        if (j <= last) rv[i] = ld16g(row_ptr(p, j0, j) + value_at + ch * 8);
      }
    }
  }

  __device__ __forceinline__ void commit(MfmaSmem<D, DV>& sm, float* scales) const {
    if constexpr (Scaled) {
      if (static_cast<int>(threadIdx.x) < kTileKeys) scales[threadIdx.x] = rs;
      if (static_cast<int>(threadIdx.x) < kValBlocks) {
        const int ch = threadIdx.x % kValChunksPerRow, grp = threadIdx.x / kValChunksPerRow;
#pragma unroll
        for (int i = 0; i < 4; ++i) st16(&sm.k[(4 * grp + i) * MfmaSmem<D, DV>::kPitchK + ch * 8], rv[i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < kKeyPerThread; ++i) {
        const int idx = i * Threads + threadIdx.x;
        if (kKeyChunks % Threads == 0 || idx < kKeyChunks)
          st16(&sm.k[(idx / kKeyChunksPerRow) * MfmaSmem<D, DV>::kPitchK + (idx % kKeyChunksPerRow) * 8], rk[i]);
      }
    }
    if (static_cast<int>(threadIdx.x) < kValBlocks) {
      const int ch = threadIdx.x % kValChunksPerRow, grp = threadIdx.x / kValChunksPerRow;
      uint16_t* dst = &sm.vt[(8 * ch) * MfmaSmem<D, DV>::kPitchV + 4 * (grp ^ (ch & 15))];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int dw = e >> 1;
        u32x2 v;
        if (e & 1) {
          v[0] = (rv[0][dw] >> 16) | (rv[1][dw] & 0xffff0000u);
          v[1] = (rv[2][dw] >> 16) | (rv[3][dw] & 0xffff0000u);
        } else {
          v[0] = (rv[0][dw] & 0xffffu) | (rv[1][dw] << 16);
          v[1] = (rv[2][dw] & 0xffffu) | (rv[3][dw] << 16);
        }
        *reinterpret_cast<u32x2*>(dst + e * MfmaSmem<D, DV>::kPitchV) = v;
      }
    }
  }
};

// Where the 4-key group `grp` (0 .. 15) of value channel c lies in the transposed image.
template <int D, int DV>
__device__ __forceinline__ const uint16_t* vt_group(const MfmaSmem<D, DV>& sm, int c, int grp) {
  return &sm.vt[c * MfmaSmem<D, DV>::kPitchV + 4 * (grp ^ ((c >> 3) & 15))];
}

// The rows of one wave against the staged tile.  RB row blocks of 16 (row = 16 rb + lane % 16); the wave takes NKS of the
// tile's four 16-key subtiles, from ks_lo on (a prompt's wave all four, a decode wave one: the four waves of a decode
// workgroup split every tile between them and each keeps statistics of its own).
template <int D, int DV, int RB>
struct WaveRows {
  bf16x8 q[RB][D / 32];
  f32x4v o[RB][DV / 16];
  float m[RB], l[RB];          // running maximum of the row; this lane's share of the denominator
  int pos[RB];                 // position of the row's query (-1: no such row)
  int first[RB];               // the first key it sees
  float ba[RB], bb[RB];
};

// tanh through the hardware's exponential: 1 - 2 / (exp(2 x) + 1), exact at both ends (exp2 -> inf gives 1, -> 0 gives -1)
__device__ __forceinline__ float tanh_fast(float x) {
  return 1.f - 2.f * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x * 2.8853900817779268f) + 1.f);
}

// Scaled (SCALED_KEY rows): `scales` holds a factor per key of the tile, the bias is linear in the distance (its
// coefficient, in the base-2 domain, in w.ba) and there is no cap.
template <int D, int DV, int RB, int NKS, bool Masked, bool Scaled>
__device__ __forceinline__ void attend_tile(WaveRows<D, DV, RB>& w, const MfmaSmem<D, DV>& sm, const float* scales,
                                            const hymeta_sink_attention_args& a, int j0, int ks_lo) {
  static_assert(NKS == 4 || NKS == 1, "all of a tile's subtiles or one");
  const int lane = threadIdx.x & 63, n = lane & 15, g4 = lane >> 4;
  constexpr int PK = MfmaSmem<D, DV>::kPitchK;
  f32x4v s[RB][NKS];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) s[rb][ks] = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
    for (int st = 0; st < D / 32; ++st) {
      const bf16x8 kf = __builtin_bit_cast(bf16x8, ld16(&sm.k[(16 * (ks_lo + ks) + n) * PK + 32 * st + 8 * g4]));
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) s[rb][ks] = mfma16(kf, w.q[rb][st], s[rb][ks]);
    }
  // lane holds, per row block, the scores of its row (n) against keys j0 + 16 (ks_lo + ks) + 4 g4 + r.  Everything from
  // here to the weights is in the base-2 domain (scores times log2 e; the bias' coefficient is unchanged, as
  // a ln x * log2 e = a log2 x): one v_log and one v_exp per score and no multiplications around them.  The running
  // maximum, and with it the sink's score 0, mean the same in both domains.
  const float scale2 = a.scale * 1.4426950408889634f;
  const bool bias = a.bias_mode == HYMETA_BIAS_LOG_DISTANCE;
  // capped scores: softcap tanh(score / softcap), moved into the base-2 domain like the others
  const bool capped = a.softcap > 0.f;
  const float cap2 = a.softcap * 1.4426950408889634f, cap_in = capped ? a.scale / a.softcap : 0.f;
  uint32_t phi[RB][NKS][2], plo[RB][NKS][2];       // the weights' bf16 high and low parts, two per dword
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int pos = w.pos[rb];
    // distance of the lane's key r of subtile ks: fd0 - (16 ks + r)
    const float fd0 = static_cast<float>(pos - j0 - 16 * ks_lo - 4 * g4);
    float mx = -INFINITY;
    const float near = -w.ba[rb] * fd0;            // (Scaled) the linear bias of the lane's first key, sign included
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      f32x4v kscale = f32x4v{0.f, 0.f, 0.f, 0.f};
      if (Scaled) kscale = *reinterpret_cast<const f32x4v*>(scales + 16 * (ks_lo + ks) + 4 * g4) * scale2;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float sc;
        if (Scaled) {
          sc = fmaf(s[rb][ks][r], kscale[r], fmaf(w.ba[rb], static_cast<float>(16 * ks + r), near));
        } else {
          sc = s[rb][ks][r] * scale2;
          if (capped) sc = cap2 * tanh_fast(s[rb][ks][r] * cap_in);
          if (bias) sc = fmaf(-w.ba[rb], __log2f(fmaf(w.bb[rb], fd0 - static_cast<float>(16 * ks + r), 1.f)), sc);
        }
        if (Masked) {
          const int j = j0 + 16 * (ks_lo + ks) + 4 * g4 + r;
          sc = (j <= pos && (j >= w.first[rb] || j < a.keep_first)) ? sc : -INFINITY;
        }
        s[rb][ks][r] = sc;
        mx = fmaxf(mx, sc);
      }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(w.m[rb], mx);
    // (masked tiles only) a row with nothing visible so far and no sink keeps m = -inf: weights and correction are 0
    const bool empty = Masked && m_new == -INFINITY;
    const float corr = empty ? 0.f : __builtin_amdgcn_exp2f(w.m[rb] - m_new);
    float sum = 0.f;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
      for (int r2 = 0; r2 < 2; ++r2) {
        float p[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          p[u] = empty ? 0.f : __builtin_amdgcn_exp2f(s[rb][ks][2 * r2 + u] - m_new);
          sum += p[u];
        }
        const uint32_t hi = pack_bf16x2(p[0], p[1]);
        phi[rb][ks][r2] = hi;
        plo[rb][ks][r2] = pack_bf16x2(p[0] - lo_bf(hi), p[1] - hi_bf(hi));
      }
    w.l[rb] = w.l[rb] * corr + sum;
    w.m[rb] = m_new;
#pragma unroll
    for (int cb = 0; cb < DV / 16; ++cb) w.o[rb][cb] *= corr;
  }
  if constexpr (NKS == 4) {
#pragma unroll
    for (int cb = 0; cb < DV / 16; ++cb)
#pragma unroll
      for (int kp = 0; kp < 2; ++kp) {
        // k index 8 g4 + e of the product: keys 16 (2 kp) + 4 g4 + e for e < 4, 16 (2 kp + 1) + 4 g4 + e - 4 after
        const u32x2 v0 = *reinterpret_cast<const u32x2*>(vt_group<D, DV>(sm, 16 * cb + n, 8 * kp + g4));
        const u32x2 v1 = *reinterpret_cast<const u32x2*>(vt_group<D, DV>(sm, 16 * cb + n, 8 * kp + 4 + g4));
        const bf16x8 vf = __builtin_bit_cast(bf16x8, (u32x4{v0[0], v0[1], v1[0], v1[1]}));
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          const bf16x8 ph = __builtin_bit_cast(bf16x8, (u32x4{phi[rb][2 * kp][0], phi[rb][2 * kp][1], phi[rb][2 * kp + 1][0], phi[rb][2 * kp + 1][1]}));
          const bf16x8 pl = __builtin_bit_cast(bf16x8, (u32x4{plo[rb][2 * kp][0], plo[rb][2 * kp][1], plo[rb][2 * kp + 1][0], plo[rb][2 * kp + 1][1]}));
          w.o[rb][cb] = mfma16(vf, ph, w.o[rb][cb]);
          w.o[rb][cb] = mfma16(vf, pl, w.o[rb][cb]);
        }
      }
  } else {
#pragma unroll
    for (int cb = 0; cb < DV / 16; ++cb) {
      const bf16x4 vf = __builtin_bit_cast(bf16x4, *reinterpret_cast<const u32x2*>(vt_group<D, DV>(sm, 16 * cb + n, 4 * ks_lo + g4)));
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const bf16x4 ph = __builtin_bit_cast(bf16x4, (u32x2{phi[rb][0][0], phi[rb][0][1]}));
        const bf16x4 pl = __builtin_bit_cast(bf16x4, (u32x2{plo[rb][0][0], plo[rb][0][1]}));
        w.o[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(vf, ph, w.o[rb][cb], 0, 0, 0);
        w.o[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(vf, pl, w.o[rb][cb], 0, 0, 0);
      }
    }
  }
}

template <int D, int DV, int RB>
__device__ __forceinline__ void load_q(WaveRows<D, DV, RB>& w, int rb, const uint16_t* qrow) {
  const int g4 = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int st = 0; st < D / 32; ++st)
    w.q[rb][st] = qrow ? __builtin_bit_cast(bf16x8, ld16g(qrow + 32 * st + 8 * g4)) : bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
}

// Whether every key of the tile from j0 on is visible to every query position in [p_lo, p_hi] (first_hi: the first key p_hi
// sees) / none of them to any (first_lo: the first key p_lo sees).
__device__ __forceinline__ bool tile_open(int j0, int p_lo, int first_hi) { return j0 + kTileKeys - 1 <= p_lo && j0 >= first_hi; }
__device__ __forceinline__ bool tile_shut(const hymeta_sink_attention_args& a, int j0, int first_lo) {
  return j0 + kTileKeys - 1 < first_lo && j0 >= a.keep_first;
}

// The bias' constants of head h as attend_tile wants them.
template <int D, int DV, int RB>
__device__ __forceinline__ void load_bias(WaveRows<D, DV, RB>& w, int rb, const hymeta_sink_attention_args& a, int h) {
  w.ba[rb] = a.bias_mode ? a.bias_a[h] : 0.f;
  if (a.bias_mode == HYMETA_BIAS_LINEAR_DISTANCE) w.ba[rb] *= 1.4426950408889634f;
  w.bb[rb] = a.bias_mode == HYMETA_BIAS_LOG_DISTANCE ? a.bias_b[h] : 0.f;
}

// Short portions of prompts over few keys, rows of HYMETA_KV_SHARED_KEY with keys of more than 192 elements (more of either:
// row_pipe.h, few_long_keys has the line; shorter keys and other rows: row_attn.h, wide_latent.h): grid = (tiles of 16 rows per wave,
// heads, sequences); sequences of fewer than `least` rows are left to the decode form.  4 waves: the query fragments (D / 8
// registers) and the staging registers do not leave a wave of 8 its accumulators within 256 registers.  Bound by LDS, whose tile
// every wave reads whole for 16 rows: about 5 us a tile of 64 keys of 512, but 5 around them, where row_pipe.h's blocks take 2.8 and 14.
constexpr int kPrefillWaves = 4, kPrefillRows = 16 * kPrefillWaves;

template <int D, int DV>
__global__ __launch_bounds__(64 * kPrefillWaves) void sink_attention_prefill_shared_kernel(hymeta_sink_attention_args a, int least) {
  constexpr int kRows = kPrefillRows;
  constexpr int kImages = 2 * sizeof(MfmaSmem<D, DV>) <= 159 * 1024 ? 2 : 1;        // (160 KB of LDS)
  __shared__ MfmaSmem<D, DV> sm[kImages];
  // (a prompt's later rows see more keys: the row blocks are handed out from the last on, all heads of a block side by side)
  const int lin = blockIdx.x + gridDim.x * blockIdx.y;
  const int s = blockIdx.z, h = lin % gridDim.y, tile = gridDim.x - 1 - lin / gridDim.y;
  const int row0 = a.query_start_loc[s];
  const int q = a.query_start_loc[s + 1] - row0;
  if (q < least || tile * kRows >= q) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 15, g4 = lane >> 4;
  const int g = h / (a.num_heads / a.num_kv_heads);
  const int ctx = a.seq_lens[s] - q;
  const int32_t* bt = a.block_tables + static_cast<int64_t>(s) * a.block_table_stride;
  WaveRows<D, DV, 1> w;
  const int wrow = tile * kRows + wave * 16, r = wrow + n;
  const bool ok = r < q;
  w.pos[0] = ok ? ctx + r : -1;
  w.first[0] = first_key(a, ctx + r);
  load_bias<D, DV, 1>(w, 0, a, h);
  w.m[0] = a.sink ? (a.sink_logits ? a.sink_logits[h] * 1.4426950408889634f : 0.f) : -INFINITY;
  w.l[0] = (a.sink && g4 == 0) ? 1.f : 0.f;          // the sink's exp(m - m), counted once per row
  load_q<D, DV, 1>(w, 0, ok ? static_cast<const uint16_t*>(a.q) + static_cast<int64_t>(row0 + r) * a.q_stride_t + static_cast<int64_t>(h) * D : nullptr);
#pragma unroll
  for (int cb = 0; cb < DV / 16; ++cb) w.o[0][cb] = f32x4v{0.f, 0.f, 0.f, 0.f};
  const int block_last = ctx + min(q, tile * kRows + kRows) - 1;      // last key any row of the block sees
  const int wave_last = ctx + min(q, wrow + 16) - 1;
  const int first_lo = first_key(a, ctx + wrow), first_hi = first_key(a, wave_last);           // of the wave's rows
  const int j_first = first_key(a, ctx + tile * kRows) / kTileKeys * kTileKeys;
  // the tiles of the kept first keys that lie before the window's first tile come first, then the window's
  const int keep_end = bounded(a) ? min((a.keep_first + kTileKeys - 1) / kTileKeys * kTileKeys, j_first) : 0;
  const int j_start = keep_end > 0 ? 0 : j_first;
  auto next = [&](int j0) { return (j0 < keep_end && j0 + kTileKeys >= keep_end) ? j_first : j0 + kTileKeys; };
  // two LDS images: while the waves multiply tile t out of one, tile t + 1 goes into the other and the loads of tile
  // t + 2 are in flight; one barrier per tile
  TileStage<D, DV, 64 * kPrefillWaves, HYMETA_KV_SHARED_KEY> stage;
  stage.value_at = D + g * DV;
  stage.issue(a, bt, g, j_start, block_last);
  stage.commit(sm[0], nullptr);
  if (kImages == 2 && next(j_start) <= block_last) stage.issue(a, bt, g, next(j_start), block_last);
  __syncthreads();
  if constexpr (kImages == 2) {
    int buf = 0;
    for (int j0 = j_start; j0 <= block_last; j0 = next(j0), buf ^= 1) {
      const int j1 = next(j0), j2 = next(j1);
      if (j1 <= block_last) stage.commit(sm[buf ^ 1], nullptr);
      if (j2 <= block_last) stage.issue(a, bt, g, j2, block_last);
      if (wrow < q && j0 <= wave_last && !tile_shut(a, j0, first_lo)) {
        // tiles whose every key is visible to every row of the wave need no mask
        if (tile_open(j0, ctx + wrow, first_hi)) attend_tile<D, DV, 1, 4, false, false>(w, sm[buf], nullptr, a, j0, 0);
        else attend_tile<D, DV, 1, 4, true, false>(w, sm[buf], nullptr, a, j0, 0);
      }
      __syncthreads();
    }
  } else {
    // one image (tiles of long rows): the next tile's loads are in flight while this one is multiplied and go into LDS
    // behind a barrier
    for (int j0 = j_start; j0 <= block_last; j0 = next(j0)) {
      const bool more = next(j0) <= block_last;
      if (more) stage.issue(a, bt, g, next(j0), block_last);
      if (wrow < q && j0 <= wave_last && !tile_shut(a, j0, first_lo)) {
        if (tile_open(j0, ctx + wrow, first_hi)) attend_tile<D, DV, 1, 4, false, false>(w, sm[0], nullptr, a, j0, 0);
        else attend_tile<D, DV, 1, 4, true, false>(w, sm[0], nullptr, a, j0, 0);
      }
      __syncthreads();
      if (more) {
        stage.commit(sm[0], nullptr);
        __syncthreads();
      }
    }
  }
  float l = w.l[0];
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (r >= q) return;
  float inv = l > 0.f ? 1.f / l : 0.f;
  if (a.head_gate) inv *= sigmoid_exact(bf2f(static_cast<const uint16_t*>(a.head_gate)[static_cast<int64_t>(row0 + r) * a.head_gate_stride_t + h]));
  uint16_t* out = static_cast<uint16_t*>(a.out) + (static_cast<int64_t>(row0 + r) * a.num_heads + h) * DV;
#pragma unroll
  for (int cb = 0; cb < DV / 16; ++cb) {
    f32x4v o = w.o[0][cb] * inv;
    if (a.elem_gate) {
      float gate[4];
      ActBf16::ld4(static_cast<const uint16_t*>(a.elem_gate) + static_cast<int64_t>(row0 + r) * a.elem_gate_stride_t + static_cast<int64_t>(h) * DV + 16 * cb + 4 * g4, gate);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] *= ActBf16::sigmoid(gate[e]);
    }
    *reinterpret_cast<u32x2*>(out + 16 * cb + 4 * g4) = u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
  }
}

// Partial of a (sequence, key/value head, slice, wave): per query head of the group DV weighted values, then the
// maximum and denominator, rows padded to whole 16 bytes.
__host__ __device__ inline size_t partial_row_floats(int dv) { return static_cast<size_t>(dv) + 4; }
constexpr int kDecodeWaves = 4;
// LDS images of a decode workgroup: two (the next tile goes into the other image while this one is multiplied) where
// both fit in 72 KB, which leaves two workgroups on a compute unit; one for larger tiles, so that three or four
// workgroups overlap each other instead.
template <int D, int DV>
struct DecodeImages {
  static constexpr int value = 2 * sizeof(MfmaSmem<D, DV>) <= 72 * 1024 ? 2 : 1;
};
// Whether the four waves of a decode workgroup merge their partials through LDS (the tile images, free after the last
// tile, hold two waves' rows at a time: waves 2, 3 hand theirs to waves 0, 1, then wave 1 to wave 0) and write one
// partial per slice: a quarter of the partials' traffic and of the combine's work.
template <int D, int DV, int RB>
struct DecodeMerge {
  static constexpr bool value = DecodeImages<D, DV>::value * sizeof(MfmaSmem<D, DV>) >= sizeof(float) * 2 * 16 * RB * (DV + 4);
};

// Decode: a workgroup per (sequence with one row, key/value head, slice of the keys); rows = the group's query heads; the
// four waves share the staged tiles and take a 16-key subtile each.  Every wave writes its (maximum, denominator,
// weighted values) per head; the combine kernel merges them and the sink.
template <int D, int DV, int RB, int Layout>
__global__ __launch_bounds__(64 * kDecodeWaves) void sink_attention_decode_mfma_kernel(hymeta_sink_attention_args a, int splits, int tiles_per_split, HeadSlice hs) {
  constexpr int kImages = DecodeImages<D, DV>::value;
  constexpr bool kScaled = Layout == HYMETA_KV_SCALED_KEY;
  __shared__ MfmaSmem<D, DV> sm[kImages];
  __shared__ __attribute__((aligned(16))) float s_scale[kImages][kScaled ? kTileKeys : 4];
  int s = blockIdx.z, g = blockIdx.y, split = blockIdx.x;
  if (Layout == HYMETA_KV_SHARED_KEY) {
    // The value groups of a (sequence, split) read the same key tiles.  Workgroups go to the chip's 8 dies (each with an
    // L2 of its own) round robin by their number: a one-dimensional grid numbered so that those groups follow each other
    // on ONE die, which then fetches the keys from memory once instead of once per group.
    const int chunk = blockIdx.x >> 3, die = blockIdx.x & 7;
    const int pair = (chunk / a.num_kv_heads) * 8 + die;
    if (pair >= splits * a.num_seqs) return;
    g = chunk % a.num_kv_heads, s = pair / splits, split = pair % splits;
  }
  const int t = a.query_start_loc[s];
  if (a.query_start_loc[s + 1] - t != 1) return;
  const int pos = a.seq_lens[s] - 1;
  const int group = a.num_heads / a.num_kv_heads;
  const int HG = hs.count ? hs.count : group;            // this launch's rows
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 15, g4 = lane >> 4;
  // The sequence's tiles, numbered v = 0 ..: without a window tile v holds the keys from 64 v on, split as the host says.
  // With a window: the tiles of the kept first keys that lie before the window's first tile, then the window's tiles
  // (tiles wholly before the window are not read), dealt evenly over the splits.
  int kept_tiles = 0, window_from = 0, num_tiles = pos / kTileKeys + 1, per = tiles_per_split;
  const int first = first_key(a, pos);
  if (bounded(a)) {
    window_from = first / kTileKeys * kTileKeys;
    kept_tiles = min((a.keep_first + kTileKeys - 1) / kTileKeys * kTileKeys, window_from) / kTileKeys;
    num_tiles = kept_tiles + (pos - window_from) / kTileKeys + 1;
    per = (num_tiles + splits - 1) / splits;
  }
  const int v_lo = split * per, v_hi = min(num_tiles, v_lo + per) - 1;
  auto tile = [&](int v) { return v < kept_tiles ? v * kTileKeys : window_from + (v - kept_tiles) * kTileKeys; };
  constexpr bool kMerge = DecodeMerge<D, DV, RB>::value;
  float* part = static_cast<float*>(a.workspace) +
                (((static_cast<size_t>(s) * a.num_kv_heads + g) * splits + split) * (kMerge ? 1 : kDecodeWaves) + (kMerge ? 0 : wave)) *
                    (HG * partial_row_floats(DV));
  const int32_t* bt = a.block_tables + static_cast<int64_t>(s) * a.block_table_stride;
  WaveRows<D, DV, RB> w;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int r = 16 * rb + n;
    const bool ok = r < HG;
    const int h = g * group + hs.first + (ok ? r : 0);
    w.pos[rb] = ok ? pos : -1;
    w.first[rb] = first;
    load_bias<D, DV, RB>(w, rb, a, h);
    w.m[rb] = -INFINITY;
    w.l[rb] = 0.f;
    load_q<D, DV, RB>(w, rb, ok ? static_cast<const uint16_t*>(a.q) + static_cast<int64_t>(t) * a.q_stride_t + static_cast<int64_t>(h) * D : nullptr);
#pragma unroll
    for (int cb = 0; cb < DV / 16; ++cb) w.o[rb][cb] = f32x4v{0.f, 0.f, 0.f, 0.f};
  }
  TileStage<D, DV, 64 * kDecodeWaves, Layout> stage;
  if (Layout == HYMETA_KV_SHARED_KEY) stage.value_at = D + g * DV;
  if (v_lo <= v_hi) {
    stage.issue(a, bt, g, tile(v_lo), pos);
    stage.commit(sm[0], s_scale[0]);
    if (kImages == 2 && v_lo + 1 <= v_hi) stage.issue(a, bt, g, tile(v_lo + 1), pos);
  }
  __syncthreads();
  if constexpr (kImages == 2) {
    int buf = 0;
    for (int v = v_lo; v <= v_hi; ++v, buf ^= 1) {
      const int j0 = tile(v);
      if (v + 1 <= v_hi) stage.commit(sm[buf ^ 1], s_scale[buf ^ 1]);
      if (v + 2 <= v_hi) stage.issue(a, bt, g, tile(v + 2), pos);
      if (j0 + 16 * wave <= pos) {
        if (tile_open(j0, pos, first)) attend_tile<D, DV, RB, 1, false, kScaled>(w, sm[buf], s_scale[buf], a, j0, wave);
        else attend_tile<D, DV, RB, 1, true, kScaled>(w, sm[buf], s_scale[buf], a, j0, wave);
      }
      __syncthreads();
    }
  } else {
    // one image: the next tile's loads are in flight while this one is multiplied and go into LDS behind a barrier
    for (int v = v_lo; v <= v_hi; ++v) {
      const int j0 = tile(v);
      const bool more = v + 1 <= v_hi;
      if (more) stage.issue(a, bt, g, tile(v + 1), pos);
      if (j0 + 16 * wave <= pos) {
        if (tile_open(j0, pos, first)) attend_tile<D, DV, RB, 1, false, kScaled>(w, sm[0], s_scale[0], a, j0, wave);
        else attend_tile<D, DV, RB, 1, true, kScaled>(w, sm[0], s_scale[0], a, j0, wave);
      }
      __syncthreads();
      if (more) {
        stage.commit(sm[0], s_scale[0]);
        __syncthreads();
      }
    }
  }
  constexpr int kRowF = DV + 4;
  float* lds = reinterpret_cast<float*>(&sm[0]);            // (the loop ended on a barrier: nobody reads the tiles any more)
  float lr[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    float l = w.l[rb];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    lr[rb] = l;
  }
  // this wave's rows into LDS place `slot`, or (to == part) into the workspace
  auto put = [&](float* to, int rows_limit) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const int r = 16 * rb + n;
      if (r >= rows_limit) continue;
      float* pr = to + r * kRowF;
      if (g4 == 0) pr[DV] = w.m[rb], pr[DV + 1] = lr[rb];
#pragma unroll
      for (int cb = 0; cb < DV / 16; ++cb) *reinterpret_cast<f32x4v*>(pr + 16 * cb + 4 * g4) = w.o[rb][cb];
    }
  };
  // another wave's rows from LDS merged into this wave's
  auto take = [&](const float* from) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const float* pr = from + (16 * rb + n) * kRowF;
      const float mp = pr[DV], lp = pr[DV + 1];
      const float m = fmaxf(w.m[rb], mp);
      const float f = w.m[rb] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(w.m[rb] - m);      // (a wave that saw no key of the row)
      const float fp = mp == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mp - m);
#pragma unroll
      for (int cb = 0; cb < DV / 16; ++cb) w.o[rb][cb] = w.o[rb][cb] * f + *reinterpret_cast<const f32x4v*>(pr + 16 * cb + 4 * g4) * fp;
      lr[rb] = lr[rb] * f + lp * fp;
      w.m[rb] = m;
    }
  };
  if constexpr (kMerge) {
    static_assert(kDecodeWaves == 4, "the merge is a tree over four waves");
    if (wave >= 2) put(lds + (wave - 2) * 16 * RB * kRowF, 16 * RB);
    __syncthreads();
    if (wave < 2) take(lds + wave * 16 * RB * kRowF);
    __syncthreads();
    if (wave == 1) put(lds, 16 * RB);
    __syncthreads();
    if (wave == 0) {
      take(lds);
      put(part, HG);
    }
  } else {
    put(part, HG);
  }
}

// Merge a row's partials (`splits` of them, `stride` floats apart from `base` on), add the sink, normalise, store bf16: one
// workgroup per (row, head) and part of the columns.  Bound by round trips to memory: the threads read the partials' statistics
// side by side (one each) and, with them in flight, their first partials' values, agree on the row's maximum, and leave every
// partial's factor in LDS; groups of a thread per four columns take the partials in turn.  Values asked for behind the statistics,
// four at a time around a branch -> so, us: 28 heads of 128, 3 rows at 20000 keys 31.7 -> 28.8, 9 at 5000 13.9 -> 12.0; 16 heads of 128
// on a latent, a row at 20000 41.1 -> 18.5.
constexpr int kCombineThreads = 128;
constexpr int kMaxPartials = 512 * kDecodeWaves;
// Up to as many partials a (row, head) goes to the kernel that holds them all in registers: more partials are for few rows, which
// leave the chip room for a workgroup each.
constexpr int kFewPartials = 8;
// Columns of a workgroup where up to kPartRows (row, head) pairs have more partials: a row of 512 then has four workgroups that take
// the partials four at a time, and not one whose threads all take every partial.  16 heads on 512 + 64, 3 rows at 9600 keys 47.3 ->
// 23.5 us; 28 heads, a row at 30000 60 -> 25.  More pairs fill the chip by themselves, and the parts all read the statistics: with /
// without parts 16 heads, 20 rows at 7000 keys 39.7 / 41.1, 40 50.5 / 48.9, six portions of 40 at 1200 49.6 / 42.8; 28 heads, 20 rows at 3500 40.2 / 39.3.
constexpr int kPartColumns = 128, kPartRows = 512;

// Columns c .. c + 3 of row t's head h, from the weighted values and the weights' sum.
__device__ __forceinline__ void store_row(const hymeta_sink_attention_args& a, f32x4v acc, float l, int64_t t, int h, int c) {
  float inv = l > 0.f ? 1.f / l : 0.f;
  if (a.head_gate) inv *= sigmoid_exact(bf2f(static_cast<const uint16_t*>(a.head_gate)[t * a.head_gate_stride_t + h]));
  acc *= inv;
  if (a.elem_gate) {
    float gate[4];
    ActBf16::ld4(static_cast<const uint16_t*>(a.elem_gate) + t * a.elem_gate_stride_t + static_cast<int64_t>(h) * a.v_dim + c, gate);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] *= ActBf16::sigmoid(gate[e]);
  }
  *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.out) + (t * a.num_heads + h) * a.v_dim + c) =
      u32x2{pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3])};
}

// Whether a partial has seen no key, by its maximum and the sum of its weights: where every tile it saw held a NaN it has no
// maximum either, but a NaN for a sum, which the row's result keeps.
__device__ __forceinline__ bool no_keys(float m, float l) { return m == -INFINITY && l == 0.f; }

struct CombineScratch {
  __attribute__((aligned(16))) f32x4v acc[kCombineThreads];
  float f[kMaxPartials], red[2][kCombineThreads / 64];
};
// Batch: partials whose values a thread has in flight together, the first ones beside the statistics.
template <int Batch>
__device__ __forceinline__ void combine_row_in(CombineScratch& lds, const hymeta_sink_attention_args& a, const float* base, size_t stride, int splits, int64_t t, int h) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, DV = a.v_dim, cols = DV / gridDim.z;
  const int quads = cols / 4, turns = kCombineThreads / quads, turn = tid / quads, c = blockIdx.z * cols + 4 * (tid % quads);
  auto stat = [&](int sp) { return *reinterpret_cast<const float2*>(base + sp * stride + DV); };
  f32x4v x[Batch];
  auto fetch = [&](int sp0) __attribute__((always_inline)) {         // (past the last one: read again)
#pragma unroll
    for (int u = 0; u < Batch; ++u) x[u] = *reinterpret_cast<const f32x4v*>(base + min(sp0 + u * turns, splits - 1) * stride + c);
  };
  // (the partials' maxima are in the base-2 domain, as the waves kept them)
  const float sink2 = a.sink_logits ? a.sink_logits[h] * 1.4426950408889634f : 0.f;
  float m = a.sink ? sink2 : -INFINITY;
  const float2 own = stat(min(tid, splits - 1));       // this thread's first partial
  fetch(turn);
  if (tid < splits) m = fmaxf(m, own.x);
  for (int sp = tid + kCombineThreads; sp < splits; sp += kCombineThreads) m = fmaxf(m, stat(sp).x);
  m = wave_max(m);
  if (lane == 0) lds.red[0][wave] = m;
  __syncthreads();
  m = fmaxf(lds.red[0][0], lds.red[0][1]);
  float l = 0.f;
  for (int sp = tid; sp < splits; sp += kCombineThreads) {
    const float2 p = sp == tid ? own : stat(sp);
    const float f = no_keys(p.x, p.y) ? -1.f : __builtin_amdgcn_exp2f(p.x - m);
    lds.f[sp] = f;
    if (!(f < 0.f)) l = fmaf(p.y, f, l);
  }
  l = wave_sum(l);
  if (lane == 0) lds.red[1][wave] = l;
  __syncthreads();
  l = (lds.red[1][0] + lds.red[1][1]) + (a.sink ? __builtin_amdgcn_exp2f(sink2 - m) : 0.f);
  f32x4v acc = f32x4v{0.f, 0.f, 0.f, 0.f};
  for (int sp0 = turn; sp0 < splits;) {
#pragma unroll
    for (int u = 0; u < Batch; ++u) {
      const int sp = sp0 + u * turns;
      const float f = sp < splits ? lds.f[sp] : -1.f;
      if (!(f < 0.f)) acc += x[u] * f;
    }
    sp0 += Batch * turns;
    if (sp0 < splits) fetch(sp0);
  }
  if (turns > 1) {
    lds.acc[tid] = acc;
    __syncthreads();
    if (turn == 0)
      for (int k = 1; k < turns; ++k) acc += lds.acc[tid + k * quads];
  }
  if (turn == 0) store_row(a, acc, l, t, h, c);
}
__device__ __forceinline__ void combine_row(const hymeta_sink_attention_args& a, const float* base, size_t stride, int splits, int64_t t, int h) {
  __shared__ CombineScratch lds;
  const int work = splits * (a.v_dim / gridDim.z), each = 4 * kCombineThreads;       // (values, and how many one partial per thread is)
  if (work <= each) combine_row_in<1>(lds, a, base, stride, splits, t, h);
  else if (work <= 4 * each) combine_row_in<4>(lds, a, base, stride, splits, t, h);
  else combine_row_in<8>(lds, a, base, stride, splits, t, h);
}

// How the keys of portions are cut: into `splits` slices at most, whose partials lie at `parts`, [row][head][splits]; blocks of
// up to `whole` tiles of 64 keys are not cut.
constexpr int kLeastTiles = 2;                 // of a slice
struct PortionSlices {
  int splits = 1, whole = 0, least = 2;        // least: rows from which a sequence is a portion
  float* parts = nullptr;
};
constexpr int kPortionRows = 128;              // (query, head) rows of a block, the heads of a key/value head side by side

// The keys that rows at positions p_first .. p_hi see, in tiles of Keys: first the kept first keys that lie before the window's
// first tile, then the window's.  Rows in front of the sequence, at positions below 0, see nothing.
struct BlockKeys {
  int from, kept, tiles, size;
  __device__ __forceinline__ int first(int t) const { return t < kept ? t * size : from + (t - kept) * size; }
  __device__ __forceinline__ int slices(const PortionSlices& ps) const {
    return tiles * size <= ps.whole * kTileKeys ? 1 : max(1, min(ps.splits, tiles * size / (kLeastTiles * kTileKeys)));
  }
};
template <int Keys>
__device__ __forceinline__ BlockKeys block_keys(const hymeta_sink_attention_args& a, int p_first, int p_hi) {
  BlockKeys b;
  b.size = Keys;
  b.from = first_key(a, max(0, p_first)) / Keys * Keys;
  b.kept = bounded(a) ? min((a.keep_first + Keys - 1) / Keys * Keys, b.from) / Keys : 0;
  b.tiles = p_hi < 0 ? 0 : b.kept + (p_hi - b.from) / Keys + 1;
  return b;
}
// Block `number` of the step's portions.
__device__ __forceinline__ PieceAt portion_block(const hymeta_sink_attention_args& a, int number, const PortionSlices& ps) {
  const int group = a.num_heads / a.num_kv_heads;
  return piece_at(a.query_start_loc, a.num_seqs, number, [=, least = ps.least](int q) { return q >= least ? (q * group + kPortionRows - 1) / kPortionRows : 0; });
}
constexpr int kWideKeys = 32;                  // a tile of the kernels over wide latents

// grid = (sequences + rows where portions' keys were cut, heads, parts of the columns): the rows of single-row sequences, and the rows of portions whose
// blocks were cut.  One launch for both: a step of both takes no more launches than without slices.  A row's portion is found in
// one round trip for 64 sequences (one read behind the other: 300 whole rows beside 63 single ones took 78.2 us, so 76.2).
__global__ __launch_bounds__(kCombineThreads) void sink_attention_combine_kernel(hymeta_sink_attention_args a, int splits, HeadSlice hs, PortionSlices ps) {
  // (splits: partials per (sequence, key/value head): one per slice, or one per wave of a slice)
  const int group = a.num_heads / a.num_kv_heads, HG = hs.count ? hs.count : group;
  const int g = blockIdx.y / HG, r = blockIdx.y % HG, in_group = hs.first + r, h = g * group + in_group;
  const size_t row = partial_row_floats(a.v_dim);
  const int singles = ps.least > 1 ? a.num_seqs : 0;   // (else single rows are portions)
  if (blockIdx.x < singles) {
    const int s = blockIdx.x, t = a.query_start_loc[s];
    if (a.query_start_loc[s + 1] - t != 1) return;
    const size_t stride = HG * row;
    combine_row(a, static_cast<const float*>(a.workspace) + (static_cast<size_t>(s) * a.num_kv_heads + g) * splits * stride + r * row, stride, splits, t, h);
    return;
  }
  const PieceAt at = piece_at(a.query_start_loc, a.num_seqs, blockIdx.x - singles, [](int q) { return q; });
  if (at.seq < 0 || at.rows < ps.least) return;              // (rows behind the last portion have no partials)
  const int t = at.row0 + at.index, ctx = a.seq_lens[at.seq] - at.rows, rows = at.rows * group, r0 = (at.index * group + in_group) / kPortionRows * kPortionRows;
  const int p_first = ctx + r0 / group, p_hi = ctx + (min(rows, r0 + kPortionRows) - 1) / group;
  const int n = a.v_dim > 128 ? block_keys<kWideKeys>(a, p_first, p_hi).slices(ps) : block_keys<kTileKeys>(a, p_first, p_hi).slices(ps);
  if (n > 1) combine_row(a, ps.parts + (static_cast<size_t>(t) * a.num_heads + h) * ps.splits * row, row, n, t, h);
}

// The same for single rows of at most N partials where no portion's keys were cut: every thread reads all of its four columns'
// partials and their statistics at once, v_dim / 4 threads to a (row, head), as many heads as fit in a workgroup; no LDS, no
// barriers.  grid = (sequences, head groups).  A workgroup per (row, head) needs four round trips and two barriers for them, and
// more than 3840 of them (LDS) are not on the chip at once.  28 heads of 128 with the kernel in front, a workgroup each -> so (and
// with the serial loop), us: 236 rows at 79 keys 27.4 -> 23.1 (24.9), 256 at 1024 111.0 -> 105.3 (108.5), 64 at 4096 101.6 ->
// 99.9 (102.1), 16 at 4096 (8 partials) 30.5 -> 29.2 (36.1); 64 x 16 heads of 512 at 4096 70.9 -> 69.8.
template <int N>
__global__ __launch_bounds__(kCombineThreads) void sink_attention_combine_few_kernel(hymeta_sink_attention_args a, int splits, HeadSlice hs) {
  const int s = blockIdx.x, t = a.query_start_loc[s];
  const int group = a.num_heads / a.num_kv_heads, HG = hs.count ? hs.count : group, DV = a.v_dim;
  const int quads = DV / 4, each = kCombineThreads / quads, at = blockIdx.y * each + threadIdx.x / quads, c = 4 * (threadIdx.x % quads);
  if (a.query_start_loc[s + 1] - t != 1 || threadIdx.x >= each * quads || at >= HG * a.num_kv_heads) return;
  const int g = at / HG, r = at % HG, h = g * group + hs.first + r;
  const size_t row = partial_row_floats(DV), stride = HG * row;
  const float* base = static_cast<const float*>(a.workspace) + (static_cast<size_t>(s) * a.num_kv_heads + g) * splits * stride + r * row;
  f32x4v x[N];
  float2 stat[N];                                      // a partial's maximum (base-2 domain) and denominator
#pragma unroll
  for (int sp = 0; sp < N; ++sp) {                     // (past the last one: read again)
    const float* part = base + min(sp, splits - 1) * stride;
    stat[sp] = *reinterpret_cast<const float2*>(part + DV);
    x[sp] = *reinterpret_cast<const f32x4v*>(part + c);
  }
  const float sink2 = a.sink_logits ? a.sink_logits[h] * 1.4426950408889634f : 0.f;
  float m = a.sink ? sink2 : -INFINITY;
#pragma unroll
  for (int sp = 0; sp < N; ++sp) m = fmaxf(m, stat[sp].x);
  float l = a.sink ? __builtin_amdgcn_exp2f(sink2 - m) : 0.f;
  f32x4v acc = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int sp = 0; sp < N; ++sp)
    if (sp < splits && !no_keys(stat[sp].x, stat[sp].y)) {
      const float f = __builtin_amdgcn_exp2f(stat[sp].x - m);
      l = fmaf(stat[sp].y, f, l);
      acc += x[sp] * f;
    }
  store_row(a, acc, l, t, h, c);
}

}  // namespace
}  // namespace hymeta

#include "row_attn.h"
#include "row_pipe.h"
#include "wide_latent.h"

namespace hymeta {
namespace {

// Head sizes the matrix-core kernels are built for.  A value inside its key: a latent of 64 or 128 followed by a rotated
// part of 32 or 64 (the kernels above), or a latent of 256 / 384 / 512 followed by a rotated part of 64 (wide_latent.h).
inline bool mfma_shape(const hymeta_sink_attention_args& a) {
  bool dims = (a.head_dim == 64 || a.head_dim == 128) && (a.v_dim == 64 || a.v_dim == 128);
  if (a.kv_layout == HYMETA_KV_VALUE_IN_KEY)
    dims = ((a.v_dim == 64 || a.v_dim == 128) && (a.head_dim == a.v_dim + 32 || a.head_dim == a.v_dim + 64)) ||
           ((a.v_dim == 256 || a.v_dim == 384 || a.v_dim == 512) && a.head_dim == a.v_dim + 64);
  // one key for all heads: the concatenated keys of 1 / 2 / 4 / 8 key/value heads of 64 or 128
  if (a.kv_layout == HYMETA_KV_SHARED_KEY)
    dims = (a.head_dim == 64 || a.head_dim == 128 || a.head_dim == 256 || a.head_dim == 512) && (a.v_dim == 64 || a.v_dim == 128);
  // key and value in one vector
  if (a.kv_layout == HYMETA_KV_SCALED_KEY)
    dims = a.head_dim == a.v_dim && (a.head_dim == 32 || a.head_dim == 64 || a.head_dim == 96 || a.head_dim == 128) &&
           a.bias_mode != HYMETA_BIAS_LOG_DISTANCE && a.softcap <= 0.f;
  else if (a.bias_mode == HYMETA_BIAS_LINEAR_DISTANCE) dims = false;
  if (a.elem_gate && (a.elem_gate_stride_t % 4 != 0 || reinterpret_cast<uintptr_t>(a.elem_gate) % 8 != 0)) dims = false;
  return a.act_dtype == HYMETA_BF16 && dims && a.q_stride_t % 8 == 0 &&
         (a.block_size & (a.block_size - 1)) == 0 &&
         (reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.kv_cache) | reinterpret_cast<uintptr_t>(a.out)) % 16 == 0;
}

// Tiles of 64 keys a decode row reads at most: all of its sequence's, or with a window or a chunk the kept first keys' and
// that span's, however long the sequence is.
inline int decode_tiles(int max_seq_len, int64_t span = 0, int keep_first = 0) {
  const int tiles = (max_seq_len + kTileKeys - 1) / kTileKeys;
  if (span <= 0) return tiles;
  const int64_t seen = (static_cast<int64_t>(keep_first) + kTileKeys - 1) / kTileKeys + (span - 1) / kTileKeys + 2;
  return static_cast<int>(std::min<int64_t>(seen, tiles));
}
inline int decode_tiles(const hymeta_sink_attention_args& a) {
  return decode_tiles(a.max_seq_len, a.chunk > 0 ? a.chunk : static_cast<int64_t>(a.window_left) + 1, a.keep_first);
}

inline int decode_splits(int num_seqs, int num_heads, int num_kv_heads, int tiles) {
  // Workgroups aimed at: a workgroup's fixed cost (query fragments, first tile, the merge of its waves, its partial) grows
  // with the query heads it carries, so fewer, longer workgroups pay.  Measured at 64 sequences x 4096 keys: 28 heads on
  // one row of 192: 93 / 67 / 56 / 87 us at 1024 / 512 / 256 / 128; 16 heads on it: 53 / 40 / 45; 4 key/value heads with
  // 7 query heads each: 125 / 114 / 168.
  const int target = num_heads / num_kv_heads > 16 ? 256 : 512;
  const int splits = (target + num_seqs * num_kv_heads - 1) / (num_seqs * num_kv_heads);
  return std::max(1, std::min(splits, tiles));
}

inline int64_t decode_partial_bytes(int num_seqs, int num_heads, int num_kv_heads, int v_dim, int max_seq_len) {
  const int splits = decode_splits(num_seqs, num_heads, num_kv_heads, decode_tiles(max_seq_len < 1 ? 1 : max_seq_len));
  return static_cast<int64_t>(num_seqs) * splits * kDecodeWaves * num_heads * static_cast<int64_t>(partial_row_floats(v_dim)) * 4;
}

// Bound on the portions' blocks of 128 rows: as many of the longest as there are sequences, or the rows' and one begun per
// portion of `least` rows or more.
inline int64_t portion_blocks(int num_tokens, int num_seqs, int group, int max_query_len, int least = 2) {
  const int64_t each = (static_cast<int64_t>(max_query_len) * group + kPortionRows - 1) / kPortionRows;
  return std::max<int64_t>(1, std::min<int64_t>(each * num_seqs, static_cast<int64_t>(num_tokens) * group / kPortionRows + std::min(num_seqs, num_tokens / least)));
}
// Slices a portion's keys are cut into: where the blocks that the step's portions are worth (long_portions) do not fill the chip
// (`target` workgroups) and the workspace has room for the partials (bounded: every row of the step has a place).  A slice's
// queries, its first tile and its partial cost about two tiles of 64 keys, and a (row, head) of the merge about 1 / 768 of one,
// so that blocks of fewer tiles stay whole.  7 rows x 28 heads behind 6000 keys: 299 -> 25 us; 40 rows x 28 heads on latents of
// 512 + 64, twice: 592 -> 77; 300 rows on latents of 128 + 64, twice: 233 -> 101.  Slices of two tiles and more: of four, 64 rows
// x 28 heads behind 400 keys took 29.0 us (26.0 with a workgroup per head), three times 40 28.3 (24.5), 8 behind 650 27.4 (30.6);
// of two 23.4, 24.9 and 23.9, at which the host's call stands; of three between them.
//
// Beside single rows, whose keys say nothing of the portion's, the merge's look at every row of the step (1 to 3 us) is lost on a
// portion that begins its sequence.  Up to kFewBlocks, where one behind many keys would have nothing but its own tiles to wait
// for, it is worth it (with at most kMostNumbers numbers of blocks, most of which have none): 40 rows x 28 heads behind 6000
// keys beside 63 single rows take 161 us where they took 417 whole, with a window of 1024 47 where they took 85 (329 and 75 with
// a workgroup per head); without keys in front of them 41 (38).  Above, only where all numbers fit the chip.
constexpr int64_t kMostPartialBytes = 96 << 20, kFewBlocks = 32, kMostNumbers = 2048;
inline int64_t portion_partial_bytes(int num_tokens, int num_heads, int v_dim) {
  return static_cast<int64_t>(num_tokens) * num_heads * static_cast<int64_t>(partial_row_floats(v_dim)) * 4;
}
inline PortionSlices portion_slices(int num_tokens, int num_seqs, int num_heads, int num_kv_heads, int v_dim, int max_query_len, int tiles, int head_dim = 0) {
  PortionSlices ps;
  const int group = std::max(1, num_heads / num_kv_heads), target = v_dim > 128 || head_dim > 192 ? 256 : 512;       // one workgroup on a compute unit (wide_latent.h, long keys), or two
  const int64_t each = (static_cast<int64_t>(max_query_len) * group + kPortionRows - 1) / kPortionRows, portions = long_portions(num_tokens, num_seqs, max_query_len);
  const int64_t blocks = each * portions * num_kv_heads;
  int64_t most = std::min<int64_t>(tiles / kLeastTiles, kMostPartialBytes / portion_partial_bytes(num_tokens, num_heads, v_dim));
  if (num_seqs > portions) most = std::min<int64_t>(most, (blocks > kFewBlocks ? target : kMostNumbers) / (portion_blocks(num_tokens, num_seqs, group, max_query_len) * num_kv_heads));
  ps.whole = static_cast<int>(std::min<int64_t>(tiles, std::max<int64_t>(2 * kLeastTiles - 1, portions * max_query_len * num_heads / 768)));
  if (tiles > ps.whole) ps.splits = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(target / blocks, most)));
  // (an odd stride: the first slices alone, where blocks stay whole, are on all of the chip's 8 dies)
  if (num_seqs > portions && blocks <= kFewBlocks && ps.splits > 2) ps.splits -= 1 - ps.splits % 2;
  return ps;
}
inline bool one_launch(const hymeta_sink_attention_args& a, const PortionSlices& ps, int most);
inline bool long_shared_keys(const hymeta_sink_attention_args& a);
inline bool few_single_rows(const hymeta_sink_attention_args& a);
inline PortionSlices portion_slices(const hymeta_sink_attention_args& a) {
  PortionSlices ps;
  if (a.max_query_len <= 1) return ps;
  ps = portion_slices(a.num_tokens, a.num_seqs, a.num_heads, a.num_kv_heads, a.v_dim, a.max_query_len, decode_tiles(a), a.head_dim);
  // Long keys are cut beside few single rows only.  Where the portions' launch takes those as well (one_launch), the slices have the
  // room of the decode form's partials.
  const bool long_keys = long_shared_keys(a), along = ps.splits > 1 && one_launch(a, ps, 0);
  if (long_keys && ps.splits > 1 && !few_single_rows(a)) ps.splits = 1;
  const int64_t decode = long_keys && along ? 0 : decode_partial_bytes(a.num_seqs, a.num_heads, a.num_kv_heads, a.v_dim, a.max_seq_len);
  const int64_t room = (static_cast<int64_t>(a.workspace_bytes) - decode) / portion_partial_bytes(a.num_tokens, a.num_heads, a.v_dim);
  ps.splits = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(ps.splits, room)));
  if (long_keys && along && ps.splits > 1 && !one_launch(a, ps, 0)) ps.splits = 1;      // (fewer, longer slices, which no longer do)
  ps.parts = static_cast<float*>(a.workspace) + decode / 4;
  return ps;
}
inline dim3 portion_grid(const hymeta_sink_attention_args& a, const PortionSlices& ps) {
  return dim3(static_cast<uint32_t>(portion_blocks(a.num_tokens, a.num_seqs, a.num_heads / a.num_kv_heads, a.max_query_len, ps.least) * ps.splits * a.num_kv_heads));
}
// Whether the portions' launch takes the single rows as well, as portions of one row: the decode form is not launched then, nor,
// where no keys are cut, its merge, which cost 5 to 8 us where a step has no single row.  Without cut keys only where no row sees
// more than `most` tiles of 64 keys, which a workgroup walks alone (about 1.5 us each), and the single rows that there may be find
// room beside each other.  28 heads of 128 with 4 key/value heads: six portions of 147 rows 28.9 -> 22.2 us, three of 100 behind 100
// 25.8 -> 19.3 (at which the host's call stood); 40 rows beside 63 single ones, behind 400 36.6 -> 34.7, behind 900 47.4 -> 47.0.  A
// tile of the wide latents' kernel costs three times as much: six portions of 33 rows on 512 + 64 27.5 -> 21.3.  Where keys are cut
// the single rows' are as well; few of them, as a slice of theirs has a workgroup of 128 rows to itself: 7 rows behind 6000 26.8 ->
// 20.6 us, 40 beside 8 single ones 50.3 -> 46.4 (latents of 128 + 64: 48.0 -> 38.3), 8 beside 15 behind 3000 40.7 -> 34.5 (of each
// about 5 the host's shorter call).  With one key/value head, whose single rows fill a fifth of a block, a quarter as many: 300 rows beside 8
// single ones of 4096 keys on latents of 128 + 64 46 -> 49, beside 63 75 -> 86.  A logarithm per score makes them dearer: 40 rows with nothing
// in front beside 15 single ones of 4096 keys 39.7 -> 42.3, but 2 behind 3000 beside 15 of 3000 40.3 -> 37.0.
// Long keys have one workgroup on a compute unit, so single rows go along where they take no more rounds of units than the portions do
// without them: 40 rows beside 63 single ones of 100 keys of 512, 28 heads, in 264 workgroups 23.9, in two launches 22.0; beside 127
// 53.9 and 43.6, 40 beside 127 of 400 keys of 256 68 and 57; 40 beside 48 of 60 keys, 204 workgroups, 17 and 22.
// Of their cut keys a single row's workgroup walks a slice alone while portions that begin their sequence are done with their few tiles:
// up to 16 tiles of 64 keys, or 8 where a tile takes several pages (a copy's addresses are looked up row by row).  All of it by the
// portions' launch -> in two: 190 and 339 rows of 16 heads of 256 beside four of up to 7552 keys in pages of 16 262 -> 59 us, 513 beside six of
// up to 7311 142 -> 57, 346 beside three of up to 3208 140 -> 49; rows of portions behind many keys lose the other launch, 129 and 18 behind 2000
// beside twelve 54 -> 71.  520 steps of one to four
// portions and up to 16 single rows: 0.29 to 1.39 of the time, 0.96 on average.
constexpr int kFewTiles = 16, kFewWideTiles = 2, kManySingleRows = 512, kLongKeyUnits = 256, kFewSingleRows = 4;
constexpr int kAlongTiles = 16, kAlongPagedTiles = 8;
inline bool long_shared_keys(const hymeta_sink_attention_args& a) { return a.kv_layout == HYMETA_KV_SHARED_KEY && a.head_dim > 192; }
inline bool few_single_rows(const hymeta_sink_attention_args& a) {
  return a.num_seqs - long_portions(a.num_tokens, a.num_seqs, a.max_query_len) <= kFewSingleRows * std::min(a.num_kv_heads, 4);
}
inline bool one_launch(const hymeta_sink_attention_args& a, const PortionSlices& ps, int most) {
  const int64_t portions = long_portions(a.num_tokens, a.num_seqs, a.max_query_len), singles = a.num_seqs - portions;
  if (a.max_query_len <= 1) return false;
  if (ps.splits > 1) {
    const int along = a.block_size < kTileKeys ? kAlongPagedTiles : kAlongTiles;
    return few_single_rows(a) && (!long_shared_keys(a) || singles == 0 || (decode_tiles(a) + ps.splits - 1) / ps.splits <= along);
  }
  if (decode_tiles(a) > most) return false;
  if (!long_shared_keys(a)) return singles * a.num_kv_heads <= kManySingleRows;
  const int64_t each = (static_cast<int64_t>(a.max_query_len) * (a.num_heads / a.num_kv_heads) + kPortionRows - 1) / kPortionRows;
  const int64_t units = each * portions * a.num_kv_heads;
  return units + singles * a.num_kv_heads <= (units + kLongKeyUnits - 1) / kLongKeyUnits * kLongKeyUnits || singles == 0;
}
// Long keys: whether sink_attention_prefill_shared_kernel takes the portions (and, `alone`, the single rows): keys of four tiles at most
// and all workgroups at once.  Its time -> row_pipe.h's, us, 28 heads of 512, 48 rows: one tile 10.4 -> 16.6, two 14.9 -> 22.8, four
// 25.0 -> 27.3, six 34.8 -> 32.5; four tiles, four portions of 128 rows (224 workgroups) 26.9 -> 28.1, of 200 (448) 48.2 -> 28.2.
constexpr int kFewLongTiles = 4;
inline bool few_long_keys(const hymeta_sink_attention_args& a, bool alone) {
  const int64_t portions = long_portions(a.num_tokens, a.num_seqs, a.max_query_len), each = (a.max_query_len + kPrefillRows - 1) / kPrefillRows;
  return decode_tiles(a) <= kFewLongTiles && (each * portions + (alone ? a.num_seqs - portions : 0)) * a.num_heads <= kLongKeyUnits;
}
void launch_combine(const hymeta_sink_attention_args& a, hipStream_t st, int splits, HeadSlice hs, const PortionSlices& ps) {
  const int heads = hs.count ? hs.count * a.num_kv_heads : a.num_heads;
  if (ps.splits == 1 && splits <= kFewPartials) {
    const int each = kCombineThreads / (a.v_dim / 4);
    const dim3 grid(a.num_seqs, (heads + each - 1) / each);
    if (splits <= 2) hipLaunchKernelGGL(sink_attention_combine_few_kernel<2>, grid, dim3(kCombineThreads), 0, st, a, splits, hs);
    else if (splits <= 4) hipLaunchKernelGGL(sink_attention_combine_few_kernel<4>, grid, dim3(kCombineThreads), 0, st, a, splits, hs);
    else hipLaunchKernelGGL(sink_attention_combine_few_kernel<kFewPartials>, grid, dim3(kCombineThreads), 0, st, a, splits, hs);
    return;
  }
  const int64_t rows = (ps.least > 1 ? a.num_seqs : 0) + static_cast<int64_t>(ps.splits > 1 ? a.num_tokens : 0);
  const bool apart = a.v_dim > kPartColumns && rows * heads <= kPartRows && std::max(splits, ps.splits) > kFewPartials;
  const dim3 grid(static_cast<unsigned>(rows), heads, apart ? a.v_dim / kPartColumns : 1);
  hipLaunchKernelGGL(sink_attention_combine_kernel, grid, dim3(kCombineThreads), 0, st, a, splits, hs, ps);
}

template <int C>
int launch_wide_latent(const hymeta_sink_attention_args& a, hipStream_t st) {
  const int group = a.num_heads / a.num_kv_heads;
  PortionSlices ps = portion_slices(a);
  const bool alone = one_launch(a, ps, kFewWideTiles);
  if (alone) ps.least = 1;
  if (a.max_query_len > 1) {
    if (a.softcap <= 0.f && a.bias_mode == 0) hipLaunchKernelGGL((latent_prefill_kernel<C, true>), portion_grid(a, ps), dim3(64 * kWideWaves), 0, st, a, ps);
    else hipLaunchKernelGGL((latent_prefill_kernel<C, false>), portion_grid(a, ps), dim3(64 * kWideWaves), 0, st, a, ps);
  }
  if (alone) {
    if (ps.splits > 1) launch_combine(a, st, 0, HeadSlice{}, ps);
    return launch_status();
  }
  // one workgroup per compute unit (its rings fill the LDS): as many as there are units
  const int64_t slices = (group + kLatentHeads - 1) / kLatentHeads, items = static_cast<int64_t>(a.num_seqs) * a.num_kv_heads;
  const int splits = static_cast<int>(std::min<int64_t>((256 + items * slices - 1) / (items * slices), decode_tiles(a)));
  const dim3 grid(static_cast<uint32_t>((items * splits + 7) / 8 * 8 * slices));
  hipLaunchKernelGGL((latent_decode_kernel<C>), grid, dim3(64 * kLatentWaves), 0, st, a, splits);
  launch_combine(a, st, splits, HeadSlice{}, ps);
  return launch_status();
}

template <int D, int DV, int Layout = HYMETA_KV_KEY_THEN_VALUE>
int launch_mfma(const hymeta_sink_attention_args& a, hipStream_t st) {
  PortionSlices ps;
  if (a.max_query_len > 1) {
    ps = portion_slices(a);
    const bool alone = one_launch(a, ps, kFewTiles);
    if (alone) ps.least = 1;
    const dim3 grid = portion_grid(a, ps);
    bool done = false;
    if constexpr (D > 192) {
      done = few_long_keys(a, alone);
      if (done) {
        ps.splits = 1;
        const dim3 all((a.max_query_len + kPrefillRows - 1) / kPrefillRows, a.num_heads, a.num_seqs);
        hipLaunchKernelGGL((sink_attention_prefill_shared_kernel<D, DV>), all, dim3(64 * kPrefillWaves), 0, st, a, ps.least);
      }
    }
    // a kernel per rule of the scores; a cap and a bias together, which no design has, in the general one
    auto launch = [&](auto rule) {
      constexpr int Rule = decltype(rule)::value;
      if (done) return;
      if constexpr (D > 192 || ((Layout == HYMETA_KV_KEY_THEN_VALUE || Layout == HYMETA_KV_SHARED_KEY) && Rule != kAnyRule))
        hipLaunchKernelGGL((row_pipe_kernel<D, DV, Layout, Rule>), grid, dim3(256), 0, st, a, ps);
      else hipLaunchKernelGGL((row_prefill_kernel<D, DV, Layout, Rule>), grid, dim3(256), 0, st, a, ps);
    };
    const bool log_bias = a.bias_mode == HYMETA_BIAS_LOG_DISTANCE, capped = a.softcap > 0.f;
    if (Layout == HYMETA_KV_SCALED_KEY || (!log_bias && !capped)) launch(std::integral_constant<int, kPlain>{});
    else if constexpr (Layout == HYMETA_KV_KEY_THEN_VALUE) {
      if (!capped) launch(std::integral_constant<int, kLogBias>{});
      else if (!log_bias) launch(std::integral_constant<int, kCapped>{});
      else launch(std::integral_constant<int, kAnyRule>{});
    } else if constexpr (Layout != HYMETA_KV_SCALED_KEY) {
      launch(std::integral_constant<int, kAnyRule>{});
    }
    if (alone) {
      if (ps.splits > 1) launch_combine(a, st, 0, HeadSlice{}, ps);
      return launch_status();
    }
  }
  // sequences with a single row: every step but a pure prompt step has some; a prompt of one token is one too
  const int splits = decode_splits(a.num_seqs, a.num_heads, a.num_kv_heads, decode_tiles(a));
  const int tiles = (a.max_seq_len + kTileKeys - 1) / kTileKeys;
  const int tiles_per_split = (tiles + splits - 1) / splits;
  const dim3 grid = Layout == HYMETA_KV_SHARED_KEY ? dim3((splits * a.num_seqs + 7) / 8 * 8 * a.num_kv_heads) : dim3(splits, a.num_kv_heads, a.num_seqs);
  const int group = a.num_heads / a.num_kv_heads;
  for (int first = 0; first < group; first += kRowsPerWave) {
    const HeadSlice hs{first, group - first < kRowsPerWave ? group - first : kRowsPerWave};
    int parts;
    if (hs.count <= 16) {
      hipLaunchKernelGGL((sink_attention_decode_mfma_kernel<D, DV, 1, Layout>), grid, dim3(64 * kDecodeWaves), 0, st, a, splits, tiles_per_split, hs);
      parts = splits * (DecodeMerge<D, DV, 1>::value ? 1 : kDecodeWaves);
    } else {
      hipLaunchKernelGGL((sink_attention_decode_mfma_kernel<D, DV, 2, Layout>), grid, dim3(64 * kDecodeWaves), 0, st, a, splits, tiles_per_split, hs);
      parts = splits * (DecodeMerge<D, DV, 2>::value ? 1 : kDecodeWaves);
    }
    launch_combine(a, st, parts, hs, ps);
  }
  return launch_status();
}

}  // namespace

}  // namespace hymeta

using namespace hymeta;

extern "C" int hymeta_qk_norm_cache(const hymeta_qk_norm_cache_args* args, hymeta_stream_t stream) {
  if (!args_ok(args)) return HYMETA_ERR_INVALID_ARG;
  const hymeta_qk_norm_cache_args& a = *args;
  if (a.num_tokens < 0 || a.num_heads <= 0 || a.num_kv_heads <= 0 || a.head_dim <= 0 || a.v_dim <= 0 || a.block_size <= 0 ||
      a.num_blocks < 0)
    return HYMETA_ERR_INVALID_ARG;
  if (!act_dtype_ok(a.act_dtype)) return HYMETA_ERR_UNSUPPORTED;
  if (a.num_tokens == 0) return HYMETA_OK;
  if (!a.qkv || (a.slot_mapping && !a.kv_cache)) return HYMETA_ERR_INVALID_ARG;
  if (a.qkv_stride_t < static_cast<int64_t>(a.num_heads + a.num_kv_heads) * a.head_dim + static_cast<int64_t>(a.num_kv_heads) * a.v_dim)
    return HYMETA_ERR_INVALID_ARG;
  hipStream_t st = begin_launches(stream);
  if (a.act_dtype == HYMETA_BF16) hipLaunchKernelGGL(qk_norm_cache_kernel<ActBf16>, dim3(a.num_tokens), dim3(256), 0, st, a);
  else hipLaunchKernelGGL(qk_norm_cache_kernel<ActF32>, dim3(a.num_tokens), dim3(256), 0, st, a);
  return launch_status();
}

extern "C" int hymeta_scaled_key_cache(const hymeta_scaled_key_cache_args* args, hymeta_stream_t stream) {
  if (!args_ok(args)) return HYMETA_ERR_INVALID_ARG;
  const hymeta_scaled_key_cache_args& a = *args;
  if (a.num_tokens < 0 || a.num_heads <= 0 || a.num_kv_heads <= 0 || a.head_dim <= 0 || a.num_blocks < 0) return HYMETA_ERR_INVALID_ARG;
  if (!act_dtype_ok(a.act_dtype)) return HYMETA_ERR_UNSUPPORTED;
  if (a.num_tokens == 0) return HYMETA_OK;
  if (!a.qk || !a.q_weight || !a.k_weight || a.qk_stride_t < static_cast<int64_t>(a.num_heads + a.num_kv_heads) * a.head_dim) return HYMETA_ERR_INVALID_ARG;
  if (a.slot_mapping && (!a.kv_cache || a.block_size <= 0 || reinterpret_cast<uintptr_t>(a.kv_cache) % 16 != 0)) return HYMETA_ERR_INVALID_ARG;
  if (a.temp_coef != 0.f && (!a.positions || !(a.temp_every > 0.0))) return HYMETA_ERR_INVALID_ARG;
  hipStream_t st = begin_launches(stream);
  const int bytes = a.act_dtype == HYMETA_BF16 ? 2 : 4;
  // four elements a lane where a head and a row are whole fours and a head fits a wave
  const bool vec = a.head_dim % 4 == 0 && a.head_dim <= 256 && a.qk_stride_t % 4 == 0 && reinterpret_cast<uintptr_t>(a.qk) % (4 * bytes) == 0;
  int lanes = 64;
  if (vec) {
    lanes = 1;
    while (4 * lanes < a.head_dim) lanes *= 2;
  }
  const dim3 grid(a.num_tokens), block(256);
  if (a.act_dtype == HYMETA_BF16) {
    if (vec) hipLaunchKernelGGL((scaled_key_cache_kernel<ActBf16, true>), grid, block, 0, st, a, lanes);
    else hipLaunchKernelGGL((scaled_key_cache_kernel<ActBf16, false>), grid, block, 0, st, a, lanes);
  } else {
    if (vec) hipLaunchKernelGGL((scaled_key_cache_kernel<ActF32, true>), grid, block, 0, st, a, lanes);
    else hipLaunchKernelGGL((scaled_key_cache_kernel<ActF32, false>), grid, block, 0, st, a, lanes);
  }
  return launch_status();
}

extern "C" size_t hymeta_sink_attention_workspace_bytes(int32_t num_seqs, int32_t num_heads, int32_t num_kv_heads, int32_t v_dim,
                                                        int32_t max_seq_len) {
  if (num_seqs <= 0 || num_heads <= 0 || num_kv_heads <= 0 || v_dim <= 0) return 0;
  return static_cast<size_t>(decode_partial_bytes(num_seqs, num_heads, num_kv_heads, v_dim, max_seq_len));
}

extern "C" size_t hymeta_sink_attention_portion_workspace_bytes(int32_t num_tokens, int32_t num_seqs, int32_t num_heads, int32_t num_kv_heads,
                                                                int32_t v_dim, int32_t max_query_len, int32_t max_seq_len, int64_t span,
                                                                int32_t keep_first) {
  const size_t single = hymeta_sink_attention_workspace_bytes(num_seqs, num_heads, num_kv_heads, v_dim, max_seq_len);
  if (num_tokens <= 0 || single == 0 || max_query_len <= 1 || max_seq_len < 1) return single;
  const int splits = portion_slices(num_tokens, num_seqs, num_heads, num_kv_heads, v_dim, max_query_len, decode_tiles(max_seq_len, span, keep_first)).splits;
  return single + (splits > 1 ? static_cast<size_t>(splits * portion_partial_bytes(num_tokens, num_heads, v_dim)) : 0);
}

extern "C" int hymeta_sink_attention(const hymeta_sink_attention_args* args, hymeta_stream_t stream) {
  if (!args_ok(args)) return HYMETA_ERR_INVALID_ARG;
  const hymeta_sink_attention_args& a = *args;
  if (a.num_tokens < 0 || a.num_seqs < 0 || a.num_heads <= 0 || a.num_kv_heads <= 0 || a.head_dim <= 0 || a.v_dim <= 0 ||
      a.block_size <= 0 || a.num_blocks < 0)
    return HYMETA_ERR_INVALID_ARG;
  if (a.num_heads % a.num_kv_heads != 0) return HYMETA_ERR_INVALID_ARG;
  if (!act_dtype_ok(a.act_dtype)) return HYMETA_ERR_UNSUPPORTED;
  if (a.head_dim > kMaxHeadDim || a.v_dim > 64 * kMaxVChunks) return HYMETA_ERR_UNSUPPORTED;
  if (a.bias_mode < HYMETA_BIAS_NONE || a.bias_mode > HYMETA_BIAS_LINEAR_DISTANCE) return HYMETA_ERR_UNSUPPORTED;
  if (a.kv_layout < HYMETA_KV_KEY_THEN_VALUE || a.kv_layout > HYMETA_KV_SCALED_KEY) return HYMETA_ERR_UNSUPPORTED;
  if (a.kv_layout == HYMETA_KV_SCALED_KEY && (a.v_dim != a.head_dim || reinterpret_cast<uintptr_t>(a.kv_cache) % 16 != 0)) return HYMETA_ERR_INVALID_ARG;
  if (a.window_left >= 0 && a.keep_first < 0) return HYMETA_ERR_INVALID_ARG;
  if (a.chunk < 0 || (a.chunk > 0 && (a.window_left >= 0 || a.keep_first != 0))) return HYMETA_ERR_INVALID_ARG;
  if (a.kv_layout == HYMETA_KV_VALUE_IN_KEY && a.v_dim > a.head_dim) return HYMETA_ERR_INVALID_ARG;
  if (a.num_tokens == 0 || a.num_seqs == 0) return HYMETA_OK;
  if (!a.q || !a.kv_cache || !a.out || !a.block_tables || !a.query_start_loc || !a.seq_lens) return HYMETA_ERR_INVALID_ARG;
  if (a.bias_mode != HYMETA_BIAS_NONE && (!a.bias_a || (a.bias_mode == HYMETA_BIAS_LOG_DISTANCE && !a.bias_b))) return HYMETA_ERR_INVALID_ARG;
  if (a.elem_gate && a.elem_gate_stride_t < static_cast<int64_t>(a.num_heads) * a.v_dim) return HYMETA_ERR_INVALID_ARG;
  if (a.softcap < 0.f || (a.head_gate && a.head_gate_stride_t < a.num_heads)) return HYMETA_ERR_INVALID_ARG;
  if (a.num_heads > 65535) return HYMETA_ERR_UNSUPPORTED;
  hipStream_t st = begin_launches(stream);
  if (mfma_shape(a) && a.max_query_len >= 1 && a.max_seq_len >= 1) {
    const size_t need = hymeta_sink_attention_workspace_bytes(a.num_seqs, a.num_heads, a.num_kv_heads, a.v_dim, a.max_seq_len);
    if (!a.workspace || a.workspace_bytes < need) return HYMETA_ERR_WORKSPACE;
    if (a.num_seqs > 65535 || a.num_heads > 65535) return HYMETA_ERR_UNSUPPORTED;
    if (a.kv_layout == HYMETA_KV_VALUE_IN_KEY) {
      if (a.v_dim == 64) return a.head_dim == 96 ? launch_mfma<96, 64, HYMETA_KV_VALUE_IN_KEY>(a, st) : launch_mfma<128, 64, HYMETA_KV_VALUE_IN_KEY>(a, st);
      if (a.v_dim == 128) return a.head_dim == 160 ? launch_mfma<160, 128, HYMETA_KV_VALUE_IN_KEY>(a, st) : launch_mfma<192, 128, HYMETA_KV_VALUE_IN_KEY>(a, st);
      return a.v_dim == 256 ? launch_wide_latent<256>(a, st) : a.v_dim == 384 ? launch_wide_latent<384>(a, st) : launch_wide_latent<512>(a, st);
    }
    if (a.kv_layout == HYMETA_KV_SCALED_KEY) {
      constexpr int kScaled = HYMETA_KV_SCALED_KEY;
      return a.head_dim == 32 ? launch_mfma<32, 32, kScaled>(a, st) : a.head_dim == 64 ? launch_mfma<64, 64, kScaled>(a, st)
           : a.head_dim == 96 ? launch_mfma<96, 96, kScaled>(a, st) : launch_mfma<128, 128, kScaled>(a, st);
    }
    if (a.kv_layout == HYMETA_KV_SHARED_KEY) {
      constexpr int kShared = HYMETA_KV_SHARED_KEY;
      if (a.v_dim == 64)
        return a.head_dim == 64 ? launch_mfma<64, 64, kShared>(a, st) : a.head_dim == 128 ? launch_mfma<128, 64, kShared>(a, st)
             : a.head_dim == 256 ? launch_mfma<256, 64, kShared>(a, st) : launch_mfma<512, 64, kShared>(a, st);
      return a.head_dim == 64 ? launch_mfma<64, 128, kShared>(a, st) : a.head_dim == 128 ? launch_mfma<128, 128, kShared>(a, st)
           : a.head_dim == 256 ? launch_mfma<256, 128, kShared>(a, st) : launch_mfma<512, 128, kShared>(a, st);
    }
    if (a.head_dim == 64 && a.v_dim == 64) return launch_mfma<64, 64>(a, st);
    if (a.head_dim == 64 && a.v_dim == 128) return launch_mfma<64, 128>(a, st);
    if (a.head_dim == 128 && a.v_dim == 64) return launch_mfma<128, 64>(a, st);
    return launch_mfma<128, 128>(a, st);
  }
  const dim3 grid(a.num_tokens, a.num_heads);
  if (a.act_dtype == HYMETA_BF16) hipLaunchKernelGGL(sink_attention_rows_kernel<ActBf16>, grid, dim3(64), 0, st, a);
  else hipLaunchKernelGGL(sink_attention_rows_kernel<ActF32>, grid, dim3(64), 0, st, a);
  return launch_status();
}
