// Prompts' portions of the attention over paged rows, key and value apart, up to 128 elements each, or one key of 256 or 512
// for all heads: included by sink_attn.hip.
#pragma once

#include "row_attn.h"

namespace hymeta {
namespace {

// Grid, rows, softmax and the parts of the weights as in row_prefill_kernel.  A wave's step is a pipeline over two tiles: the
// products of the scores of tile t + 1, then those of tile t's weights with its values, with vector work of other keys between
// them, the weights of tile t first and, as far as a rule asks for more than a scaling, the scores of tile t + 1 behind them.
// The matrix pipe so runs under the wave's own vector work.  Keys and values lie in images of their own, two each; what a tile's
// bookkeeping needs is worked out in front of the loop.
//
// Bound by the vector and the matrix pipe together: with a logarithmic bias they are busy 69 and 56 % of the time, the waves wait 15 %
// of theirs, and the clock is 1.9 GHz, where kernels that use either pipe less run at 2.4.  Row_prefill_kernel -> here on one box:
// 8192 rows x 28 heads of 128 with 4 key/value heads, logarithmic bias 754 -> 695 us, a window of 1024 201 -> 184; three portions
// of 700 behind 1000 94.8 -> 75; six of 324 behind 818, window 1024, 60.6 -> 49; four of 1500 behind 3000, 16 heads, chunks of
// 2048, 120 -> 111; 4000 rows capped, window 1024, 115 -> 108.
//
// Long keys (256 or 512 elements, which all heads share): one wave on a SIMD, whose registers then hold the queries (128), the
// weighted values and two tiles' scores (64 each); the images of 64 keys fill the LDS.  All weights of a tile are formed under the
// products of the next scores, four fifths of the step.  A wave of 16 rows that read the whole tile for them was bound by LDS; with
// 32 rows the matrix pipe (1.45 us a tile of 64 keys of 512) and the lone wave's issue add up: 2.76 us a tile, of which the copies'
// issue takes 0.36, exponentials and rounding 0.30, half of the key reads 0.09; around a block's tiles lie about 12 us, half of them
// its queries' 128 KB from memory, which all compute units ask for at once.  28 heads, 4 value heads of 128, window 1024, with a
// workgroup per 64 rows and head -> here, back to back: 8192 rows 1275 -> 450 us; 2048 behind 4096 390 -> 134; four of 300 behind 2000 208 -> 71; five
// of 10 behind 5955, keys cut into slices, 97 -> 26; 300 rows alone 33 -> 26.  Level or slower: copies issued among the slots (459),
// fragments read 10 slots ahead (452), no barrier to the compiler's order between slots (a sixth slower).
template <int D, int DV, int Layout, int Rule>
__global__ __launch_bounds__(256, D > 192 ? 1 : 2) void row_pipe_kernel(hymeta_sink_attention_args a, PortionSlices ps) {
  static_assert(Layout == HYMETA_KV_KEY_THEN_VALUE || Layout == HYMETA_KV_SHARED_KEY, "the value lies apart from the key");
  constexpr bool Shared = Layout == HYMETA_KV_SHARED_KEY, Wide = D > 192;
  constexpr int kSteps = D / 16, CB = DV / 32, kWaves = 4, kRows = 32 * kWaves;
  constexpr int kKeyChunks = D / 8, kValueChunks = DV / 8, kKeyPitch = 2 * D, kValuePitch = 2 * DV;
  static_assert(kRows == kPortionRows && (D == 64 || D == 128 || D == 256 || D == 512) && (DV == 64 || DV == 128), "an instruction copies whole rows");
  constexpr int kKeyImage = kTileKeys * kKeyPitch, kValueImage = kTileKeys * kValuePitch;
  __shared__ __attribute__((aligned(16))) char s_k[2][kKeyImage];
  __shared__ __attribute__((aligned(16))) char s_v[2][kValueImage];

  auto uniform = [](int x) __attribute__((always_inline)) { return __builtin_amdgcn_readfirstlane(x); };
  const int group = uniform(a.num_heads / a.num_kv_heads);
  const int item = uniform(blockIdx.x / a.num_kv_heads), g = blockIdx.x - item * a.num_kv_heads;
  const int number = uniform(item / ps.splits), split = item - number * ps.splits;
  const PieceAt block = portion_block(a, number, ps);
  const int s = uniform(block.seq), row0 = block.row0, q = block.rows, rows = q * group;
  if (s < 0) return;
  const int r0 = ((rows - 1) / kRows - uniform(block.index)) * kRows;     // (the longest rows first)
  const int lane = threadIdx.x & 63, n = lane & 31, hh = lane >> 5;
  const int wave = uniform(threadIdx.x >> 6);
  const int ctx = a.seq_lens[s] - q, w0 = r0 + 32 * wave;
  auto pos_of = [&](int row) __attribute__((always_inline)) { return ctx + uniform(min(row, rows - 1) / group); };
  const int p_hi = pos_of(r0 + kRows - 1);
  const BlockKeys keys = block_keys<kTileKeys>(a, pos_of(r0), p_hi);
  const int splits = uniform(keys.slices(ps));
  if (split >= splits) return;
  const int from = uniform(keys.from), kept = uniform(keys.kept), tiles = uniform(keys.tiles);
  const int per = uniform((tiles + splits - 1) / splits), t_lo = split * per, t_hi = min(tiles, t_lo + per);
  auto key0 = [&](int t) __attribute__((always_inline)) { return t < kept ? t * kTileKeys : from + (t - kept) * kTileKeys; };

  // this lane's row (past the last one: that one again); it holds the row's scores against half of a tile's keys, its partner
  // lane +- 32 the others
  const bool ok = w0 + n < rows;
  const int r = min(w0 + n, rows - 1), qi = r / group, h = g * group + r - qi * group, pos = ctx + qi;
  const float ba = a.bias_mode ? -a.bias_a[h] : 0.f, bb = a.bias_mode == HYMETA_BIAS_LOG_DISTANCE ? a.bias_b[h] : 0.f;
  const bool sink = a.sink && splits == 1;            // (of several slices of the keys none has the sink: the merge adds it)
  bool unset = !sink;                                 // the row has seen neither a key nor a sink
  float ref = sink && a.sink_logits ? a.sink_logits[h] * 1.4426950408889634f : 0.f;      // of the exponentials, base 2
  float l = sink && hh == 0 ? 1.f : 0.f;              // the sink's exp(ref - ref), counted once per row
  // (a scale of 0: the queries are 0 and the scale 1, so that a masked score's -inf is not multiplied by 0)
  const float scale = a.scale == 0.f ? 1.f : fabsf(a.scale), scale2 = scale * 1.4426950408889634f;
  const float cap_in = a.softcap > 0.f ? scale / a.softcap : 0.f, cap2 = a.softcap * 1.4426950408889634f;
  u32x4 qf[kSteps];                                   // (with the scale's sign, so that scores grow with their products)
  auto load_queries = [&]() __attribute__((always_inline)) {
    const uint16_t* qrow = static_cast<const uint16_t*>(a.q) + static_cast<int64_t>(row0 + qi) * a.q_stride_t + static_cast<int64_t>(h) * D + 8 * hh;
    const uint32_t sign = a.scale < 0.f ? 0x80008000u : 0u, kept_bits = a.scale == 0.f ? 0u : ~0u;
#pragma unroll
    for (int st = 0; st < kSteps; ++st) {
      qf[st] = ld16g(qrow + 16 * st);
#pragma unroll
      for (int e = 0; e < 4; ++e) qf[st][e] = (qf[st][e] & kept_bits) ^ sign;
    }
  };
  if (!Wide) load_queries();
  f32x16 o[CB];                                       // O^T: columns 32 cb + 8 i + 4 hh + e of the lane's row, i, e < 4
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[cb][i] = 0.f;

  // tiles that the wave's rows see (the kept ones: any), and those [clear_lo, clear_hi) that they all see whole
  const bool any = w0 < rows;
  const int w_lo = pos_of(w0), w_hi = pos_of(w0 + 31);
  const int seen_lo = kept > 0 ? 0 : uniform(first_key(a, max(w_lo, 0)) - from) / kTileKeys, seen_hi = any && w_hi >= 0 ? (w_hi - from) / kTileKeys + kept : -1;
  const int clear_lo = kept + max(0, uniform(first_key(a, max(w_hi, 0))) - from + kTileKeys - 1) / kTileKeys, clear_hi = w_lo >= from ? kept + (w_lo + 1 - from) / kTileKeys : 0;

  // ---- copies: an instruction takes whole rows of an image, the wave's i-th the rows kRowsEach (wave + 4 i) ..
  constexpr int kKeyRows = 64 / kKeyChunks, kValueRows = 64 / kValueChunks;
  const int64_t row_bytes = 2 * (Shared ? D + static_cast<int64_t>(a.num_kv_heads) * DV : static_cast<int64_t>(a.num_kv_heads) * (D + DV));
  const char* kglob = static_cast<const char*>(a.kv_cache) + (Shared ? 0 : 2 * static_cast<int64_t>(g) * (D + DV));
  const char* vglob = kglob + 2 * (Shared ? D + g * DV : D);
  const int32_t* bt = a.block_tables + static_cast<int64_t>(s) * a.block_table_stride;
  const int shift = __builtin_ctz(a.block_size), mask = a.block_size - 1;
  auto value_twist = [](int row) __attribute__((always_inline)) { return kValueChunks == 16 ? (row & 3) << 2 : (row & 2) << 1; };
  // (long keys: an instruction's few rows leave the chunk order to its number as well, in bits that no row's offset has)
  auto key_chunk = [&](int ln, int i) __attribute__((always_inline)) -> uint32_t {
    return 16 * ((ln % kKeyChunks) ^ ChunkOrder<kKeyChunks>::twist(kKeyRows * (wave + kWaves * i) + ln / kKeyChunks));
  };
  auto turn = [](int i) __attribute__((always_inline)) -> uint32_t { return 16 * ((kKeyRows * kWaves * i >> 2) & 3); };
  auto value_chunk = [&](int ln) __attribute__((always_inline)) -> uint32_t { return 16 * ((ln % kValueChunks) ^ value_twist(ln / kValueChunks)); };
  const uint32_t kplace = static_cast<uint32_t>(lane / kKeyChunks * row_bytes) + key_chunk(lane, 0);
  const uint32_t vplace = static_cast<uint32_t>(lane / kValueChunks * row_bytes) + value_chunk(lane);
  const char* kwave = kglob + kKeyRows * wave * row_bytes;
  const char* vwave = vglob + kValueRows * wave * row_bytes;
  // the first `whole` tiles: 64 rows of one page that some row of the block sees (the last one may have fewer)
  const int whole = a.block_size >= kTileKeys && row_bytes < (1 << 27) ? (p_hi + 1 - key0(tiles - 1) >= kTileKeys ? tiles : tiles - 1) : 0;
  // lane = tile % 64 holds where a tile's first row lies, for 64 tiles from the last refill on
  int64_t tile_at = 0;
  auto refill = [&](int t) __attribute__((always_inline)) {
    const int tile = t + ((lane - t) & 63);
    if (tile >= min(whole, t_hi)) return;
    const int j = key0(tile);
    tile_at = ((static_cast<int64_t>(bt[j >> shift]) << shift) + (j & mask)) * row_bytes;
  };
  auto copy_tile = [&](int t, bool value, char* image) __attribute__((always_inline)) {
    const int each = value ? kValueRows : kKeyRows, copies = (value ? kValueChunks : kKeyChunks) / kWaves;
    if (t < whole) {
      const uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(tile_at), t & 63);
      const int hi = __builtin_amdgcn_readlane(static_cast<int>(tile_at >> 32), t & 63);
      const char* base = (value ? vwave : kwave) + ((static_cast<int64_t>(hi) << 32) | lo);
#pragma unroll
      for (int i = 0; i < copies; ++i) {
        copy16_to_lds(base, value ? vplace : kplace ^ turn(i), image + 1024 * (wave + kWaves * i));
        base += kWaves * each * row_bytes;
      }
      return;
    }
    // rows past the last that the block sees repeat it (their weights are zero)
    int ln = lane;
    asm volatile("" : "+v"(ln));                      // (nothing of this is kept in registers over the other tiles)
    const int j0 = key0(t), row_in = ln / (value ? kValueChunks : kKeyChunks);
#pragma unroll Wide ? 4 : 1
    for (int i = 0; i < copies; ++i) {
      const int j = min(j0 + each * (wave + kWaves * i) + row_in, p_hi);
      const int64_t row = (static_cast<int64_t>(bt[j >> shift]) << shift) + (j & mask);
      copy16_to_lds((value ? vglob : kglob) + row * row_bytes + (value ? value_chunk(ln) : key_chunk(ln, i)), image + 1024 * (wave + kWaves * i));
    }
  };

  // ---- LDS offsets of this lane's fragments.  Keys: row n, chunk 2 st + hh.  Values: a tile's 16-key step i takes its keys
  // 8 i + 4 hh + e and 32 keys further on, which are the keys whose weights the lane holds
  constexpr int kOffsets = kSteps < 8 ? kSteps : 8;   // (those of a chunk 16 further on lie 256 bytes behind)
  int koff[kOffsets], voff[CB];
#pragma unroll
  for (int st = 0; st < kOffsets; ++st) koff[st] = n * kKeyPitch + 16 * ((2 * st + hh) ^ ChunkOrder<kKeyChunks>::twist(n));
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const int R = 4 * hh + ((lane & 15) >> 2), chunk = 4 * cb + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    voff[cb] = R * kValuePitch + 16 * (chunk ^ value_twist(R)) + 8 * (lane & 1);
  }
  // (long keys: LDS addresses, of which the images' are out of an instruction's reach, moved from image to image behind each tile)
  uint32_t kat[kOffsets], vat[CB];
#pragma unroll
  for (int i = 0; i < kOffsets; ++i) kat[i] = lds_address(s_k[0]) + koff[i];
#pragma unroll
  for (int i = 0; i < CB; ++i) vat[i] = lds_address(s_v[0]) + voff[i];
  auto other_image = [&](auto& at, int count, int by) __attribute__((always_inline)) {
    if (!Wide) return;
#pragma unroll
    for (int i = 0; i < count; ++i) {
      at[i] += by;
      asm volatile("" : "+v"(at[i]));                 // (not formed from the first image's for every read)
    }
  };
  f32x16 sa[2], sb[2];                                // scores: keys 32 x + 8 i + 4 hh + e of a tile, element 4 i + e of [x]
  // Fragment f of a step: f < 2 kSteps of the keys (step f / 2 of the head, half f % 2 of the tile), else of the values (16 keys
  // (f - 2 kSteps) / CB, columns 32 (f % CB) ..)
  constexpr int NQ = 2 * kSteps, NF = NQ + 4 * CB, kAhead = Wide ? 6 : 3;
  constexpr int kUnder = Wide ? 16 : 7;               // of a tile's 16 slices of weights: under the products of the scores
  auto fragment = [&](const char* kimg, const char* vimg, int f) __attribute__((always_inline)) {
    if (Wide && f < NQ) return *(const __attribute__((address_space(3))) u32x4*)(kat[(f >> 1) % kOffsets] + (f >> 1) / kOffsets * 256 + (f & 1) * 32 * kKeyPitch);
    if (Wide) {
      const uint32_t v = vat[(f - NQ) % CB] + (f - NQ) / CB * 8 * kValuePitch;
      const u32x2 v0 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_bf16x4*)v));
      const u32x2 v1 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_bf16x4*)(v + 32 * kValuePitch)));
      return u32x4{v0[0], v0[1], v1[0], v1[1]};
    }
    if (f < NQ) return ld16(kimg + koff[(f >> 1) % kOffsets] + (f >> 1) / kOffsets * 256 + (f & 1) * 32 * kKeyPitch);
    const char* v = vimg + voff[(f - NQ) % CB] + (f - NQ) / CB * 8 * kValuePitch;
    const u32x2 v0 = __builtin_bit_cast(u32x2, read_transposed(v)), v1 = __builtin_bit_cast(u32x2, read_transposed(v + 32 * kValuePitch));
    return u32x4{v0[0], v0[1], v1[0], v1[1]};
  };
  auto product = [](const u32x4& x, const u32x4& y, const f32x16& c) __attribute__((always_inline)) {
    return mfma32(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), c);
  };
  // Scores in the base-2 domain, less the reference, where that takes more than a scaling: elements e of both halves.  (The
  // logarithm's argument comes from the exact distance: formed from the tile's it would lose 64 of the coefficient's ulps, on the
  // nearest keys of a steep bias all of itself.)
  auto bend = [&](f32x16 (&sc)[2], int e, float d0) __attribute__((always_inline)) {
    if (Rule == kPlain) return;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const float away = static_cast<float>(32 * x + 8 * (e >> 2) + (e & 3));
      if (Rule == kAnyRule) {                         // (no cap: the product scaled; no bias: ba = bb = 0)
        const float plain = fmaf(sc[x][e], scale2, -ref), capped = fmaf(cap2, tanh_fast(sc[x][e] * cap_in), -ref);
        sc[x][e] = fmaf(ba, __builtin_amdgcn_logf(fmaf(bb, d0 - away, 1.f)), a.softcap > 0.f ? capped : plain);
      } else if (Rule == kLogBias) sc[x][e] = fmaf(ba, __builtin_amdgcn_logf(fmaf(bb, d0 - away, 1.f)), fmaf(sc[x][e], scale2, -ref));
      else sc[x][e] = fmaf(cap2, tanh_fast(sc[x][e] * cap_in), -ref);
    }
  };
  auto distance = [&](int t) __attribute__((always_inline)) { return static_cast<float>(pos - key0(t) - 4 * hh); };
  // After the scores of tile t: mask them, move the reference where they ask for it
  auto settle = [&](int t, f32x16 (&sc)[2], float mx) __attribute__((always_inline)) {
    if (t < clear_lo || t >= clear_hi) {
      const int first = first_key(a, pos);
      int j0 = key0(t) + 4 * hh;
      asm volatile("" : "+v"(j0));                    // (keeps the compiler from working this out on every tile)
      mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        const int j = j0 + 32 * (i >> 4) + 8 * ((i & 15) >> 2) + (i & 3);
        sc[i >> 4][i & 15] = (j <= pos && (j >= first || j < a.keep_first)) ? sc[i >> 4][i & 15] : -INFINITY;
        mx = __builtin_elementwise_maximum(mx, sc[i >> 4][i & 15]);
      }
    }
    const float over = Rule == kPlain ? fmaf(mx, scale2, -ref) : mx;
    if (__any(over > kLazyMax2 || (unset && mx > -INFINITY))) {
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float top = Rule == kPlain ? fmaf(mx, scale2, -ref) : mx;
      const bool up = top > kLazyMax2 || (unset && mx > -INFINITY);
      const float corr = up ? (unset ? 0.f : __builtin_amdgcn_exp2f(-top)) : 1.f;
      if (up) ref += top;
      unset = unset && !up;
      l *= corr;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) o[cb] *= corr;
      if (Rule != kPlain) {
#pragma unroll
        for (int i = 0; i < 32; ++i) sc[i >> 4][i & 15] -= up ? top : 0.f;
      }
    }
  };
  auto top_of = [&](const f32x16 (&sc)[2], float mx, int e) __attribute__((always_inline)) {
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(mx, sc[0][e]), sc[1][e]);
  };
  // The first tile's scores alone
  auto lead = [&](int t, const char* kimg, f32x16 (&next)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 32; ++i) next[i >> 4][i & 15] = 0.f;
#pragma unroll
    for (int f = 0; f < NQ; ++f) next[f & 1] = product(fragment(kimg, kimg, f), qf[f >> 1], next[f & 1]);
    const float d0 = distance(t);
    float mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      bend(next, e, d0);
      mx = top_of(next, mx, e);
    }
    settle(t, next, mx);
  };
  // Weights of tile t (scores `cur`) times its values, and the scores of tile t + 1.  A slot is a fragment's products, the read of
  // one a few slots ahead and a slice of the vector work: pairs of weights (kUnder of 16 under the scores' products), then scores
  auto step = [&](int t, const char* kimg, const char* vimg, f32x16 (&cur)[2], f32x16 (&next)[2]) __attribute__((always_inline)) {
    u32x4 fr[NF], hi[4], lo[4];                       // a weight's bf16 parts, of 16 keys, as the second product's operand
    const float d0 = distance(t + 1);
    float mx = -INFINITY;
#pragma unroll
    for (int f = 0; f < kAhead; ++f) fr[f] = fragment(kimg, vimg, f);
#pragma unroll
    for (int i = 0; i < 32; ++i) next[i >> 4][i & 15] = 0.f;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      if (f + kAhead < NF) fr[f + kAhead] = fragment(kimg, vimg, f + kAhead);
      if (f < NQ) {
        next[f & 1] = product(fr[f], qf[f >> 1], next[f & 1]);
      } else {
        const int i = (f - NQ) / CB, cb = (f - NQ) % CB;
        o[cb] = product(fr[f], hi[i], o[cb]);
        o[cb] = product(fr[f], lo[i], o[cb]);
      }
      const int p_lo = f < NQ ? f * kUnder / NQ : kUnder + (f - NQ) * (16 - kUnder) / (5 * CB / 2);
      const int p_hi_ = f < NQ ? (f + 1) * kUnder / NQ : kUnder + (f + 1 - NQ) * (16 - kUnder) / (5 * CB / 2);
#pragma unroll
      for (int p = p_lo; p < (p_hi_ < 16 ? p_hi_ : 16); ++p) {
        const int i = p >> 2, e = p & 3, x = 4 * i + 2 * (e & 1);
        const float w0_ = __builtin_amdgcn_exp2f(Rule == kPlain ? fmaf(cur[e >> 1][x], scale2, -ref) : cur[e >> 1][x]);
        const float w1_ = __builtin_amdgcn_exp2f(Rule == kPlain ? fmaf(cur[e >> 1][x + 1], scale2, -ref) : cur[e >> 1][x + 1]);
        l += w0_ + w1_;
        const uint32_t pair = pack_bf16x2(w0_, w1_);
        hi[i][e] = pair;
        lo[i][e] = pack_bf16x2(w0_ - lo_bf(pair), w1_ - hi_bf(pair));
      }
      // the next tile's scores, over the slots behind the first product
      const int e_lo = f <= NQ ? 0 : (f - NQ - 1) * 16 / (NF - NQ - 1), e_hi = f <= NQ ? 0 : (f - NQ) * 16 / (NF - NQ - 1);
#pragma unroll
      for (int e = e_lo; e < e_hi; ++e) {
        if (Rule != kAnyRule) bend(next, e, d0);
        if (Rule != kAnyRule) mx = top_of(next, mx, e);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (Rule == kAnyRule) {                           // (in the slots it takes the loop past what the compiler unrolls)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        bend(next, e, d0);
        mx = top_of(next, mx, e);
      }
    }
    asm volatile("" : "+v"(mx), "+v"(l));
    if (t + 1 < t_hi) settle(t + 1, next, mx);
  };

#pragma unroll
  for (int i = 0; i < 32; ++i) sa[i >> 4][i & 15] = sb[i >> 4][i & 15] = -INFINITY;
  if (t_lo < t_hi) {
    refill(t_lo);
    copy_tile(t_lo, false, s_k[0]);
    if (Wide) load_queries();                         // (32 KB a wave, which the first keys don't wait for)
    copies_landed_barrier();
    copy_tile(t_lo, true, s_v[0]);
    if (t_lo + 1 < t_hi) copy_tile(t_lo + 1, false, s_k[1]);
    lead(t_lo, s_k[0], sa);
    other_image(kat, kOffsets, kKeyImage);
    // tile t: images (t - t_lo) & 1
    auto iterate = [&](int t, auto image, f32x16 (&cur)[2], f32x16 (&next)[2]) __attribute__((always_inline)) {
      constexpr int even = decltype(image)::value;
      copies_landed_barrier();                        // keys of t + 1 and values of t are there, and nobody reads the images they leave
      if (t + 2 < t_hi) copy_tile(t + 2, false, s_k[even]);
      if (t + 1 < t_hi) copy_tile(t + 1, true, s_v[1 - even]);
      if (t + 1 < seen_lo || t > seen_hi) {
#pragma unroll
        for (int i = 0; i < 32; ++i) next[i >> 4][i & 15] = -INFINITY;
      } else {
        step(t, s_k[1 - even], s_v[even], cur, next);
      }
      other_image(kat, kOffsets, even ? kKeyImage : -kKeyImage);
      other_image(vat, CB, even ? -kValueImage : kValueImage);
    };
    constexpr std::integral_constant<int, 0> first{};
    constexpr std::integral_constant<int, 1> second{};
    int t = t_lo;
    for (; t + 1 < t_hi; t += 2) {
      iterate(t, first, sa, sb);
      iterate(t + 1, second, sb, sa);
      if (((t - t_lo) & 31) == 30) refill(t + 2);
    }
    if (t < t_hi) iterate(t, first, sa, sb);
  }
  l += __shfl_xor(l, 32, 64);
  if (!ok) return;
  const int64_t token = row0 + qi;
  if (splits > 1) {
    float* part = ps.parts + ((token * a.num_heads + h) * ps.splits + split) * partial_row_floats(DV);
    if (hh == 0) part[DV] = unset ? -INFINITY : ref, part[DV + 1] = l;
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
