// Activation element types of the kernels that run in bf16 or in fp32 (act_dtype of their argument
// structs): loads widen to fp32, stores round once.
#pragma once

#include <algorithm>
#include <utility>

#include "common.h"

namespace hymeta {

struct ActBf16 {
  typedef uint16_t elem;
  static constexpr int kDtype = HYMETA_BF16;
  static __device__ __forceinline__ float ld(const elem* p) { return bf2f(*p); }
  static __device__ __forceinline__ void st(elem* p, float v) { *p = f2bf(v); }
  static __device__ __forceinline__ float round(float v) { return bf16_round(v); }
  // four consecutive elements, 8-byte aligned
  static __device__ __forceinline__ void ld4(const elem* p, float* v) {
    const u32x2 t = *reinterpret_cast<const u32x2*>(p);
    v[0] = lo_bf(t[0]), v[1] = hi_bf(t[0]), v[2] = lo_bf(t[1]), v[3] = hi_bf(t[1]);
  }
  static __device__ __forceinline__ void st4(elem* p, const float* v) {
    *reinterpret_cast<u32x2*>(p) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  }
  // fp32 in, fp32 out, the hardware's exponential (about 2 ulp): where the inputs carry 8 bits
  static __device__ __forceinline__ float sigmoid(float x) { return 1.f / (1.f + __expf(-x)); }
};

struct ActF32 {
  typedef float elem;
  static constexpr int kDtype = HYMETA_F32;
  static __device__ __forceinline__ float ld(const elem* p) { return *p; }
  static __device__ __forceinline__ void st(elem* p, float v) { *p = v; }
  static __device__ __forceinline__ float round(float v) { return v; }
  // four consecutive elements, 16-byte aligned
  static __device__ __forceinline__ void ld4(const elem* p, float* v) {
    const f32x4 t = *reinterpret_cast<const f32x4*>(p);
    v[0] = t[0], v[1] = t[1], v[2] = t[2], v[3] = t[3];
  }
  static __device__ __forceinline__ void st4(elem* p, const float* v) { *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]}; }
  static __device__ __forceinline__ float sigmoid(float x) { return 1.f / (1.f + expf(-x)); }
};

inline bool act_dtype_ok(int d) { return d == HYMETA_BF16 || d == HYMETA_F32; }

// Sum over the 64 lanes of a wave, result in every lane.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// Sum over a workgroup of `Waves` waves; `red` is Waves floats of LDS.  Every thread gets the sum.  The
// summation order is fixed (lanes by butterfly, waves in order), so a row's statistic does not depend
// on which workgroup computes it.
template <int Waves>
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  __syncthreads();                       // red may still be read from the call before
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int w = 0; w < Waves; ++w) s += red[w];
  return s;
}

// Sequence of a token row: the s with query_start_loc[s] <= t < query_start_loc[s + 1].
__device__ __forceinline__ int seq_of_row(const int32_t* query_start_loc, int num_seqs, int t) {
  int lo = 0, hi = num_seqs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (query_start_loc[mid] <= t) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// How many portions of max_query_len rows the rows of a step are worth, beyond the one row that every sequence has: the work
// beside which single rows (decode) and short portions count for what they are.
inline int64_t long_portions(int num_tokens, int num_seqs, int max_query_len) {
  const int64_t more = std::max(max_query_len - 1, 1);
  return std::max<int64_t>(1, std::min<int64_t>(num_seqs, (static_cast<int64_t>(num_tokens) - num_seqs + more - 1) / more));
}

template <int X> struct Const { static constexpr int value = X; };

// f(0), f(1), ... f(N - 1) with constants
template <int N, typename F, int... I>
__device__ __forceinline__ void unrolled(const F& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void unrolled(const F& f) { unrolled<N>(f, std::make_integer_sequence<int, N>{}); }

// Inclusive sums over a wave's lanes: within 16 lanes, then the rows of 16 lanes before.
template <typename T>
__device__ __forceinline__ T lane_sums(T x) {
  auto add = [&](auto ctrl, auto rows_mask) {
    x += __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, decltype(rows_mask)::value, 0xf, false));
  };
  add(Const<0x111>{}, Const<0xf>{}), add(Const<0x112>{}, Const<0xf>{}), add(Const<0x114>{}, Const<0xf>{}), add(Const<0x118>{}, Const<0xf>{});
  add(Const<0x142>{}, Const<0xa>{}), add(Const<0x143>{}, Const<0xc>{});
  return x;
}

// Every sequence of a step falls into pieces(its rows) pieces, numbered through: the sequence of piece `number` (wave-uniform;
// -1: there is no such piece), that one's rows, and which of its pieces it is.  A wave takes 64 sequences at a time.
struct PieceAt { int seq, row0, rows, index; };
template <typename F>
__device__ __forceinline__ PieceAt piece_at(const int32_t* query_start_loc, int num_seqs, int number, const F& pieces) {
  const int lane = threadIdx.x & 63;
  for (int s0 = 0; s0 < num_seqs; s0 += 64) {
    const int s = min(s0 + lane, num_seqs - 1), row0 = query_start_loc[s], rows = s0 + lane < num_seqs ? query_start_loc[s + 1] - row0 : 0;
    const int mine = pieces(rows), upto = lane_sums(mine);
    const uint64_t past = __ballot(number < upto);
    if (past != 0) {
      const int at = __builtin_ctzll(past);
      return PieceAt{s0 + at, __builtin_amdgcn_readlane(row0, at), __builtin_amdgcn_readlane(rows, at), number - __builtin_amdgcn_readlane(upto - mine, at)};
    }
    number -= __builtin_amdgcn_readlane(upto, 63);
  }
  return PieceAt{-1, 0, 0, 0};
}

__device__ __forceinline__ float sigmoid_exact(float x) { return 1.f / (1.f + expf(-x)); }

__device__ __forceinline__ float clamped_glu(float gate, float up, float limit, float alpha) {
  const float g = fminf(gate, limit);
  const float u = fminf(fmaxf(up, -limit), limit);
  return g * sigmoid_exact(alpha * g) * (u + 1.f);
}

}  // namespace hymeta
