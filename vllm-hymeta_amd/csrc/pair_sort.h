// The (token, choice) pairs of a routed block, counted and ordered by expert, in one workgroup.
#pragma once

#include "act_types.h"

namespace hymeta {
namespace {

constexpr int kSortThreads = 1024;

struct PairSort {
  const int32_t* ids;            // expert of every pair; from `experts` on: an identity expert's, left out
  int pairs, experts;
  int local_begin, local_end;    // pairs of other experts are counted, but get no slot (pair_pos -1)
  int32_t *expert_offsets, *sorted_pair, *pair_pos;
};

// One workgroup: counts the pairs per expert in LDS, prefix, slots (the order inside an expert's run depends on the atomics'
// arrival; every pair's row is computed on its own, so the results do not).  Bound by the trips to memory of a thread's pairs,
// eight of which are asked for at once, and the counters' conflicts.  Ranks by ballots, 16 experts a wave, took 17 us on
// 8192 pairs: one compute unit issues all of it.
__global__ __launch_bounds__(kSortThreads) void sort_pairs_kernel(PairSort s) {
  __shared__ int s_count[HYMETA_MOE_TABLE_MAX_EXPERTS];
  __shared__ int s_off[HYMETA_MOE_TABLE_MAX_EXPERTS + 1];
  constexpr int kAtOnce = 8;
  const int tid = threadIdx.x, E = s.experts;
  for (int e = tid; e < E; e += kSortThreads) s_count[e] = 0;
  __syncthreads();
  auto each_pair = [&](auto f) {
    for (int p0 = tid; p0 < s.pairs; p0 += kAtOnce * kSortThreads) {
      int id[kAtOnce];
#pragma unroll
      for (int i = 0; i < kAtOnce; ++i) id[i] = s.ids[min(p0 + i * kSortThreads, s.pairs - 1)];
#pragma unroll
      for (int i = 0; i < kAtOnce; ++i)
        if (p0 + i * kSortThreads < s.pairs) f(p0 + i * kSortThreads, id[i]);
    }
  };
  each_pair([&](int, int e) {
    if (e < E) atomicAdd(&s_count[e], 1);
  });
  __syncthreads();
  if (tid == 0) {
    int run = 0;
    for (int e = 0; e < E; ++e) {
      s_off[e] = run;
      run += s_count[e];
    }
    s_off[E] = run;
  }
  __syncthreads();
  for (int e = tid; e <= E; e += kSortThreads) s.expert_offsets[e] = s_off[e];
  for (int e = tid; e < E; e += kSortThreads) s_count[e] = 0;
  __syncthreads();
  each_pair([&](int p, int e) {
    int place = -1;
    if (e < E && e >= s.local_begin && e < s.local_end) {
      place = s_off[e] + atomicAdd(&s_count[e], 1);
      s.sorted_pair[place] = p;
    }
    s.pair_pos[p] = place;
  });
}

}  // namespace
}  // namespace hymeta
