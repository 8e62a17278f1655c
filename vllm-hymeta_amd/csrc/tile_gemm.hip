// Matrix products of prompts.  A workgroup of four waves forms 256 rows x 256 weight rows, 128 x 128 a wave in
// v_mfma_f32_16x16x32_bf16 / v_mfma_i32_16x16x64_i8 (in BYTES the two walk their operands identically); both operands
// are copied from memory straight into LDS, 128 bytes of every row a step, two steps' images.  Tiles of at most 128 rows take
// 64 x 128 a wave.
//
// What bounds it is power, then the way from L2 into LDS: with operands of zeros that every workgroup shares the loop runs at
// 2.0 PFLOP/s, with random ones at 1.55, a whole problem at 1.36 (8192 rows, 37888 x 3584 in bf16: 1640 us, 2000 through the
// tiles of 256 that waited for their rows in registers; the library's product 1680) and in int8 at 2.47 (900 us; 1120).  Hence
//  * 128 x 128 a wave: fragments are read from LDS as rarely as registers allow (256 accumulation registers, one wave on a
//    SIMD).  Products of 16 x 16 x 32 move half the accumulator bytes of 32 x 32 x 16 for the same work: 1390 against 1300
//    TFLOP/s.
//  * the order of instructions is fixed by hand: a fragment of the next half step is read behind every fourth product, a
//    copy asked for behind every sixth (all at once blocks the wave behind the address path; behind every eighth the last
//    copy has too little time).  The barrier that frees an image stands in front of a step's second half, whose fragments
//    are in registers by then.
//  * tiles are dealt to the eight dies in runs of 32 neighbours, which share an L2: 12 panels a step where a row of tiles
//    would read 33 (2030 -> 1810 us), and the dies' runs share what they read from memory (routed experts, 8192 rows of 3584
//    columns, both products: 3210 -> 2970 us against a run of experts a die).
//  * neighbours share the fetching of what comes from beyond their L2: each touches every 8th step of its x panel and every
//    deep-th of its w panel, ahead of the copies, as loads whose 4 bytes a line go to a scrap of LDS (1790 -> 1610 us;
//    all lines by all workgroups: 1880).
// One matrix of so few tiles that they leave the chip idle is cut along K instead (tile_gemm_slices): every unit takes a slice of
// one tile, whose fp32 sums a reducing consumer adds.
// Workgroups that walk their tiles as one stream of steps, the next one's copies ahead of the present one's sums, were built:
// 2 % slower in bf16 and level in int8 on 8192 rows, 6 % slower on 2048 rows of 8 experts (what is done once a tile costs every step,
// and nobody evens out tiles of few rows).
#include "tile_gemm.h"

#include "act_types.h"
#include "lds_copy.h"

#include <algorithm>
#include <type_traits>

namespace hymeta {
namespace {

constexpr int kTile = 256;                       // rows and weight rows of a tile
constexpr int kStep = 128;                       // bytes of a row in a step
constexpr int kImage = kTile * kStep;            // one operand's step
constexpr int kDies = 8, kUnits = 32;            // dies, and compute units of a die that share its L2
constexpr int kDeep = 4, kWide = 8;              // row and column tiles of a block of neighbours
constexpr int kMaxTileExperts = 64;              // a lane each
constexpr int kHalfRows = 128;                   // tiles of at most these rows take half the products
constexpr int kAhead = 3;                        // steps between a touched line and its products
constexpr int kMinSteps = 4;
constexpr int kMaxSlices = 16, kSliceSteps = 24, kFewSliceTiles = 32, kSliceSums = 14 << 20;      // tile_gemm_slices' rule

// f(0), f(1) .. f(N - 1) with the numbers as constants
template <int N, int I = 0, typename F>
__device__ __forceinline__ void each(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    each<N, I + 1>(f);
  }
}

template <bool I8> struct TileAcc { typedef f32x4 type; };
template <> struct TileAcc<true> { typedef i32x4 type; };

// c += a b, in place and in the order written: left to itself the compiler gives a product another destination than its
// addend and pays with copies between the register files (int8: 84 of them, with waits, beside 64 products).
template <bool I8>
__device__ __forceinline__ void tile_mma(const u32x4& a, const u32x4& b, typename TileAcc<I8>::type& c) {
  if constexpr (I8) asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

// Until the last products have left the matrix pipe: the compiler, which counts the cycles in front of a use, does not know
// them as products.  Stands at the end of every run of products, where it may move accumulators.
__device__ __forceinline__ void settle() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 9" :::);
  __builtin_amdgcn_sched_barrier(0);
}

// 16 bytes a lane (a row's piece) or 4 (a line's first bytes, a table's entry) from base + offset into LDS at `place` + 16 or 4
// times the lane, not through registers.
__device__ __forceinline__ void copy16(const char* base, uint32_t offset, uint32_t place) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(place), "v"(offset), "s"(base) : "memory");
}
__device__ __forceinline__ void copy4(const char* base, uint32_t offset, uint32_t place) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(place), "v"(offset), "s"(base) : "memory");
}

// Where a workgroup works: slots [row, row + rows) of expert e, column tile `col`; its place in the block of neighbours.
struct Place {
  int e, row, rows, col;
  int deep, depth;
  int slice, step0, steps;          // the steps of K it takes: all, or those of a slice
};

// The tiles of all experts stand in one order, a lane per expert.  An expert's tiles go in blocks of up to kDeep row tiles x
// kWide column tiles, the blocks of one run of columns next to each other: 32 tiles in a row are about one block, which a die's
// units take together (12 panels a step where a row of tiles would read 33), and the eight blocks of a round share what they
// read from memory.  The columns are swept once for every 32 row tiles, whose x stays in the last-level cache.  In a last, incomplete round of at most half the units every tile is cut into halves of 128 rows, which take
// 0.6 of a tile's time.  Wave-uniform; false: nothing to do.
__device__ __forceinline__ bool find_place(const TileGemmArgs& a, int lane, Place* p) {
  constexpr int kRound = kDies * kUnits;
  const int cols = a.N / kTile, experts = a.expert_offsets != nullptr ? a.expert_end - a.expert_begin : 1;
  int lo = 0, hi = a.max_rows;
  if (a.expert_offsets != nullptr) {
    const int i = a.expert_begin + min(lane, experts - 1);
    lo = a.expert_offsets[i], hi = a.expert_offsets[i + 1];
  }
  int upto = lane < experts ? ((hi - lo + kTile - 1) / kTile) * cols : 0;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int v = __shfl_up(upto, d, 64);
    if (lane >= d) upto += v;
  }
  const int total = __builtin_amdgcn_readlane(upto, 63), whole = total / kRound * kRound, rest = total - whole;
  const int block = blockIdx.x, die = block % kDies;
  int t, half = -1;
  if (block < whole) {
    t = block / kRound * kRound + die * kUnits + block % kRound / kDies;
  } else {
    const int first = rest * die / kDies, count = rest * (die + 1) / kDies - first;
    int j = (block - whole) / kDies;
    if (rest <= kRound / 2) {
      if (j >= 2 * count) return false;
      half = j >= count, j -= half ? count : 0;
    }
    if (j >= count) return false;
    t = whole + first + j;
  }
  const int at = __popcll(__ballot(upto <= t));              // experts whose tiles all lie in front of t
  const int of_expert = t - (at > 0 ? __builtin_amdgcn_readlane(upto, at - 1) : 0);
  lo = __builtin_amdgcn_readlane(lo, at), hi = __builtin_amdgcn_readlane(hi, at);
  constexpr int kSweep = kDeep * kDies;
  const int sweep = of_expert / (kSweep * cols), in = of_expert - sweep * kSweep * cols;
  lo += sweep * kSweep * kTile;
  const int row_tiles = min(kSweep, (hi - lo + kTile - 1) / kTile);
  const int col0 = in / (kWide * row_tiles) * kWide, wide = min(kWide, cols - col0), in_cols = in - col0 * row_tiles;
  const int deep = (row_tiles + (row_tiles + kDeep - 1) / kDeep - 1) / ((row_tiles + kDeep - 1) / kDeep);
  const int row0 = in_cols / (deep * wide) * deep, in_block = in_cols - row0 * wide;
  p->depth = min(deep, row_tiles - row0);
  p->deep = in_block % p->depth;
  p->col = col0 + in_block / p->depth;
  p->e = a.expert_offsets != nullptr ? a.expert_begin + at : 0;
  p->row = lo + (row0 + p->deep) * kTile + (half > 0 ? kHalfRows : 0);
  p->rows = min(half >= 0 ? kHalfRows : kTile, hi - p->row);
  p->slice = 0, p->step0 = 0, p->steps = a.k_bytes / kStep;
  return p->rows > 0;
}

// One matrix cut along K, a slice's tiles stand next to each other, the row tiles of a column first, and
// a die takes an eighth of the row: about one slice, whose x its L2 then reads once and whose weights no other die asks for.
__device__ __forceinline__ bool find_slice(const TileGemmArgs& a, Place* p) {
  const int row_tiles = (a.max_rows + kTile - 1) / kTile, tiles = row_tiles * (a.N / kTile), total = tiles * a.slices;
  const int block = blockIdx.x, die = block % kDies, first = total * die / kDies, count = total * (die + 1) / kDies - first, j = block / kDies;
  if (j >= count) return false;
  const int all = a.k_bytes / kStep, in = (first + j) % tiles;
  p->slice = (first + j) / tiles;
  p->step0 = all * p->slice / a.slices, p->steps = all * (p->slice + 1) / a.slices - p->step0;
  p->deep = in % row_tiles, p->depth = row_tiles, p->col = in / row_tiles;
  p->e = 0, p->row = p->deep * kTile, p->rows = min(kTile, a.max_rows - p->row);
  return true;
}

__device__ __forceinline__ int divided(const TileGemmArgs& a, int r) {
  return a.a_rows_div == 1 ? r : static_cast<int>(__umulhi(static_cast<uint32_t>(r), a.a_rows_inv));
}

// What a tile's sums are scaled with, brought along with the copies.
struct TileTables {
  float factor[kTile], x_scale[kTile], w_scale[kTile];
  uint16_t bias[kTile];
};

constexpr int kSums = -1;                        // in an activation's place: the sums themselves, a slice's into its slab
template <int Act> constexpr bool kGatedAct = Act != HYMETA_GEMM_ACT_NONE && Act != kSums;

template <int Act>
__device__ __forceinline__ float apply_act(const TileGemmArgs& a, float gate, float up) {
  const float g = bf16_round(gate), u = bf16_round(up);
  if constexpr (Act == HYMETA_GEMM_ACT_SILU) return g * sigmoidf(g) * u;
  else if constexpr (Act == HYMETA_GEMM_ACT_SILU_EXACT) return g * sigmoid_exact(g) * u;
  else return clamped_glu(g, u, a.act_limit, a.act_alpha);
}

// Rows of w in an image: 64 a wave; where an activation follows, a wave's 128 columns are 64 gate rows and their 64 up rows.
template <bool I8, int Act, int MI>
__device__ __forceinline__ void tile_body(const TileGemmArgs& a, const Place& p, char* sm) {
  typedef typename TileAcc<I8>::type acc_t;
  constexpr bool Gated = kGatedAct<Act>;
  constexpr int NJ = 8;                                      // a wave's products: 16 MI rows x 128 weight rows
  constexpr int kReads = MI + NJ, kProducts = MI * NJ;       // of half a step
  constexpr int XC = MI, kCopies = XC + 8;                   // a wave's copies of a step, 8 rows each of x and of w
  constexpr int kReadEvery = MI == 8 ? 4 : 2, kCopyEvery = MI == 8 ? 6 : 4;
  // a step's first kEarly copies are asked for in the second half of the step before the last, the others half a step later
  constexpr int kEarly = MI == 8 ? 10 : 8, kLast = kCopies - kEarly;
  static_assert(kReads * kReadEvery <= kProducts && kEarly * kCopyEvery <= kProducts && kLast * kCopyEvery <= kProducts, "reads and copies find their places");
  const TileTables& tables = *reinterpret_cast<const TileTables*>(sm + 4 * kImage);
  const uint32_t lds = __builtin_amdgcn_readfirstlane(lds_address(sm)), tables_at = lds + 4 * kImage, scrap = tables_at + sizeof(TileTables);

  const int tid = threadIdx.x, lane = tid & 63, c = lane >> 4, n = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int steps = p.steps;
  const char* const xb = a.x + static_cast<int64_t>(p.step0) * kStep;

  // A copy of a wave brings 8 rows x 128 bytes; a row's 16-byte chunks lie XOR-ed with (row / 2) % 8, which with the pitch of
  // 128 bytes spreads the sixteen rows of a fragment read over all banks.  Rows past the end re-read the last row.
  const int l3 = lane >> 3, swizzled = (lane & 7) ^ (l3 >> 1);
  const uint32_t wo[2] = {static_cast<uint32_t>(l3 * a.k_bytes + 16 * swizzled), static_cast<uint32_t>(l3 * a.k_bytes + 16 * (swizzled ^ 4))};
  auto slot_of = [&](int r) { return p.row + min(r, p.rows - 1); };
  auto source = [&](int r) { return a.a_rows != nullptr ? divided(a, a.a_rows[slot_of(r)]) : slot_of(r); };
  uint32_t xo[XC];
#pragma unroll
  for (int j = 0; j < XC; ++j)
    xo[j] = static_cast<uint32_t>(source(32 * j + 8 * wave + l3)) * static_cast<uint32_t>(a.x_stride) + 16 * (swizzled ^ (wave & 1 ? 4 : 0));
  const uint32_t touch_x = static_cast<uint32_t>(source(tid)) * static_cast<uint32_t>(a.x_stride), touch_w = static_cast<uint32_t>(lane) * a.k_bytes;
  const int64_t weight_row = Gated ? static_cast<int64_t>(wave & 1) * (a.N / 2) + p.col * (kTile / 2) + 64 * (wave >> 1) : p.col * kTile + 64 * wave;
  const char* const wb = a.w + static_cast<int64_t>(p.e) * a.w_stride_e + weight_row * a.k_bytes + static_cast<int64_t>(p.step0) * kStep;
  auto copy1 = [&](int step, int j, int image) {             // x and w by turns while both last
    if (j < 2 * XC && j % 2 == 0) {
      copy16(xb + step * kStep, xo[j / 2], lds + image + 1024 * (4 * (j / 2) + wave));
    } else {
      const int i = j < 2 * XC ? j / 2 : j - XC;
      copy16(wb + step * kStep + static_cast<int64_t>(8 * i) * a.k_bytes, wo[i & 1], lds + image + kImage + 1024 * (8 * wave + i));
    }
  };
  // the tables, a thread per row or column
  auto bring = [&](const void* base, uint32_t index, size_t table) { copy4(static_cast<const char*>(base), 4u * index, tables_at + static_cast<uint32_t>(table) + 256 * wave); };
  if (a.row_scale != nullptr) bring(a.row_scale, a.scale_rows != nullptr ? a.scale_rows[slot_of(tid)] : slot_of(tid), offsetof(TileTables, factor));
  if constexpr (I8) {
    bring(a.x_scale, source(tid), offsetof(TileTables, x_scale));
    bring(a.w_scale + static_cast<int64_t>(p.e) * a.N + weight_row, lane, offsetof(TileTables, w_scale));
  }
  if (!Gated && a.bias != nullptr && wave < 2) bring(a.bias, p.col * (kTile / 2) + tid, offsetof(TileTables, bias));

  int off[2];                                                // a fragment's place for this lane: row n, chunk 4 half + c
#pragma unroll
  for (int h = 0; h < 2; ++h) off[h] = n * kStep + 16 * ((4 * h + c) ^ ((n >> 1) & 7));
  const int xat = 16 * MI * wm * kStep, wat = kImage + 128 * wn * kStep;
  acc_t acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
  u32x4 xf[2][MI], wf[2][NJ];
  auto read1 = [&](int image, int h, int i) {                // in the order in which the products ask for them
    if (i == 0) wf[h][0] = ld16(sm + image + wat + off[h]);
    else if (i <= MI) xf[h][i - 1] = ld16(sm + image + xat + off[h] + 16 * (i - 1) * kStep);
    else wf[h][i - MI] = ld16(sm + image + wat + off[h] + 16 * (i - MI) * kStep);
  };

  int image = 0, other = 2 * kImage;                         // where this step's and the next one's images lie
#pragma unroll
  for (int j = 0; j < kCopies; ++j) copy1(0, j, image);
#pragma unroll
  for (int j = 0; j < kEarly; ++j) copy1(1, j, other);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kEarly) : "memory");
#pragma unroll
  for (int i = 0; i < kReads; ++i) read1(image, 0, i);
  int touch_x_at = p.col & (kWide - 1), touch_w_at = p.deep; // the next steps at which lines are this workgroup's to touch
  // (past the last step the copies repeat it into an image that nobody reads any more)
  for (int it = 0; it < steps; ++it) {
    const int coming = min(it + 1, steps - 1), fresh = min(it + 2, steps - 1), ahead = min(it + kAhead, steps - 1);
    each<2>([&](auto half) {
      constexpr int h = decltype(half)::value;
      if constexpr (h == 1) copies_landed_barrier();         // this step's fragments are in registers, the next step's rows in LDS
      each<kProducts>([&](auto number) {
        constexpr int k = decltype(number)::value;
        if constexpr (k % kReadEvery == 0 && k / kReadEvery < kReads) {
          read1(h == 1 ? other : image, h ^ 1, k / kReadEvery);
          __builtin_amdgcn_sched_barrier(0);
        }
        tile_mma<I8>(wf[h][k / MI], xf[h][k % MI], acc[k % MI][k / MI]);
        if constexpr (k % kCopyEvery == 1 && k / kCopyEvery < (h == 1 ? kEarly : kLast)) {
          __builtin_amdgcn_sched_barrier(0);
          copy1(h == 1 ? fresh : coming, (h == 1 ? 0 : kEarly) + k / kCopyEvery, h == 1 ? image : other);
        }
        if constexpr (h == 1 && k == kProducts / 4 + 1) {
          if (it == touch_x_at) copy4(xb + ahead * kStep, touch_x, scrap), touch_x_at += kWide;
        }
        if constexpr (h == 1 && k == kProducts / 2 + 1) {
          if (it == touch_w_at) copy4(wb + ahead * kStep, touch_w, scrap), touch_w_at += p.depth;
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      settle();
    });
    const int t = image;
    image = other, other = t;
  }
  copies_landed_barrier();

  if constexpr (Act == kSums) {
    acc_t* out = reinterpret_cast<acc_t*>(a.slabs) + ((static_cast<int64_t>(p.slice) * a.max_rows + p.row) * a.N + p.col * kTile + 128 * wn + 4 * c) / 4;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int row = 16 * (MI * wm + i) + n;
      if (row < p.rows) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) out[static_cast<int64_t>(row) * (a.N / 4) + 4 * j] = acc[i][j];
      }
    }
    return;
  }
  // acc[i][j][r] = C[row 16 (MI wm + i) + n][tile column 128 wn + 16 j + 4 c + r].  Scales on the sums, one rounding, an
  // activation over the rounded pairs; lanes trade with the next 16 so that each stores 16 bytes of a row.
  const bool scaled = a.row_scale != nullptr, biased = !Gated && a.bias != nullptr;
  constexpr int kOutCols = Gated ? 64 : 128;                 // of a wave
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int row = 16 * (MI * wm + i) + n;
    asm volatile("" ::: "memory");                           // (else the tables of all rows and columns are held, and spilled)
    const float factor = scaled ? tables.factor[row] : 1.f, xs = I8 ? tables.x_scale[row] : 1.f;
    uint16_t* out = a.out + static_cast<int64_t>(p.row + row) * a.out_stride + (2 * p.col + wn) * kOutCols + 16 * (c & 1) + 8 * (c >> 1);
    auto values = [&](int j) {
      f32x4 v, b = {0.f, 0.f, 0.f, 0.f};
      const int col = 128 * wn + 16 * j + 4 * c;
      if constexpr (!Gated) {
        const u32x2 raw = *reinterpret_cast<const u32x2*>(&tables.bias[col]), bits = biased ? raw : u32x2{0, 0};
        b = f32x4{lo_bf(bits[0]), hi_bf(bits[0]), lo_bf(bits[1]), hi_bf(bits[1])};
      }
      if constexpr (I8) {
        const f32x4 ws = *reinterpret_cast<const f32x4*>(&tables.w_scale[col]);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = w8a8_scaled(acc[i][j][r], xs, ws[r], b[r]) * factor;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (acc[i][j][r] + b[r]) * factor;
      }
      return v;
    };
    auto piece = [&](int j) {                                // 4 columns of the output
      f32x4 v = values(j);
      if constexpr (Gated) {
        const f32x4 up = values(j + 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = apply_act<Act>(a, v[r], up[r]);
      }
      return u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    };
#pragma unroll
    for (int j = 0; j < kOutCols / 16; j += 2) {
      __builtin_amdgcn_sched_barrier(0);
      const u32x2 even = piece(j), odd = piece(j + 1);
      const auto first = __builtin_amdgcn_permlane16_swap(even[0], odd[0], false, false);
      const auto second = __builtin_amdgcn_permlane16_swap(even[1], odd[1], false, false);
      if (row < p.rows) st16(out + 16 * j, u32x4{first[0], second[0], first[1], second[1]});
    }
  }
}

template <bool I8, int Act>
__global__ __launch_bounds__(256, 1) void tile_gemm_kernel(TileGemmArgs a) {
  __shared__ __attribute__((aligned(16))) char sm[4 * kImage + sizeof(TileTables) + 256];
  Place p;
  if (Act == kSums ? !find_slice(a, &p) : !find_place(a, threadIdx.x & 63, &p)) return;
  if (p.rows > kHalfRows) tile_body<I8, Act, 8>(a, p, sm);
  else tile_body<I8, Act, 4>(a, p, sm);
}

}  // namespace

bool tile_gemm_fits(const TileGemmArgs& a) {
  const int64_t source = a.a_rows != nullptr ? (a.max_rows + a.a_rows_div - 1) / a.a_rows_div : a.max_rows;
  const int64_t row_tiles = a.max_rows / kTile + 1 + kMaxTileExperts;
  constexpr int64_t kReach = int64_t{1} << 32;               // of a 32-bit offset
  return a.max_rows > 0 && a.k_bytes % kStep == 0 && a.k_bytes >= kMinSteps * kStep && a.N > 0 && a.N % kTile == 0 && (a.act == HYMETA_GEMM_ACT_NONE || a.bias == nullptr) && a.out_stride % 8 == 0 &&
         a.x_stride % 16 == 0 && a.w_stride_e % 16 == 0 && a.x_stride >= 0 && source * a.x_stride < kReach && int64_t{64} * a.k_bytes < kReach / 2 &&
         (a.a_rows == nullptr || (a.a_rows_div >= 1 && static_cast<int64_t>(a.max_rows) * a.a_rows_div < kReach / 2)) &&
         (a.expert_offsets == nullptr || a.expert_end - a.expert_begin <= kMaxTileExperts) && row_tiles * (a.N / kTile) < (int64_t{1} << 26);
}

// The partial sums go to memory and back: 9 slices of 512 x 3584 are 66 MB, 25 of 83 us.  Bf16 with weights from memory, the
// product and a residual norm that adds its slices, us against the library's product and the norm; in brackets with a launch that
// reduces them; weight rows x K and rows (slices, steps of a slice):
//   3584 x 18944: 300 rows 104 -> 70 (100 -> 69) (9, 32), 512 201 -> 86, 768 184 -> 103, 1024 194 -> 129, 1536 284 -> 172, 2048 374 -> 238 (2, 148)
//   3584 x 9472: 513 66 -> 59 (61 -> 56) (6, 24), 768 80 -> 65, 1025 89 -> 86 (82 -> 88) (3, 49), 1536 112 -> 99 (104 -> 96)
//   8192 x 28672: 300 227 -> 185 (214 -> 180) (4, 112), 512 320 -> 225; 5120 x 13824: 300 83 -> 72 (79 -> 69) (6, 36), 1024 154 -> 132
//   2048 x 11008: 1280 92 -> 68 (86 -> 66) (6, 28); 1024 x 16384: 2048 103 -> 76 (97 -> 73) (8, 32)
// Few tiles are cut whatever the matrix.  With more, the library fills the chip by itself on matrices that are not deep (2048 x 8192 at
// 1536 rows 62 -> 64, reduced 56 -> 62; 3072 x 8192 at 900 63 -> 64), that have few columns, whose sums the norm reads a short row at a time
// (512 x 9216 at 6000 73 -> 79), where the tiles' last rows or the slices leave units idle and a launch reduces them (the two of
// 1025 rows above; 1536 x 8960 at 2561 79 -> 82; kSliceSums floats of sums are 7 / 8 of the chip), in two slices that do not fill it or of
// narrow matrices (2048 x 16384 at 3072 185 -> 189, 4096 x 16384 at 1500 191 -> 193), and where the rows of wide ones lie whole 32 KB apart
// (8192 x 16384 at 330 rows 121 -> 138, 6144 x 16384 at 513 138 -> 140): those are left to it.  Weights that the last-level cache still holds
// favour the library by a tenth.  Tiles of 128 rows: 4 % to 14 % slower on 3584 x 18944, 7 % to 11 % faster on 3584 x 9472 up to 512 rows.
int tile_gemm_slices(const TileGemmArgs& a, bool reduced) {
  if (a.expert_offsets != nullptr || a.a_rows != nullptr || a.act != HYMETA_GEMM_ACT_NONE || !tile_gemm_fits(a)) return 1;
  const int64_t tiles = static_cast<int64_t>((a.max_rows + kTile - 1) / kTile) * (a.N / kTile), k = a.k_bytes / 2;
  const int slices = static_cast<int>(std::min<int64_t>(kDies * kUnits / tiles, kMaxSlices));
  if (slices < 2 || a.k_bytes / kStep / slices < kSliceSteps || k < 2 * static_cast<int64_t>(a.N)) return 1;
  if (tiles <= kFewSliceTiles) return slices;
  const bool deep = k >= 8704, filled = static_cast<int64_t>(a.max_rows) * a.N * slices >= kSliceSums;
  if (a.N < 1280 || !(deep || (!reduced && a.N >= 3584 && k >= 7168))) return 1;
  if (!filled && (a.N < 2048 || (reduced && k < 13824))) return 1;
  if (a.N >= 6144 && k % 16384 == 0) return 1;
  return slices > 2 || (tiles >= 100 && a.N >= 2560 && k >= 4 * static_cast<int64_t>(a.N)) ? slices : 1;
}

void tile_gemm_launch(const TileGemmArgs& args, bool int8, hipStream_t s) {
  TileGemmArgs a = args;
  if (a.slices > 1) {
    const int total = (a.max_rows + kTile - 1) / kTile * (a.N / kTile) * a.slices;
    const dim3 all((total + kDies - 1) / kDies * kDies);
    hipLaunchKernelGGL((tile_gemm_kernel<false, kSums>), all, dim3(256), 0, s, a);
    return;
  }
  if (a.a_rows != nullptr) a.a_rows_inv = a.a_rows_div > 1 ? static_cast<uint32_t>((uint64_t{1} << 32) / a.a_rows_div + 1) : 0;
  // the host knows the rows, not how the experts share them; and the halves of a last round
  const int64_t row_tiles = (a.max_rows + kTile - 1) / kTile + (a.expert_offsets != nullptr ? a.expert_end - a.expert_begin : 0);
  const dim3 grid(static_cast<unsigned>((row_tiles * (a.N / kTile) + kDies - 1) / kDies * kDies + kDies * kUnits / 2)), block(256);
#define HYMETA_TILE_LAUNCH(I8, ACT) hipLaunchKernelGGL((tile_gemm_kernel<I8, ACT>), grid, block, 0, s, a)
  if (a.act == HYMETA_GEMM_ACT_SILU) {
    if (int8) HYMETA_TILE_LAUNCH(true, HYMETA_GEMM_ACT_SILU);
    else HYMETA_TILE_LAUNCH(false, HYMETA_GEMM_ACT_SILU);
  } else if (a.act == HYMETA_GEMM_ACT_SILU_EXACT) {
    HYMETA_TILE_LAUNCH(false, HYMETA_GEMM_ACT_SILU_EXACT);
  } else if (a.act == HYMETA_GEMM_ACT_CLAMPED_GLU) {
    HYMETA_TILE_LAUNCH(false, HYMETA_GEMM_ACT_CLAMPED_GLU);
  } else {
    if (int8) HYMETA_TILE_LAUNCH(true, HYMETA_GEMM_ACT_NONE);
    else HYMETA_TILE_LAUNCH(false, HYMETA_GEMM_ACT_NONE);
  }
#undef HYMETA_TILE_LAUNCH
}

}  // namespace hymeta
