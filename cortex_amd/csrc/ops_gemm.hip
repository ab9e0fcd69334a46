// ops_gemm.hip -- gemm! of float matrices on the bfloat16 matrix cores, three pieces to a float (split_mfma.h).
//
// What bounds it.  A product of 128 x 128 x 32 is 24 matrix instructions for each of eight waves, 1536 cycles of a compute
// unit's matrix cores, and measured about 2800: the splitting (4.5 vector instructions a float, of which 64 products are
// made) takes 450 of the difference, waits for memory 250, reads of fragments and the barrier the rest.  Beyond that the
// clock gives way: at these rates it stands at 1.8 to 2.0 of 2.4 GHz, and more instructions a cycle lower it further
// (matrix instructions alone, on normal operands: 1770 of 2500 TFLOP/s, 295 in floats).
//
// Times of products, in us, the library's second: [1024, 4096] over 4096 k, b stored [n][k] 197 and 271, stored [k][n] 203
// and 261; [4096, 4096] over 1024, both stored [k][.] 214 and 274; 4096 cubed 725 and 1121; 2048 cubed 94 and 133;
// [64, 4096] over 4096 24 and 114; [128, 784] over 128 4.5 and 7.2; [128, 128] over 784 5.5 and 6.9.  Over 1350 products of
// layers of 1 to 4096 a side, whole calls one after the other: 1.62 times the library's speed in the geometric mean, 0.87 to
// 7 in 98 % of them, 0.58 at the least.  60 are below 0.95: sums of 50 to 200 k over half a million results and more
// ([878, 1290] over 66 9.2 and 6.3); of 400 to 1500 over 200 to 500 tiles of 32 x 32 ([851, 572] over 1451 27.7 and 16.1); a few
// results over 2700 k and more, where two launches cost what they gain ([2, 56] over 3909 15.1 and 12.8); and chains of blocks
// that just miss a round.  They are not handed back: the library's errors are two to seven times as large there.
// Errors against 64 bits, of the library's: 0.05 to 1.0, 0.30 in the median.
//
// Tiles and their choice: below, at expected_time.
#include <algorithm>
#include <optional>

#include "common.h"
#include "gemm.h"
#include "split_mfma.h"

using namespace cthip;

namespace {

// Element `chunk` (of eight k) of row `row` of a tile in LDS, rows of 32 k: the chunks of a row are permuted so that eight
// consecutive rows' reads of one chunk cover 128 bytes' worth of banks once.
__device__ __forceinline__ uint32_t tile_at(uint32_t row, uint32_t chunk) { return row * 32 + ((chunk ^ (row >> 1)) & 3) * 8; }

struct GemmArgs {
  const float* a;
  const float* b;
  float* c;              // the result, or partial[split][m][n]
  int64_t lda, ldb, ldc, c_split;
  uint32_t m, n, k, m_tiles, n_tiles, units;
  uint32_t tiles_per_group;   // of k; an even number
  float alpha, beta;
  FastDiv tiles_fd, group_fd;
};

// Consecutive units of work on one die: neighbouring tiles share operands in its L2.
__device__ __forceinline__ uint32_t unit_of_block(uint32_t b, uint32_t units) {
  const uint32_t per_die = (units + kXcds - 1) / kXcds;
  return (b % kXcds) * per_die + b / kXcds;
}

// The tiles of a product in groups of kGroup rows, column after column: what a die works on at a time is as square as it
// can be.
constexpr uint32_t kGroup = 8;

struct Place {
  uint32_t split, m_tile, n_tile;
};

__device__ __forceinline__ Place place_of(const GemmArgs& a, uint32_t unit) {
  Place p;
  uint32_t rest, tile, group;
  a.tiles_fd.divmod(unit, p.split, tile);
  a.group_fd.divmod(tile, group, rest);
  const uint32_t rows = min(kGroup, a.m_tiles - group * kGroup);
  p.n_tile = rest / rows;
  p.m_tile = group * kGroup + rest - p.n_tile * rows;
  return p;
}

// Eight consecutive k of one row of an operand: kRowMajor has them side by side, else a leading dimension apart.  `base` is
// uniform and stays in scalar registers, `offset` is the lane's, in bytes.
template <bool kRowMajor>
__device__ __forceinline__ void load8(const float* base, uint32_t offset, int64_t ld, f32x4 (&to)[2]) {
  uint64_t bits = reinterpret_cast<uint64_t>(base);
  asm("" : "+s"(bits));   // or the loop keeps a 64-bit address per lane and load, for which there are no registers
  typedef __attribute__((address_space(1))) const char* Global;
  typedef f32x4 f32x4_at_4 __attribute__((aligned(4)));
  const Global p = reinterpret_cast<Global>(bits);
  if constexpr (kRowMajor) {
    to[0] = *reinterpret_cast<__attribute__((address_space(1))) const f32x4_at_4*>(p + offset);
    to[1] = *reinterpret_cast<__attribute__((address_space(1))) const f32x4_at_4*>(p + 16 + offset);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      to[e / 4][e % 4] = *reinterpret_cast<__attribute__((address_space(1))) const float*>(p + 4 * e * ld + offset);
  }
}

// c = alpha * op(a) op(b) + beta * c over tiles of BM x BN, WM x WN waves to a group, KG groups to a block.  At least 32 k.
// kA: a is stored [m][k], else [k][m]; kB: b is stored [n][k], else [k][n].
// The floats are split once, on the way into LDS.  Groups take a run of k each and are added at the end: of results with
// fewer tiles than compute units, whose blocks have a unit to themselves and wait for memory, a pair is formed in 0.87 us
// for what takes one group 0.64 twice ([1024, 1024] over 1024 20.2 and 25.6 us); three groups gained nothing more.
// Tried and not taken: tiles of 256 x 128 (no registers left beside their sums; 871 us where these take 741), prefetching
// two tiles ahead (224 and 219 us), the order of instructions within a step left to the compiler (768 and 737).
template <int BM, int BN, int WM, int WN, int KG, bool kA, bool kB>
__global__ void __launch_bounds__(64 * WM * WN * KG, 2) gemm_kernel(const GemmArgs a) {
  constexpr int BK = 32, T = 64 * WM * WN, MT = BM / WM / 32, NT = BN / WN / 32, kChunks = BK / 8;
  constexpr int UA = BM * kChunks / T, UB = BN * kChunks / T, U = UA + UB;   // runs of eight k that a lane stages
  static_assert(UA * T == BM * kChunks && UB * T == BN * kChunks, "lanes share the tiles evenly");
  constexpr int kLeft = 2 * kSplitPieces * BM * BK, kRight = 2 * kSplitPieces * BN * BK;
  __shared__ __attribute__((aligned(16))) uint16_t all_lds[KG][kLeft + kRight];
  const uint32_t unit = unit_of_block(blockIdx.x, a.units);
  if (unit >= a.units) return;
  const Place place = place_of(a, unit);
  const uint32_t group = __builtin_amdgcn_readfirstlane(threadIdx.x / T), tid = threadIdx.x % T, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint16_t* lds = all_lds[group];
  const uint32_t tiles = a.tiles_per_group, first = (place.split * KG + group) * tiles;

  // Rows beyond the result repeat the last one and are not stored.
  auto row_of = [&](int i) { return (i < UA ? kA : kB) ? ((i < UA ? i : i - UA) * T + tid) / kChunks
                                                       : ((i < UA ? i : i - UA) * T + tid) % (i < UA ? BM : BN); };
  auto chunk_of = [&](int i) { return (i < UA ? kA : kB) ? ((i < UA ? i : i - UA) * T + tid) % kChunks
                                                         : ((i < UA ? i : i - UA) * T + tid) / (i < UA ? BM : BN); };
  const float* base_a = a.a + (int64_t)(place.m_tile * BM) * (kA ? a.lda : 1);
  const float* base_b = a.b + (int64_t)(place.n_tile * BN) * (kB ? a.ldb : 1);
  uint32_t offset[U];
#pragma unroll
  for (int i = 0; i < U; ++i) {
    const uint32_t last = i < UA ? a.m - 1 - place.m_tile * BM : a.n - 1 - place.n_tile * BN, r = min(row_of(i), last);
    const uint32_t ld = (uint32_t)(i < UA ? a.lda : a.ldb);
    offset[i] = 4 * ((i < UA ? kA : kB) ? r * ld + chunk_of(i) * 8 : chunk_of(i) * 8 * ld + r);
  }
  // The last tile of k, if it is a partial one, is loaded from 32 k before the end on; what an earlier tile had is set to
  // zero, in both operands, before it is used.  Tiles beyond it are all zeros.
  auto load = [&](int i, uint32_t tile, f32x4 (&to)[2]) {
    const int64_t k0 = min((first + tile) * BK, a.k - BK);
    if (i < UA) load8<kA>(base_a + (kA ? k0 : k0 * a.lda), offset[i], a.lda, to);
    else load8<kB>(base_b + (kB ? k0 : k0 * a.ldb), offset[i], a.ldb, to);
  };
  auto drop_repeated = [&](int i, uint32_t tile, f32x4 (&r)[2]) {
    const uint32_t k0 = (first + tile) * BK;
    if (k0 + BK <= a.k) return;
    asm volatile("");   // stays a branch: as selects it would cost every tile
    const uint32_t repeated = k0 - (a.k - BK);   // of the tile's k; all of them beyond the last tile
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e / 4][e % 4] = chunk_of(i) * 8 + e < repeated ? 0.f : r[e / 4][e % 4];
  };

  f32x16 sums[2][MT][NT];   // the products of the leading pieces; all others
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < NT; ++u) sums[s][t][u] = zero16();
  const uint32_t wave_m = wave / WN * (MT * 32), wave_n = wave % WN * (NT * 32), row = lane & 31, half = lane >> 5;

  {
    const SplitWeights weights;
    f32x4 raw[U][2];
    u32x4 pieces[kSplitPieces];
    auto piece_of = [&](int i, int buffer, int p) {
      return i < UA ? &lds[(buffer * kSplitPieces + p) * BM * BK] : &lds[kLeft + (buffer * kSplitPieces + p) * BN * BK];
    };
    // half h of run i: the pieces go to LDS with the second one
    auto stage = [&](int i, int h, int buffer, uint32_t tile) {
      if (h == 0) drop_repeated(i, tile, raw[i]);
      split4(raw[i][h], pieces, 4 * h, weights);
      if (h == 0) return;
#pragma unroll
      for (int p = 0; p < kSplitPieces; ++p)
        *reinterpret_cast<u32x4*>(piece_of(i, buffer, p) + tile_at(row_of(i), chunk_of(i))) = pieces[p];
    };
    bf16x8 left[2][MT][kSplitPieces], right[2][NT][kSplitPieces];
    // piece p of an operand, k 16 * part .. + 15 of the tile
    auto fetch_left = [&](int buffer, int part, int p) {
#pragma unroll
      for (int t = 0; t < MT; ++t)
        left[part][t][p] = *reinterpret_cast<const bf16x8*>(piece_of(0, buffer, p) + tile_at(wave_m + t * 32 + row, part * 2 + half));
    };
    auto fetch_right = [&](int buffer, int part, int p) {
#pragma unroll
      for (int u = 0; u < NT; ++u)
        right[part][u][p] = *reinterpret_cast<const bf16x8*>(piece_of(UA, buffer, p) + tile_at(wave_n + u * 32 + row, part * 2 + half));
    };
    auto multiply = [&](int part, int i) {
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) {
          f32x16& to = sums[i + 1 < kSplitProducts][t][u];
          to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(left[part][t][kSplitLeft[i]], right[part][u][kSplitRight[i]], to, 0, 0, 0);
        }
    };
    // After product i of a half: pieces of the next half, those that its first product needs early, the others as the
    // present half's last use frees their registers.
    auto fetch_next = [&](int i, int buffer, int part) {
      if (i == 0) {
        fetch_left(buffer, part, 0);
        fetch_right(buffer, part, 0);
        fetch_right(buffer, part, 2);
      }
      if (i == 1) fetch_left(buffer, part, 2);
      if (i == 3) fetch_right(buffer, part, 1);
      if (i == 4) fetch_left(buffer, part, 1);
    };
    // One tile of k.  Its first half's fragments are in registers when it begins.  The products of that half run beside
    // the splitting of the next tile into the other buffer, those of the second beside the reads of the next tile's first
    // fragments: one barrier a tile, and no product waits for a read that was just issued.
    auto step = [&](uint32_t tile, int buffer) {
#pragma unroll
      for (int i = 0; i < kSplitProducts; ++i) {
        multiply(0, i);
        fetch_next(i, buffer, 1);
#pragma unroll
        for (int j = i * 2 * U / kSplitProducts; j < (i + 1) * 2 * U / kSplitProducts; ++j) {
          stage(j / 2, j % 2, buffer ^ 1, tile + 1);
          if (j % 2) load(j / 2, tile + 2, raw[j / 2]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < kSplitProducts; ++i) {
        multiply(1, i);
        fetch_next(i, buffer ^ 1, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
#pragma unroll
    for (int i = 0; i < U; ++i) load(i, 0, raw[i]);
#pragma unroll
    for (int j = 0; j < 2 * U; ++j) stage(j / 2, j % 2, 0, 0);
#pragma unroll
    for (int i = 0; i < U; ++i) load(i, 1, raw[i]);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kSplitProducts; ++i) fetch_next(i, 0, 0);
    for (uint32_t tile = 0; tile < tiles; tile += 2) {
      step(tile, 0);
      step(tile + 1, 1);
    }
  }

  bool found = false;
  float result[MT][NT][16];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float sum = sums[0][t][u][r] + sums[1][t][u][r];
        found |= not_finite(sum);
        result[t][u][r] = sum * kSplitUnscale;
      }
  if (__syncthreads_or(found)) {
    // In float: chains of a tile's 32 products, added up.
    constexpr int LD = BK + 4;
    float* left = reinterpret_cast<float*>(lds);
    float* right = left + BM * LD;
    static_assert((BM + BN) * LD * 4 <= (kLeft + kRight) * 2, "the floats fit where their pieces were");
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) result[t][u][r] = 0.f;
    for (uint32_t tile = 0; tile < tiles; ++tile) {
#pragma unroll
      for (int i = 0; i < U; ++i) {
        f32x4 raw[2];
        load(i, tile, raw);
        drop_repeated(i, tile, raw);
        float* to = (i < UA ? left : right) + row_of(i) * LD + chunk_of(i) * 8;
        *reinterpret_cast<f32x4*>(to) = raw[0];
        *reinterpret_cast<f32x4*>(to + 4) = raw[1];
      }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u) {
          f32x16 sum = zero16();
          for (int k = 0; k < BK; k += 8) {
            const f32x4 l = *reinterpret_cast<const f32x4*>(left + (wave_m + t * 32 + row) * LD + k + 4 * half);
            const f32x4 r = *reinterpret_cast<const f32x4*>(right + (wave_n + u * 32 + row) * LD + k + 4 * half);
#pragma unroll
            for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(l[e], r[e], sum, 0, 0, 0);
          }
#pragma unroll
          for (int r = 0; r < 16; ++r) result[t][u][r] += sum[r];
        }
      __syncthreads();
    }
  }

  if constexpr (KG > 1) {   // the groups' sums, added in their order
    constexpr int kCells = MT * NT * 16;
    static_assert(T * kCells * 4 <= (kLeft + kRight) * 2, "a group's sums fit its LDS");
    __syncthreads();
    if (group > 0) {
      float* to = reinterpret_cast<float*>(lds) + tid;
#pragma unroll
      for (int e = 0; e < kCells; ++e) to[e * T] = result[e / (NT * 16)][e / 16 % NT][e % 16];
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int g = 1; g < KG; ++g)
#pragma unroll
      for (int e = 0; e < kCells; ++e)
        result[e / (NT * 16)][e / 16 % NT][e % 16] += reinterpret_cast<const float*>(all_lds[g])[e * T + tid];
  }

  float* c = a.c + (int64_t)place.split * a.c_split;
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    const uint32_t n = place.n_tile * BN + wave_n + u * 32 + row;
    if (n >= a.n) continue;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t m = place.m_tile * BM + wave_m + t * 32 + 8 * (r / 4) + 4 * half + r % 4;
        if (m >= a.m) continue;
        float& cell = c[(int64_t)m * a.ldc + n];
        const float value = a.alpha * result[t][u][r];
        cell = a.beta == 0.f ? value : value + a.beta * cell;
      }
  }
}

template <bool kRowMajor>
__device__ __forceinline__ void load8_at(const float* p, int64_t ld, f32x4 (&to)[2]) {
  if constexpr (kRowMajor) {
    __builtin_memcpy(&to[0], p, 16);
    __builtin_memcpy(&to[1], p + 4, 16);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) to[e / 4][e % 4] = p[e * ld];
  }
}

// The same for results too small to fill the chip with tiles, in one launch: a block owns S x S, its W waves take every W-th
// run of 32 k each, straight from memory into the fragments, and their sums are added in LDS in their order.  In tiles of
// 16 x 16 the sums of four runs are added up there too: through 3000 k and more the error was up to 1.3 times that of shorter
// sums.  (In tiles of 32 x 32 it cost up to a fifth of the time; those have sixteen waves where a wave would take more.)
constexpr uint32_t kRunsToASum = 4;

template <int S>
struct SmallTile;
template <>
struct SmallTile<32> {
  static constexpr int kParts = 2;   // products to a run of 32 k
  using Cells = f32x16;
  static __device__ __forceinline__ Cells product(bf16x8 l, bf16x8 r, Cells sum) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(l, r, sum, 0, 0, 0);
  }
  static __device__ __forceinline__ Cells product_in_float(float l, float r, Cells sum) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(l, r, sum, 0, 0, 0);
  }
};
template <>
struct SmallTile<16> {
  static constexpr int kParts = 1;
  using Cells = f32x4;
  static __device__ __forceinline__ Cells product(bf16x8 l, bf16x8 r, Cells sum) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(l, r, sum, 0, 0, 0);
  }
  static __device__ __forceinline__ Cells product_in_float(float l, float r, Cells sum) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(l, r, sum, 0, 0, 0);
  }
};

template <int S, int W, bool kA, bool kB>
__global__ void __launch_bounds__(64 * W, 4) gemm_small_kernel(const GemmArgs a) {
  using Tile = SmallTile<S>;
  using Cells = typename Tile::Cells;
  constexpr int BK = 32, kParts = Tile::kParts, kCells = S * S / 64, E = kParts * 8;   // floats of a run to a lane
  __shared__ float partial[W][S * S];
  const uint32_t unit = unit_of_block(blockIdx.x, a.units);
  if (unit >= a.units) return;
  const Place place = place_of(a, unit);
  const uint32_t lane = threadIdx.x & 63, row = lane % S, group = lane / S;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t k_first = place.split * a.tiles_per_group * BK, k_end = min(a.k, k_first + a.tiles_per_group * BK);
  const uint32_t m = min(place.m_tile * S + row, a.m - 1), n = min(place.n_tile * S + row, a.n - 1);
  const float* left = a.a + (kA ? (int64_t)m * a.lda : m);
  const float* right = a.b + (kB ? (int64_t)n * a.ldb : n);
  // a lane's k of a run: 8 * group + 0 .. 7 and, in two parts, 16 more
  auto load = [&](uint32_t k0, f32x4 (&l)[E / 4], f32x4 (&r)[E / 4]) {
    if (k0 + BK <= k_end) {
#pragma unroll
      for (uint32_t part = 0; part < kParts; ++part) {
        const int64_t k = k0 + part * 16 + group * 8;
        load8_at<kA>(left + (kA ? k : k * a.lda), a.lda, reinterpret_cast<f32x4(&)[2]>(l[part * 2]));
        load8_at<kB>(right + (kB ? k : k * a.ldb), a.ldb, reinterpret_cast<f32x4(&)[2]>(r[part * 2]));
      }
    } else {
#pragma unroll
      for (uint32_t e = 0; e < E; ++e) {
        const uint32_t at = k0 + e / 8 * 16 + group * 8 + e % 8;
        const int64_t k = min(at, k_end - 1);
        const float x = left[kA ? k : k * a.lda], y = right[kB ? k : k * a.ldb];
        l[e / 4][e % 4] = at < k_end ? x : 0.f;
        r[e / 4][e % 4] = at < k_end ? y : 0.f;
      }
    }
  };
  Cells sums[2] = {};   // the products of the leading pieces; all others
  const SplitWeights weights;
  f32x4 l[E / 4], r[E / 4], l_next[E / 4], r_next[E / 4];
  const uint32_t k_mine = k_first + wave * BK;
  bool found = a.k == 1;   // a product by itself: the floats' is rounded once, and what the pieces leave out is not made up for
  auto add_up = [&](bool first) {
#pragma unroll
    for (int e = 0; e < kCells; ++e) {
      const float sum = sums[0][e] + sums[1][e];
      found |= not_finite(sum);
      float& cell = partial[wave][e * 64 + lane];
      cell = first ? sum * kSplitUnscale : cell + sum * kSplitUnscale;
    }
  };
  if (k_mine < k_end) load(k_mine, l, r);
  uint32_t run = 0;
  for (uint32_t k0 = k_mine; k0 < k_end; k0 += W * BK, ++run) {
    const uint32_t next = k0 + W * BK;
    if (next < k_end) load(next, l_next, r_next);
#pragma unroll
    for (int part = 0; part < kParts; ++part) {
      u32x4 lp[kSplitPieces], rp[kSplitPieces];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        split4(l[part * 2 + h], lp, 4 * h, weights);
        split4(r[part * 2 + h], rp, 4 * h, weights);
      }
#pragma unroll
      for (int i = 0; i < kSplitProducts; ++i) {
        Cells& to = sums[i + 1 < kSplitProducts];
        to = Tile::product(__builtin_bit_cast(bf16x8, lp[kSplitLeft[i]]), __builtin_bit_cast(bf16x8, rp[kSplitRight[i]]), to);
      }
    }
    if constexpr (S == 16) {
      if (run % kRunsToASum == kRunsToASum - 1) {   // behind the loads of the next run
        add_up(run < kRunsToASum);
        sums[0] = sums[1] = Cells{};
      }
    }
#pragma unroll
    for (int e = 0; e < E / 4; ++e) {
      l[e] = l_next[e];
      r[e] = r_next[e];
    }
  }
  if (S == 32 || run % kRunsToASum > 0 || run == 0) add_up(S == 32 || run < kRunsToASum);
  if (__syncthreads_or(found)) {
    Cells total = {};
    for (uint32_t k0 = k_mine; k0 < k_end; k0 += W * BK) {
      load(k0, l, r);
      Cells sum = {};
#pragma unroll
      for (int e = 0; e < E; ++e) sum = Tile::product_in_float(l[e / 4][e % 4], r[e / 4][e % 4], sum);
      total += sum;
    }
#pragma unroll
    for (int e = 0; e < kCells; ++e) partial[wave][e * 64 + lane] = total[e];
    __syncthreads();
  }
  float* c = a.c + (int64_t)place.split * a.c_split;
#pragma unroll
  for (uint32_t i = threadIdx.x; i < S * S; i += 64 * W) {
    const uint32_t e = i / 64, at_lane = i % 64;
    const uint32_t cm = place.m_tile * S + 8 * (e / 4) + 4 * (at_lane / S) + e % 4, cn = place.n_tile * S + at_lane % S;
    float sum = partial[0][i];
#pragma unroll
    for (int w = 1; w < W; ++w) sum += partial[w][i];
    if (cm >= a.m || cn >= a.n) continue;
    float& cell = c[(int64_t)cm * a.ldc + cn];
    const float value = a.alpha * sum;
    cell = a.beta == 0.f ? value : value + a.beta * cell;
  }
}

// c = alpha * (sum over the splits of partial[split]) + beta * c, in double.
__global__ void __launch_bounds__(256) gemm_sum_kernel(const float* partial, float* c, uint32_t n, int64_t ldc, uint32_t cells,
                                                       uint32_t splits, float alpha, float beta, FastDiv n_fd) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= cells) return;
  double sum = partial[i];
  for (uint32_t s = 1; s < splits; ++s) sum += (double)partial[(int64_t)s * cells + i];
  uint32_t row, col;
  n_fd.divmod(i, row, col);
  float& cell = c[(int64_t)row * ldc + col];
  cell = (float)(beta == 0.f ? alpha * sum : alpha * sum + (double)(beta * cell));
}

enum Tile { kFine, kSmallHalf, kSmall, kMedium, kMediumPair, kLarge };
struct TileShape {
  int rows, columns, groups, group_threads;
};
constexpr TileShape kTiles[] = {{16, 16, 1, 64 * 8}, {32, 32, 1, 64 * 8}, {32, 32, 1, 64 * 16}, {64, 64, 1, 256}, {64, 64, 2, 256},
                                {128, 128, 1, 512}};
constexpr bool is_small(Tile tile) { return tile < kMedium; }

template <bool kA, bool kB>
void launch(hipStream_t s, const GemmArgs& a, Tile tile) {
  const dim3 grid((a.units + kXcds - 1) / kXcds * kXcds), block(kTiles[tile].groups * kTiles[tile].group_threads);
  switch (tile) {
    case kFine: hipLaunchKernelGGL((gemm_small_kernel<16, 8, kA, kB>), grid, block, 0, s, a); break;
    case kSmallHalf: hipLaunchKernelGGL((gemm_small_kernel<32, 8, kA, kB>), grid, block, 0, s, a); break;
    case kSmall: hipLaunchKernelGGL((gemm_small_kernel<32, 16, kA, kB>), grid, block, 0, s, a); break;
    case kMedium: hipLaunchKernelGGL((gemm_kernel<64, 64, 2, 2, 1, kA, kB>), grid, block, 0, s, a); break;
    case kMediumPair: hipLaunchKernelGGL((gemm_kernel<64, 64, 2, 2, 2, kA, kB>), grid, block, 0, s, a); break;
    case kLarge: hipLaunchKernelGGL((gemm_kernel<128, 128, 2, 4, 1, kA, kB>), grid, block, 0, s, a); break;
  }
}

// How a product is formed: the tile, and into how many runs k is cut, whose products a second launch adds.
struct Plan {
  Tile tile;
  int64_t splits;
  int64_t tiles_per_group;   // of k
};

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

Plan plan_of(Tile tile, int64_t splits, int64_t k) {
  const TileShape& t = kTiles[tile];
  const int64_t k_tiles = ceil_div(k, 32), unit = is_small(tile) ? 1 : 2 * t.groups;   // a group's tiles come in pairs
  const int64_t per_split = ceil_div(ceil_div(k_tiles, splits), unit) * unit;
  return {tile, ceil_div(k_tiles, per_split), per_split / t.groups};
}

constexpr int64_t kUnits = 256;

// The launch of a sum, and its bytes at 3.3 TB/s.
double sum_time(const Plan& p, int64_t m, int64_t n) {
  return p.splits > 1 ? 2.5 + 1.2e-6 * (double)((p.splits + 1) * m * n) : 0.0;
}

// What a plan is expected to take, in microseconds: lines through the times of 420 products of 1 to 4096 a side in all
// four layouts, 95 % of which lie within 0.8 to 1.2 of them.  A unit holds one block (three of kMedium, whose steps then
// take longer); blocks beyond the chip's units wait for a round of their own.
// The line of the small kernel is that of a block of sixteen waves to 32 x 32, which was timed with the others.  The plans
// that run in its place are faster (best_small_plan); the lines to the other kernels lie where that one left them.
double expected_time(const Plan& p, int64_t m, int64_t n) {
  const TileShape& t = kTiles[p.tile];
  const int64_t blocks = ceil_div(m, t.rows) * ceil_div(n, t.columns) * p.splits;
  double us;
  if (p.tile == kMedium) {
    const int64_t full = blocks / (3 * kUnits), rest = blocks - full * 3 * kUnits, shared = full * 3 + ceil_div(rest, kUnits);
    us = 3.3 + 1.3 * (double)shared + (double)p.tiles_per_group * (0.31 * (double)(full + (rest > 0)) + 0.33 * (double)shared);
  } else {
    const double rounds = (double)ceil_div(blocks, kUnits);
    if (p.tile == kSmall) us = 2.0 + rounds * 3.0 * (double)ceil_div(p.tiles_per_group, 16);
    else if (p.tile == kMediumPair) us = 1.2 + rounds * (3.9 + 0.87 * (double)p.tiles_per_group);
    else us = 1.8 + rounds * (3.7 + 1.19 * (double)p.tiles_per_group);
  }
  constexpr double kHostOfALaunch = 2.0;
  return us + sum_time(p, m, n) + (p.splits > 1 ? kHostOfALaunch : 0.0);
}

struct Candidate {
  Tile tile;
  int64_t splits;
};

bool may_be(const Plan& p, const Candidate& c, int64_t m, int64_t n, bool may_split) {
  if (p.splits != c.splits) return false;
  return p.splits == 1 || (may_split && p.splits * m * n * (int64_t)sizeof(float) <= (int64_t)kMostProductScratch);
}

// The tile of the small kernel, its waves and its splits.  The splitting bounds it (4.5 vector instructions a float): a tile
// of 16 x 16 splits half the floats that one of 32 x 32 does, for a quarter of the products, and four times the units share the
// work.  Eight waves to a tile leave room for two and more to a unit.  Blocks that share a unit add their times, long runs of
// 16 x 16 a little more.  Lines through 8000 times of 2200 products, 96 % of which lie within 0.82 to 1.15 of them.  Us, 16 x 16,
// 32 x 32 under eight waves and under sixteen (which was all there was): [3, 8] over 1505 6.2, 10.3, 9.8; [1417, 11] over 3308
// 11.5, 21.4, 19.9; [178, 478] over 1316 10.9, 12.0, 11.6; [2940, 308] over 93 11.4, 8.5, 13.2; [2538, 17] over 3033, with a
// second launch for the sum of two halves, 14.2 in place of 22.4.
Plan best_small_plan(int64_t m, int64_t n, int64_t k, bool may_split) {
  constexpr Candidate kCandidates[] = {{kFine, 1}, {kSmallHalf, 1}, {kSmall, 1}, {kSmall, 2}};
  constexpr double kShortRuns = 5.0;
  Plan best = plan_of(kSmall, 1, k);
  double best_us = -1.0;
  for (const Candidate& c : kCandidates) {
    const Plan p = plan_of(c.tile, c.splits, k);
    const TileShape& t = kTiles[p.tile];
    const double runs = (double)p.tiles_per_group / (t.group_threads / 64);
    if (!may_be(p, c, m, n, may_split) || (p.tile == kSmallHalf && runs > kRunsToASum)) continue;
    const double shared = (double)ceil_div(ceil_div(m, t.rows) * ceil_div(n, t.columns) * p.splits, kUnits);
    double us = sum_time(p, m, n);
    if (p.tile == kSmall) us += 1.3 + shared * (2.5 + 2.3 * runs);
    else if (p.tile == kSmallHalf) us += 2.7 + shared * (1.06 + 1.24 * runs);
    else us += 2.7 + shared * (0.41 + 0.57 * runs + (shared > 1.0 ? 0.3 * std::max(0.0, runs - kShortRuns) : 0.0));
    if (best_us < 0.0 || us < best_us) {
      best = p;
      best_us = us;
    }
  }
  return best;
}

Plan best_plan(int64_t m, int64_t n, int64_t k, bool may_split) {
  constexpr Candidate kCandidates[] = {{kSmall, 1}, {kSmall, 2}, {kMedium, 1}, {kMediumPair, 1}, {kMediumPair, 2},
                                       {kMediumPair, 4}, {kMediumPair, 8}, {kLarge, 1}, {kLarge, 2}, {kLarge, 4}};
  Plan best = plan_of(kSmall, 1, k);
  double best_us = -1.0;
  for (const Candidate& c : kCandidates) {
    const Plan p = plan_of(c.tile, c.splits, k);
    if (!may_be(p, c, m, n, may_split) || (!is_small(p.tile) && k < 32)) continue;
    const double us = expected_time(p, m, n);
    if (best_us < 0.0 || us < best_us) {
      best = p;
      best_us = us;
    }
  }
  return is_small(best.tile) ? best_small_plan(m, n, k, may_split) : best;
}

bool overlap(const float* a, int64_t a_count, const float* b, int64_t b_count) {
  const uintptr_t a0 = reinterpret_cast<uintptr_t>(a), b0 = reinterpret_cast<uintptr_t>(b);
  return a0 < b0 + (uintptr_t)b_count * sizeof(float) && b0 < a0 + (uintptr_t)a_count * sizeof(float);
}

int64_t stored(int64_t rows, int64_t cols, int64_t ld) { return (rows - 1) * ld + cols; }

}  // namespace

namespace cthip {

// Not taken: fewer than 32 k over more tiles than one round of the small kernel (the tiles of the others have 32;
// [1846, 1794] over 23 k 35 us here, 9 there), and what 32-bit indexes do not hold.
bool gemm_split_takes(const GemmProduct& p) {
  constexpr int64_t kMostLd = int64_t(1) << 22, kMostTiles = int64_t(1) << 21, kMostCells = (int64_t(1) << 31) - 1;
  // a single row of tiles has two of 16 x 16 to each; where there are more rows and so many tiles, 32 x 32 is taken
  static_assert(kMostTiles * 2 * 64 * 8 < int64_t(1) << 32, "a launch of 2^32 lanes or more is refused");
  if (p.m < 1 || p.n < 1 || p.k < 1 || p.alpha == 0.f) return false;
  if (p.lda > kMostLd || p.ldb > kMostLd || p.m * p.n > kMostCells) return false;
  const int64_t small_tiles = ceil_div(p.m, 32) * ceil_div(p.n, 32);
  if (small_tiles > kMostTiles || (p.k < 32 && small_tiles > 256)) return false;
  const int64_t in_c = stored(p.m, p.n, p.ldc);
  return !overlap(p.c, in_c, p.a, p.row_major_a ? stored(p.m, p.k, p.lda) : stored(p.k, p.m, p.lda)) &&
         !overlap(p.c, in_c, p.b, p.row_major_b ? stored(p.n, p.k, p.ldb) : stored(p.k, p.n, p.ldb));
}

int gemm_split(hipStream_t s, const GemmProduct& p) {
  Plan plan = best_plan(p.m, p.n, p.k, true);
  std::optional<ProductScratch> scratch;   // until both launches are made
  float* partial = nullptr;
  if (plan.splits > 1) {
    // no room, or none to be had while the stream is being captured: one launch
    scratch.emplace(s, (size_t)(plan.splits * p.m * p.n) * sizeof(float));
    partial = static_cast<float*>(scratch->get());
    if (!partial) plan = best_plan(p.m, p.n, p.k, false);
  }
  GemmArgs a{};
  a.a = p.a; a.b = p.b; a.c = p.c;
  a.lda = p.lda; a.ldb = p.ldb; a.ldc = p.ldc;
  a.m = (uint32_t)p.m; a.n = (uint32_t)p.n; a.k = (uint32_t)p.k;
  a.alpha = p.alpha; a.beta = p.beta;
  a.m_tiles = (uint32_t)ceil_div(p.m, kTiles[plan.tile].rows);
  a.n_tiles = (uint32_t)ceil_div(p.n, kTiles[plan.tile].columns);
  a.tiles_per_group = (uint32_t)plan.tiles_per_group;
  a.tiles_fd = FastDiv(a.m_tiles * a.n_tiles);
  a.group_fd = FastDiv(kGroup * a.n_tiles);
  a.units = (uint32_t)(a.m_tiles * a.n_tiles * plan.splits);
  if (partial) {
    a.c = partial;
    a.ldc = p.n;
    a.c_split = p.m * p.n;
    a.alpha = 1.f;
    a.beta = 0.f;
  }
  if (p.row_major_a && p.row_major_b) launch<true, true>(s, a, plan.tile);
  else if (p.row_major_a) launch<true, false>(s, a, plan.tile);
  else if (p.row_major_b) launch<false, true>(s, a, plan.tile);
  else launch<false, false>(s, a, plan.tile);
  if (partial) {
    const uint32_t cells = (uint32_t)(p.m * p.n);
    hipLaunchKernelGGL(gemm_sum_kernel, dim3((cells + 255) / 256), dim3(256), 0, s, partial, p.c, (uint32_t)p.n, p.ldc, cells,
                       (uint32_t)plan.splits, p.alpha, p.beta, FastDiv((uint32_t)p.n));
  }
  static const char* const kNames[] = {"gemm_small", "gemm_small", "gemm_small", "gemm_medium", "gemm_medium_pair", "gemm_large"};
  static const char* const kSplitNames[] = {"gemm_small+gemm_sum",  "gemm_small+gemm_sum",       "gemm_small+gemm_sum",
                                            "gemm_medium+gemm_sum", "gemm_medium_pair+gemm_sum", "gemm_large+gemm_sum"};
  note_kernel(partial ? kSplitNames[plan.tile] : kNames[plan.tile]);
  return after_launch(s);
}

}  // namespace cthip
