// ops_conv_mfma.hip -- the three float products of a convolution on the matrix cores: two families of kernels, one on
// v_mfma_f32_16x16x4 (157 TFLOP/s dense), one on the bfloat16 matrix cores with three exact pieces to a float
// (split_mfma.h), and the rules between them.
//
// What bounds them.  For 64 images of 64 x 56 x 56 under 64 windows of 3 x 3 a product is
// 14.8 GFLOP (94 us of float matrix cores, 50 of the six bfloat16 products) around an unrolled matrix of 462 MB (75 us of
// HBM), so a product and the movement of that matrix have to overlap; the library's batched products
// ran at 62 to 94 TFLOP/s with the unrolling as a pass of its own before them.  One method called over and over, us, with the
// library's products, with the float kernels and with the split ones: forward 264, 235, 193; weight
// gradient 220, 178, 150 (its sum over the splits, 5, included); input gradient with the roll back 340, 316, 234;
// [128, 16, 28, 28] under 32 windows 33, 28, 25; 67, 31, 31 (a float kernel); 36, 36, 35.  Other shapes go
// either way, and the rules of ops_conv.hip (library or not; drawn through the float kernels' times) and below (which
// family) draw the lines.
//   float: what is left is latency: 3.3 to 3.8 waves a SIMD are resident, and the matrix cores of a compute unit are busy
//     for 51 (forward), 60 (weight gradient) and 54 % (input gradient) of the time that it is.
//   split: forward and input gradient wait for their loads of single floats behind the stores of the workspace (forward 207
//     us; without its stores 159, without its loads 140, without its products 185); the weight gradient splits (27 vector
//     instructions for a matrix instruction of two waves) as long as it multiplies.
//
// Tiles of the float kernels.  A block of four waves owns BM x BN of the result.  Both operands lie in LDS as
// [row][k], k innermost, rows padded by four floats: a lane takes four consecutive k in one
// 16-byte read for four MFMAs (lanes 0..15 hold k 0..3 of a group of sixteen, lanes 16..31
// k 4..7 and so on; which k an MFMA sums is free as long as both operands agree), and the
// sixteen rows cover the 64 banks once.  LDS is double buffered, the next tile's global loads
// are issued before the MFMAs of the current one.
//
// Loads are issued without a branch around them, from addresses clamped into the operand, and
// what lies beyond it is set to zero on the way into LDS, in the last tile only: with guarded
// loads every tile waited for memory twice (at the branches' joins) before its MFMAs.
//
// Rounding.  The float matrix cores round after every product, so the error of a sum grows with the length
// of the chain.  Products are summed in chains of eight (input gradient over more than 48 channels:
// sixteen, eight in the last tile; weight gradient: sixteen, then in double), and these are added up.
// The additions are vector instructions that run while the next products do: chains of 128 took the
// same time.  Error against 64 bits, in units of the library's, geometric means and ranges over 280
// shapes: outputs 0.87 (0.40 to 1.10), input gradients 0.80 (0.33 to 1.04), weight gradients 0.45
// (0.07 to 1.08); those above 1.04 at errors of 3e-8 to 7e-8.  Chains of 128: up to 1.5, 1.3 and 1.6.
// The bfloat16 matrix cores round once for eight products.  Forward sums end with a tile of 32 k, input gradients over up to
// 64 channels run through, over more of them they end after 128 products, in the weight gradient after 64 (then in double):
// over 194 shapes errors of 0.6 to 1.0 of those of the float kernels.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "conv_gather.h"
#include "conv_products.h"
#include "split_mfma.h"

using namespace cthip;

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ f32x4 zero4() { return f32x4{0.f, 0.f, 0.f, 0.f}; }

// Four consecutive floats of a row of n >= 4 from element i on, from an address that is a multiple
// of 4 bytes.  Beyond the row's end (i + 4 > n) it loads the row's last four: fix4 moves them.
__device__ __forceinline__ f32x4 load4(const float* row, uint32_t i, uint32_t n) {
  f32x4 v;
  __builtin_memcpy(&v, row + min(i, n - 4), 16);
  return v;
}
// What load4 loaded, with zeros beyond the row's end.
__device__ __forceinline__ f32x4 fix4(f32x4 v, uint32_t i, uint32_t n) {
  const uint32_t shift = i - min(i, n - 4);
  f32x4 out;
#pragma unroll
  for (uint32_t e = 0; e < 4; ++e) {
    float x = v[e];
#pragma unroll
    for (uint32_t d = 1; d + e < 4; ++d) x = shift == d ? v[e + d] : x;
    out[e] = i + e < n ? x : 0.f;
  }
  return out;
}

// Adds the sixteen products of a tile whose left and right elements four lanes hold, four each, to
// one sum, or to two sums, eight to each.
template <int kSums>
__device__ __forceinline__ void product16(f32x4 left, f32x4 right, f32x4 (&sums)[kSums]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    sums[i % kSums] = __builtin_amdgcn_mfma_f32_16x16x4f32(left[i], right[i], sums[i % kSums], 0, 0, 0);
}
// Matrix and vector instructions stay on their side; scalar ones and memory's may pass.
__device__ __forceinline__ void keep_order() { __builtin_amdgcn_sched_barrier(0x4 | 0x10 | 0x80); }

// Consecutive units of work on one die: neighbouring tiles share rows of the input in its L2.
__device__ __forceinline__ uint32_t unit_of_block(uint32_t b, uint32_t units) {
  const uint32_t per_die = (units + kXcds - 1) / kXcds;
  return (b % kXcds) * per_die + b / kXcds;
}

// ------------------------------------------------------------- forward and backward-data

// result[m][j] = sum over k of left[m][k] * right[k][j] over the positions j of all images,
// numbered on: image after image, so that small images fill whole tiles.
//   kForward: m = out channel, k = (channel, tap); right is gathered from the input while it
//     is staged (a lane keeps one position j, k is uniform per wave: consecutive lanes read
//     consecutive input elements) and written to the workspace on the way by the first row of
//     tiles: the unrolled matrix is written once and not read back.
//   otherwise: m = (channel, tap), k = out channel; right is the output gradient, the result
//     is the workspace.
//     Which taps of its window lie in the padding is a mask per lane, worked out once (windows
//     of up to kConvMaskTaps cells).  The k of a tile are decoded side by side, one to a lane, and
//     handed round with v_readlane: decoded one after the other on the scalar unit they took
//     as long as the tile's MFMAs.
// kChains: the sums that take turns with the sixteen products of a tile.
template <int BM, bool kForward, int kChains>
__global__ void __launch_bounds__(kBlock, 4) conv_product_kernel(const ConvProductArgs a) {
  constexpr int WM = BM / 128 + 1, WN = 4 / WM, BN = 32 * WN, BK = 16, LD = BK + 4;   // waves: WM x WN
  constexpr int MT = BM / WM / 16, kCols = kBlock / BN, kStep = BK / kCols;   // lanes to a column of `right`, k of each
  constexpr int kLeft = (BM * BK / 4 + kBlock - 1) / kBlock;   // 16-byte pieces of the left tile per lane
  __shared__ __attribute__((aligned(16))) float left_lds[2][BM * LD];
  __shared__ __attribute__((aligned(16))) float right_lds[2][BN * LD];
  const uint32_t unit = unit_of_block(blockIdx.x, a.units);
  if (unit >= a.units) return;
  uint32_t n_tile, m_tile;
  a.m_tiles_fd.divmod(unit, n_tile, m_tile);
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // The position whose column of `right` this lane stages, kStep of the k of a tile.  Rows and
  // columns beyond the result repeat the last one and are not stored; k beyond the last one are
  // zeros in both operands.
  const uint32_t j = n_tile * BN + (tid & (BN - 1));
  const bool j_ok = j < a.n;
  const uint32_t k_part = wave / (BN / 64) * kStep;
  uint32_t image, pos;
  a.rows_fd.divmod(min(j, a.n - 1), image, pos);
  uint32_t taps_inside = 0, corner = 0;   // of the window at this position; its first cell, modulo 2^32
  const float* src;
  float* cells = nullptr;
  if constexpr (kForward) {
    uint32_t oy, ox;
    a.out_w_fd.divmod(pos, oy, ox);
    const int32_t iy0 = (int32_t)oy * a.sy - a.py, ix0 = (int32_t)ox * a.sx - a.px;
    corner = (uint32_t)iy0 * a.in_w + (uint32_t)ix0;
    uint32_t bit = 1;
    for (uint32_t ky = 0; ky < a.kh; ++ky)
      for (uint32_t kx = 0; kx < a.kw; ++kx, bit <<= 1)
        taps_inside |= (((uint32_t)iy0 + ky < a.in_h) & ((uint32_t)ix0 + kx < a.in_w)) ? bit : 0u;
    src = a.input + (int64_t)image * a.in_image;
    cells = a.workspace + (int64_t)image * a.conv_image + pos;
  } else {
    src = a.output + (int64_t)image * a.out_image + pos;
  }

  f32x4 left_regs[kLeft];
  float right_regs[kStep];
  uint32_t tap_bits[kStep];               // uniform: of the staged k; 0 beyond the last one

  auto load_tile = [&](uint32_t k0) {
#pragma unroll
    for (int i = 0; i < kLeft; ++i) {
      const uint32_t piece = min(i * kBlock + tid, (uint32_t)(BM * BK / 4 - 1));
      if constexpr (kForward) {
        const uint32_t m = min(m_tile * BM + piece / (BK / 4), a.m - 1);
        left_regs[i] = load4(a.weights + (int64_t)m * a.k, k0 + piece % (BK / 4) * 4, a.k);
      } else {   // the weights as stored are [k][m]: consecutive lanes take consecutive m
        const uint32_t m = min(m_tile * BM + piece % BM, a.m - 1), k = k0 + piece / BM * 4;
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e) left_regs[i][e] = a.weights[(int64_t)min(k + e, a.k - 1) * a.m + m];
      }
    }
    const uint32_t k_first = k0 + k_part;
    if constexpr (kForward) {
      const uint32_t my_k = k_first + (lane & (kStep - 1));
      uint32_t channel, tap, ky, kx;
      a.taps_fd.divmod(my_k, channel, tap);
      a.kw_fd.divmod(tap, ky, kx);
      const uint32_t my_cell = channel * a.in_plane + ky * a.in_w + kx;
      const uint32_t my_bit = my_k < a.k ? 1u << tap : 0u;
#pragma unroll
      for (int e = 0; e < kStep; ++e) {
        tap_bits[e] = __builtin_amdgcn_readlane(my_bit, e);
        const uint32_t cell = corner + __builtin_amdgcn_readlane(my_cell, e);
        right_regs[e] = src[taps_inside & tap_bits[e] ? cell : 0u];
      }
    } else {
#pragma unroll
      for (uint32_t e = 0; e < kStep; ++e) right_regs[e] = src[min(k_first + e, a.k - 1) * a.n_rows];
    }
  };
  auto store_tile = [&](uint32_t k0, int buffer) {
    const bool last = k0 + BK > a.k;
    const uint32_t k_first = k0 + k_part;
    if (last) {
      asm volatile("");   // stays a branch: as selects it would cost every tile
#pragma unroll
      for (int i = 0; i < kLeft; ++i) {
        const uint32_t piece = min(i * kBlock + tid, (uint32_t)(BM * BK / 4 - 1));
        if constexpr (kForward) {
          left_regs[i] = fix4(left_regs[i], k0 + piece % (BK / 4) * 4, a.k);
        } else {
#pragma unroll
          for (uint32_t e = 0; e < 4; ++e) left_regs[i][e] = k0 + piece / BM * 4 + e < a.k ? left_regs[i][e] : 0.f;
        }
      }
      if constexpr (!kForward) {
#pragma unroll
        for (uint32_t e = 0; e < kStep; ++e) right_regs[e] = k_first + e < a.k ? right_regs[e] : 0.f;
      }
    }
#pragma unroll
    for (int i = 0; i < kLeft; ++i) {
      const uint32_t piece = i * kBlock + tid;
      const uint32_t row = kForward ? piece / (BK / 4) : piece % BM;
      const uint32_t at = (kForward ? piece % (BK / 4) : piece / BM) * 4;
      if (BM * BK / 4 % kBlock == 0 || piece < BM * BK / 4)
        *reinterpret_cast<f32x4*>(&left_lds[buffer][row * LD + at]) = left_regs[i];
    }
    if constexpr (kForward) {
#pragma unroll
      for (int e = 0; e < kStep; ++e) right_regs[e] = taps_inside & tap_bits[e] ? right_regs[e] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < kStep; e += 4)
      *reinterpret_cast<f32x4*>(&right_lds[buffer][(tid & (BN - 1)) * LD + k_part + e]) =
          f32x4{right_regs[e], right_regs[e + 1], right_regs[e + 2], right_regs[e + 3]};
    if constexpr (kForward) {
      if (m_tile == 0 && j_ok) {
        float* to = cells + (int64_t)k_first * a.n_rows;
        if (last) {
#pragma unroll
          for (int e = 0; e < kStep; ++e)
            if (k_first + e < a.k) to[(int64_t)e * a.n_rows] = right_regs[e];
        } else {
#pragma unroll
          for (int e = 0; e < kStep; ++e) to[(int64_t)e * a.n_rows] = right_regs[e];
        }
      }
    }
  };

  f32x4 total[MT][2];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u) total[t][u] = zero4();

  load_tile(0);
  store_tile(0, 0);
  __syncthreads();
  const uint32_t row = lane & 15, group = lane >> 4;
  const uint32_t wave_m = wave / WN * (MT * 16), wave_n = wave % WN * 32;
  auto multiply = [&](int buffer, auto chains) {
    constexpr int kSums = decltype(chains)::value;
    f32x4 l4[MT], r4[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
      r4[u] = *reinterpret_cast<const f32x4*>(&right_lds[buffer][(wave_n + u * 16 + row) * LD + 4 * group]);
#pragma unroll
    for (int t = 0; t < MT; ++t)
      l4[t] = *reinterpret_cast<const f32x4*>(&left_lds[buffer][(wave_m + t * 16 + row) * LD + 4 * group]);
    // the sums of a row of tiles are added up while the next row's products run
    f32x4 sums[MT][2][kSums];
#pragma unroll
    for (int t = 0; t <= MT; ++t) {
      if (t < MT) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          sums[t][u][0] = sums[t][u][kSums - 1] = zero4();
          product16(l4[t], r4[u], sums[t][u]);
        }
      }
      if (t > 0) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const auto& sum = sums[t - 1][u];
          total[t - 1][u] += kSums == 2 ? sum[0] + sum[kSums - 1] : sum[0];
          asm volatile("" : "+v"(total[t - 1][u]));   // added here, not after the next tile's stores
        }
      }
      if constexpr (kForward || BM == 128) keep_order();
    }
  };
  // The last tile is multiplied after the loop: with its loads under a condition every tile
  // waited, ahead of its own, for whatever was in flight, the workspace's stores included.
  int buffer = 0;
  const uint32_t k_last = (a.k - 1) / BK * BK;
  for (uint32_t k0 = 0; k0 < k_last; k0 += BK) {
    load_tile(k0 + BK);
    multiply(buffer, std::integral_constant<int, kChains>());
    store_tile(k0 + BK, buffer ^ 1);
    __syncthreads();
    buffer ^= 1;
  }
  multiply(buffer, std::integral_constant<int, 2>());

  auto store_columns = [&](int u, bool whole) {
    const uint32_t out_j = n_tile * BN + wave_n + u * 16 + row;
    if (out_j >= a.n) return;
    uint32_t out_image, out_pos;
    a.rows_fd.divmod(out_j, out_image, out_pos);
    const uint32_t m0 = m_tile * BM + wave_m + 4 * group;
    float* to = (kForward ? a.output + (int64_t)out_image * a.out_image : a.workspace + (int64_t)out_image * a.conv_image) +
                out_pos + (int64_t)m0 * a.n_rows;
    const bool add = kForward && a.beta != 0.f;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float* at = to + (int64_t)(t * 16 + r) * a.n_rows;
        const float sum = total[t][u][r];
        if (whole || m0 + t * 16 + r < a.m) *at = add ? sum + a.beta * *at : sum;
      }
  };
  const bool whole = m_tile * BM + BM <= a.m;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    if (whole) store_columns(u, true);
    else store_columns(u, false);
  }
}

// ------------------------------------------------------ forward and backward-data, three pieces to a float

// A buffer of `bytes` from `base` on, below 2^31: loads beyond it return zeros, stores beyond it are dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const float* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, bytes, 0x00027000);
}
// A lane's offset beyond every buffer.  The scalar offset next to it is taken off the buffer's length before the two are
// compared, and must not exceed it.
constexpr uint32_t kOutside = 0x80000000u;
// A workspace that the last-level cache does not hold goes past the caches: a wave's loads wait for the stores in front of
// them, and those for room in the caches ([64, 64, 56, 56] under 64 windows of 3 x 3, 462 MB, us: forward 207 -> 193, input
// gradient with the roll back 248 -> 234; but [50, 248, 23, 23] under 21, 236 MB, which the roll back then reads from
// memory, 98 -> 186).  Which ones: past_the_caches.
constexpr int kStreaming = 2;
constexpr int64_t kLastLevelCache = int64_t(256) << 20;
template <bool kPast>
__device__ __forceinline__ void store_cell(float x, __amdgpu_buffer_rsrc_t cells, uint32_t at, uint32_t row) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, x), cells, at, row, kPast ? kStreaming : 0);
}

// Element `chunk` (of eight k) of row `row` of a tile in LDS, rows of 32 k: eight consecutive rows' reads of one chunk
// cover 128 bytes' worth of banks once.
__device__ __forceinline__ uint32_t tile_at(uint32_t row, uint32_t chunk) { return row * 32 + ((chunk ^ (row >> 1)) & 3) * 8; }

// Both: result[m][j] = sum over k of left[m][k] * right[k][j] over the positions j of all images, numbered on: image after
// image, so that small images fill whole tiles.  Left are the weights, right is loaded a position to a lane, k uniform, so
// that consecutive lanes read consecutive elements.
//
// A wave owns 64 positions and needs no LDS for them: what a lane holds of sixteen k of its position, split into pieces,
// v_permlane32_swap turns into the matrix cores' fragments of 32 positions each.  The weights are split by the block and go
// through LDS.

// The fragments of 2 x 32 positions from sixteen k of a lane's position.
__device__ __forceinline__ void split_positions(const float* x, bf16x8 (&r)[2][kSplitPieces], const SplitWeights& w) {
  u32x4 low[kSplitPieces], high[kSplitPieces];   // k 0 .. 7 and 8 .. 15
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    split4(f32x4{x[4 * h], x[4 * h + 1], x[4 * h + 2], x[4 * h + 3]}, low, 4 * h, w);
    split4(f32x4{x[4 * h + 8], x[4 * h + 9], x[4 * h + 10], x[4 * h + 11]}, high, 4 * h, w);
  }
#pragma unroll
  for (int p = 0; p < kSplitPieces; ++p) {
    u32x4 first, second;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const auto both = __builtin_amdgcn_permlane32_swap(low[p][e], high[p][e], false, false);
      first[e] = both[0];
      second[e] = both[1];
    }
    r[0][p] = __builtin_bit_cast(bf16x8, first);
    r[1][p] = __builtin_bit_cast(bf16x8, second);
  }
}

// The same product in float, sums of eight: what a block does that found no finite sum.  load(k0, x) loads eight k of the
// lane's position, weight(row, k) is a weight; zeros beyond the operands.
template <int MT, class Load, class Weight>
__device__ __forceinline__ void product_in_float(f32x16 (&total)[MT][2], uint32_t k_count, Load load, Weight weight) {
  const uint32_t lane = threadIdx.x & 63;
#pragma unroll
  for (int t = 0; t < MT; ++t) total[t][0] = total[t][1] = zero16();
  for (uint32_t k0 = 0; k0 < k_count; k0 += 8) {
    float x[8];
    load(k0, x);
    f32x16 sum[MT][2];
#pragma unroll
    for (int t = 0; t < MT; ++t) sum[t][0] = sum[t][1] = zero16();
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const auto both = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x[e]), __builtin_bit_cast(uint32_t, x[e + 1]),
                                                         false, false);
      const uint32_t first = both[0], second = both[1];
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const float l = weight(t * 32 + (lane & 31), k0 + e + lane / 32);
        sum[t][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(l, __builtin_bit_cast(float, first), sum[t][0], 0, 0, 0);
        sum[t][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(l, __builtin_bit_cast(float, second), sum[t][1], 0, 0, 0);
      }
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) total[t][u] += sum[t][u];
  }
}

// Forward: m = out channel, k = (channel, tap); right is gathered from the input and written to the workspace on the way by
// the first row of tiles: the unrolled matrix is written once and not read back.  Which taps of its window lie in the
// padding is a mask per lane, worked out once (windows of up to kConvMaskTaps cells); the loads of those taps go beyond the
// buffer and return zero: two vector instructions a cell.  The k of a tile are decoded side by side, one to a lane, and
// handed round with v_readlane: decoded one after the other on the scalar unit they took as long as the tile's products.
constexpr int kPositions = 256;   // of a block: a position to a lane

template <int MT, bool kPast>
__global__ void __launch_bounds__(kPositions, 2) conv_forward_kernel(const ConvProductArgs a) {
  constexpr int BM = 32 * MT, BK = 32, kPlane = BM * BK;
  __shared__ __attribute__((aligned(16))) uint16_t lds[2][kSplitPieces][kPlane];
  const uint32_t unit = unit_of_block(blockIdx.x, a.units);
  if (unit >= a.units) return;
  uint32_t n_tile, m_tile;
  a.m_tiles_fd.divmod(unit, n_tile, m_tile);
  const uint32_t tid = threadIdx.x, lane = tid & 63, row = lane & 31, half = lane >> 5;

  // Rows and positions beyond the result repeat the last one and are not stored; k beyond the last one repeat it and are
  // set to zero in both operands.
  const uint32_t j = n_tile * kPositions + tid;
  uint32_t image, pos, oy, ox;
  a.rows_fd.divmod(min(j, a.n - 1), image, pos);
  a.out_w_fd.divmod(pos, oy, ox);
  const int32_t iy0 = (int32_t)oy * a.sy - a.py, ix0 = (int32_t)ox * a.sx - a.px;
  uint32_t taps_outside = 0, bit = 1;   // of the window at this position
  for (uint32_t ky = 0; ky < a.kh; ++ky)
    for (uint32_t kx = 0; kx < a.kw; ++kx, bit <<= 1)
      taps_outside |= (((uint32_t)iy0 + ky < a.in_h) & ((uint32_t)ix0 + kx < a.in_w)) ? 0u : bit;
  // bytes, from the first row and column of the padding on, so that no window begins below the base
  const uint32_t padding = gather_padding(a.in_w, a.px, a.py), length = gather_length(a.images, (uint32_t)a.in_image, padding);
  const __amdgpu_buffer_rsrc_t source = buffer_of(a.input - padding, length * 4);
  const __amdgpu_buffer_rsrc_t cells = buffer_of(a.workspace, a.images * (uint32_t)a.conv_image * 4);
  const uint32_t from = gather_window(image, (uint32_t)a.in_image, a.in_w, padding, iy0, ix0) * 4;
  const uint32_t to = m_tile == 0 && j < a.n ? (image * (uint32_t)a.conv_image + pos) * 4 : kOutside;

  // kCount k from k0 on, decoded by the lanes and loaded
  auto gather = [&](uint32_t k0, float* x, auto count) {
    constexpr int kCount = decltype(count)::value;
    const uint32_t my_k = min(k0 + (lane & (kCount - 1)), a.k - 1);
    uint32_t channel, tap, ky, kx;
    a.taps_fd.divmod(my_k, channel, tap);
    a.kw_fd.divmod(tap, ky, kx);
    const uint32_t my_cell = gather_tap(channel, ky, kx, a.in_plane, a.in_w, length) * 4, my_shift = 31 - tap;
#pragma unroll
    for (int e = 0; e < kCount; ++e) {
      const uint32_t at = from | ((taps_outside << __builtin_amdgcn_readlane(my_shift, e)) & kOutside);
      x[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(source, at, __builtin_amdgcn_readlane(my_cell, e), 0));
    }
  };
  constexpr std::integral_constant<int, 16> kSixteen{};
  const bool stages_left = BM * 4 >= kPositions || tid < BM * 4;
  const uint32_t left_row = tid / 4, left_chunk = tid % 4;
  const float* weights = a.weights + (int64_t)min(m_tile * BM + left_row, a.m - 1) * a.k;
  f32x4 left_raw[2];
  auto load_left = [&](uint32_t k0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) left_raw[h] = load4(weights, k0 + left_chunk * 8 + h * 4, a.k);
  };
  const SplitWeights split_weights;
  auto stage_left = [&](int buffer) {
    u32x4 pieces[kSplitPieces];
    split4(left_raw[0], pieces, 0, split_weights);
    split4(left_raw[1], pieces, 4, split_weights);
    if (!stages_left) return;
#pragma unroll
    for (int p = 0; p < kSplitPieces; ++p) *reinterpret_cast<u32x4*>(&lds[buffer][p][tile_at(left_row, left_chunk)]) = pieces[p];
  };

  // The sums of a tile of 32 k: the ten small products of its halves, behind them the two large ones, so that few roundings
  // are at the size of a tile's sum and none at that of the total but its own addition.  Summed through, the leading pieces
  // apart from the others, the errors were 1.3 to 1.45 times the float kernel's over operands of one sign and up to 1.28 over
  // long sums of either; now they are 0.66 to 0.92 (k 576, normal operands 1.35e-7 -> 0.93e-7, the float kernel's 1.27e-7;
  // uniform ones 1.34e-7 -> 0.68e-7, 0.93e-7), for 0 to 4 % of the time.  Where there is one tile of rows the totals are added
  // up a tile later: right behind the products they waited for them ([32, 32, 56, 56] under 32 36.5 us, later 32.8).
  constexpr bool kLater = MT == 1;
  f32x16 sums[MT][2], total[MT][2];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u) sums[t][u] = total[t][u] = zero16();
  auto add_up = [&] {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) total[t][u] += sums[t][u];
  };
  float raw[2][16];
  bf16x8 leading[2];   // of the positions, in the first half
  auto multiply = [&](int buffer, int part, const bf16x8 (&r)[2][kSplitPieces], bool last) {
    auto weights_at = [&](int t, int half_tile, int p) {
      return *reinterpret_cast<const bf16x8*>(&lds[buffer][p][tile_at(t * 32 + row, half_tile * 2 + half)]);
    };
    bf16x8 l[MT][kSplitPieces];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int p = 0; p < kSplitPieces; ++p) l[t][p] = weights_at(t, part, p);
    if (part == 0) {
      if (kLater) add_up();
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u) sums[t][u] = zero16();
    }
#pragma unroll
    for (int i = 0; i + 1 < kSplitProducts; ++i)
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u)
          sums[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l[t][kSplitLeft[i]], r[u][kSplitRight[i]], sums[t][u], 0, 0, 0);
    if (part == 1) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const bf16x8 first = weights_at(t, 0, 0);
#pragma unroll
        for (int u = 0; u < 2; ++u) sums[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(first, leading[u], sums[t][u], 0, 0, 0);
      }
    }
    if (part == 1 || last) {
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u) sums[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l[t][0], r[u][0], sums[t][u], 0, 0, 0);
      if (!kLater) add_up();
    }
    if (part == 0) {
#pragma unroll
      for (int u = 0; u < 2; ++u) leading[u] = r[u][0];
    }
  };
  load_left(0);
  gather(0, raw[0], kSixteen);
  gather(16, raw[1], kSixteen);
  const uint32_t whole = a.k / BK * BK;
  if (whole) stage_left(0);
  load_left(BK);
  __syncthreads();
  // The whole tiles.  No branch stands in the loop: behind loads and stores that may or may not have been issued every wait
  // would be one for all of them.
  for (uint32_t k0 = 0; k0 < whole; k0 += BK) {
    const int buffer = k0 / BK & 1;
    stage_left(buffer ^ 1);   // behind the last whole tile: not used
#pragma unroll
    for (int part = 0; part < 2; ++part) {
      float* x = raw[part];
      const uint32_t k = k0 + part * 16;
#pragma unroll
      for (uint32_t e = 0; e < 16; ++e)
        store_cell<kPast>(x[e], cells, to, (k + e) * a.n_rows * 4);
      bf16x8 r[2][kSplitPieces];
      split_positions(x, r, split_weights);
      gather(k + BK, x, kSixteen);
      if (part == 0) load_left(k0 + 2 * BK);
      multiply(buffer, part, r, false);
    }
    __syncthreads();
  }
  if (whole < a.k) {
    load_left(whole);
#pragma unroll
    for (int h = 0; h < 2; ++h) left_raw[h] = fix4(left_raw[h], whole + left_chunk * 8 + h * 4, a.k);
    stage_left(0);
    __syncthreads();
#pragma unroll
    for (int part = 0; part < 2; ++part) {
      float* x = raw[part];
      const uint32_t k = whole + part * 16;
      if (k >= a.k) break;
#pragma unroll
      for (uint32_t e = 0; e < 16; ++e) {
        x[e] = k + e < a.k ? x[e] : 0.f;
        if (k + e < a.k)
          store_cell<kPast>(x[e], cells, to, (k + e) * a.n_rows * 4);
      }
      bf16x8 r[2][kSplitPieces];
      split_positions(x, r, split_weights);
      multiply(0, part, r, k + 16 >= a.k);
    }
  }

  if (kLater) add_up();
  bool found = false;
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        found |= not_finite(total[t][u][e]);
        total[t][u][e] *= kSplitUnscale;
      }
  if (__syncthreads_or(found))
    product_in_float<MT>(
        total, a.k,
        [&](uint32_t k0, float* x) {
          gather(k0, x, std::integral_constant<int, 8>());
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = k0 + e < a.k ? x[e] : 0.f;
        },
        [&](uint32_t m, uint32_t k) {
          const float w = a.weights[(int64_t)min(m_tile * BM + m, a.m - 1) * a.k + min(k, a.k - 1)];
          return k < a.k ? w : 0.f;
        });
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const uint32_t out_j = n_tile * kPositions + (tid & ~63u) + u * 32 + row;
    if (out_j >= a.n) continue;
    uint32_t out_image, out_pos;
    a.rows_fd.divmod(out_j, out_image, out_pos);
    const uint32_t m0 = m_tile * BM + 4 * half;
    float* first = a.output + (int64_t)out_image * a.out_image + out_pos + (int64_t)m0 * a.n_rows;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const uint32_t m = t * 32 + 8 * (e / 4) + e % 4;
        float* cell = first + (int64_t)m * a.n_rows;
        if (m0 + m < a.m) *cell = a.beta != 0.f ? total[t][u][e] + a.beta * *cell : total[t][u][e];
      }
  }
}

// Backward-data over few out channels (KS runs of sixteen): m = (channel, tap), k = out channel; right is the output
// gradient, the result is the workspace.  The fragments of a wave's positions stay in registers while the block goes through
// the rows in tiles of 32, whose weights are split one tile ahead: a tile is 12 * KS products between two barriers.
template <int KS, bool kPast>
__global__ void __launch_bounds__(kPositions, 2) conv_data_few_kernel(const ConvProductArgs a) {
  constexpr int BM = 32, K = 16 * KS, kChunks = K / 8, kPlane = BM * K;
  __shared__ __attribute__((aligned(16))) uint16_t lds[2][kSplitPieces][kPlane];
  const uint32_t unit = unit_of_block(blockIdx.x, a.units);
  if (unit >= a.units) return;
  uint32_t n_tile, m_part;
  a.m_tiles_fd.divmod(unit, n_tile, m_part);
  const uint32_t tid = threadIdx.x, lane = tid & 63, row = lane & 31, half = lane >> 5;
  const uint32_t m_first = m_part * a.rows_per_block, m_end = min(a.m, m_first + a.rows_per_block);
  const uint32_t j = n_tile * kPositions + tid;
  uint32_t image, pos;
  a.rows_fd.divmod(min(j, a.n - 1), image, pos);
  const __amdgpu_buffer_rsrc_t source = buffer_of(a.output, a.images * (uint32_t)a.out_image * 4);
  const uint32_t from = (image * (uint32_t)a.out_image + pos) * 4;
  auto load = [&](uint32_t k) {
    const float x = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(source, from, min(k, a.k - 1) * a.n_rows * 4, 0));
    return k < a.k ? x : 0.f;
  };
  auto lds_at = [&](uint32_t r, uint32_t chunk) {
    return r * K + (KS == 4 ? (chunk ^ r) & 7 : (chunk ^ (r >> 1)) & 3) * 8;
  };
  // the weights as stored are [k][m]: consecutive lanes take consecutive m
  const uint32_t left_row = tid % BM, left_chunk = tid / BM;
  const bool stages_left = kChunks * BM >= kPositions || left_chunk < kChunks;
  f32x4 left_raw[2];
  auto load_left = [&](uint32_t m0) {
    const float* weights = a.weights + min(m0 + left_row, a.m - 1);
#pragma unroll
    for (uint32_t e = 0; e < 8; ++e) {
      const uint32_t k = (left_chunk & (kChunks - 1)) * 8 + e;
      left_raw[e / 4][e % 4] = weights[(int64_t)min(k, a.k - 1) * a.m];
    }
  };
  const SplitWeights split_weights;
  auto stage_left = [&](int buffer) {
#pragma unroll
    for (uint32_t e = 0; e < 8; ++e) left_raw[e / 4][e % 4] = left_chunk * 8 + e < a.k ? left_raw[e / 4][e % 4] : 0.f;
    u32x4 pieces[kSplitPieces];
    split4(left_raw[0], pieces, 0, split_weights);
    split4(left_raw[1], pieces, 4, split_weights);
    if (!stages_left) return;
#pragma unroll
    for (int p = 0; p < kSplitPieces; ++p) *reinterpret_cast<u32x4*>(&lds[buffer][p][lds_at(left_row, left_chunk)]) = pieces[p];
  };

  bf16x8 r[KS][2][kSplitPieces];
  load_left(m_first);
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    float x[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) x[e] = load(ks * 16 + e);
    split_positions(x, r[ks], split_weights);
  }
  stage_left(0);
  load_left(m_first + BM);
  const __amdgpu_buffer_rsrc_t cells = buffer_of(a.workspace, a.images * (uint32_t)a.conv_image * 4);
  uint32_t to[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const uint32_t out_j = n_tile * kPositions + (tid & ~63u) + u * 32 + row;
    uint32_t out_image, out_pos;
    a.rows_fd.divmod(min(out_j, a.n - 1), out_image, out_pos);
    to[u] = out_j < a.n ? (out_image * (uint32_t)a.conv_image + out_pos + 4 * half * a.n_rows) * 4 : kOutside;
  }
  auto store_rows = [&](uint32_t m0, int u, const f32x16& value) {
#pragma unroll
    for (uint32_t e = 0; e < 16; ++e) {
      const uint32_t m = m0 + 8 * (e / 4) + e % 4;   // of the lanes' first half
      const uint32_t at = m0 + BM <= a.m || m + 4 * half < a.m ? to[u] : kOutside;
      store_cell<kPast>(value[e], cells, at, min(m, a.m - 1) * a.n_rows * 4);   // by value: a bit cast of a vector's element takes the first one
    }
  };
  float never = 0.f;   // zero, or NaN behind a sum that is not finite
  __syncthreads();
  int buffer = 0;
  for (uint32_t m0 = m_first; m0 < m_end; m0 += BM, buffer ^= 1) {
    f32x16 sums[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) sums[0][u] = sums[1][u] = zero16();
    stage_left(buffer ^ 1);
    load_left(m0 + 2 * BM);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      bf16x8 l[kSplitPieces];
#pragma unroll
      for (int p = 0; p < kSplitPieces; ++p) l[p] = *reinterpret_cast<const bf16x8*>(&lds[buffer][p][lds_at(row, ks * 2 + half)]);
#pragma unroll
      for (int i = 0; i < kSplitProducts; ++i)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          f32x16& sum = sums[i + 1 < kSplitProducts][u];
          sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l[kSplitLeft[i]], r[ks][u][kSplitRight[i]], sum, 0, 0, 0);
        }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      f32x16 value = sums[0][u] + sums[1][u];
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        never = __builtin_fmaf(value[e], 0.f, never);
        value[e] *= kSplitUnscale;
      }
      store_rows(m0, u, value);
    }
    __syncthreads();
  }
  if (__syncthreads_or(never != 0.f)) {
    for (uint32_t m0 = m_first; m0 < m_end; m0 += BM) {
      f32x16 total[1][2];
      product_in_float<1>(
          total, a.k,
          [&](uint32_t k0, float* x) {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = load(k0 + e);
          },
          [&](uint32_t m, uint32_t k) {
            const float w = a.weights[(int64_t)min(k, a.k - 1) * a.m + min(m0 + m, a.m - 1)];
            return k < a.k ? w : 0.f;
          });
      store_rows(m0, 0, total[0][0]);
      store_rows(m0, 1, total[0][1]);
    }
  }
}

// Backward-data over any number of out channels: both operands go through LDS.  Sums of four tiles of k (128 products) are
// added to the totals, in float.
template <int BM>
__global__ void __launch_bounds__(BM == 128 ? 512 : 256, 2) conv_data_kernel(const ConvProductArgs a) {
  constexpr int T = BM == 128 ? 512 : 256, BN = 128, BK = 32, WM = BM / 32, WN = T / 64 / WM, NT = BN / WN / 32;
  constexpr int kStep = BK * BN / T, kRuns = kStep / 8;   // k of a column of `right` that a lane stages, in runs of eight
  static_assert(BM * BK / 8 == T, "a run of eight k of the left operand to a lane");
  constexpr int kPlane = (BM + BN) * BK, kBuffer = kSplitPieces * kPlane;
  constexpr uint32_t kTilesToASum = 4;
  __shared__ __attribute__((aligned(16))) uint16_t lds[2 * kBuffer];   // [buffer][piece][rows of the left, of the right operand]
  const uint32_t unit = unit_of_block(blockIdx.x, a.units);
  if (unit >= a.units) return;
  uint32_t n_tile, m_tile;
  a.m_tiles_fd.divmod(unit, n_tile, m_tile);
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // The position whose column of `right` this lane stages, kStep of the k of a tile.  Rows and
  // columns beyond the result repeat the last one and are not stored; k beyond the last one repeat it and are set to
  // zero in both operands.
  const uint32_t column = tid & (BN - 1), j = n_tile * BN + column;
  const uint32_t k_part = wave / (BN / 64) * kStep;
  uint32_t image, pos;
  a.rows_fd.divmod(min(j, a.n - 1), image, pos);
  const __amdgpu_buffer_rsrc_t source = buffer_of(a.output, a.images * (uint32_t)a.out_image * 4);
  const uint32_t from = (image * (uint32_t)a.out_image + pos) * 4;

  const uint32_t left_row = tid % BM, left_chunk = tid / BM;
  const float* weights = a.weights + min(m_tile * BM + left_row, a.m - 1);
  f32x4 left_raw[2];
  float right_raw[kStep];
  auto load_left = [&](uint32_t k0) {
    const uint32_t k = min(k0, (a.k - 1) / BK * BK) + left_chunk * 8;
    // the weights as stored are [k][m]: consecutive lanes take consecutive m
#pragma unroll
    for (uint32_t e = 0; e < 8; ++e) left_raw[e / 4][e % 4] = weights[(int64_t)min(k + e, a.k - 1) * a.m];
  };
  auto load_right = [&](uint32_t k0, int run) {
    const uint32_t k_first = k0 + k_part + run * 8;
#pragma unroll
    for (uint32_t e = 0; e < 8; ++e)
      right_raw[run * 8 + e] = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(source, from, min(k_first + e, a.k - 1) * a.n_rows * 4, 0));
  };
  // k beyond the last one, in the last tile only
  auto drop_left = [&](uint32_t k0) {
    if (k0 + BK <= a.k) return;
    asm volatile("");   // stays a branch: as selects it would cost every tile
    const uint32_t k = k0 + left_chunk * 8;
#pragma unroll
    for (uint32_t e = 0; e < 8; ++e) left_raw[e / 4][e % 4] = k + e < a.k ? left_raw[e / 4][e % 4] : 0.f;
  };
  auto drop_right = [&](uint32_t k0, int run) {
    if (k0 + BK <= a.k) return;
    asm volatile("");
#pragma unroll
    for (uint32_t e = 0; e < 8; ++e) right_raw[run * 8 + e] = k0 + k_part + run * 8 + e < a.k ? right_raw[run * 8 + e] : 0.f;
  };
  const uint32_t row = lane & 31, half = lane >> 5;
  const uint32_t wave_m = wave / WN * 32, wave_n = wave % WN * (NT * 32);
  f32x16 total[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) total[u] = zero16();
  const uint32_t tiles = (a.k + BK - 1) / BK;

  {
    const SplitWeights split_weights;
    const uint32_t stage_left_at = tile_at(left_row, left_chunk);
    // the next tile: the left operand's run, and those of the right one
    auto stage_left = [&](uint32_t k0, uint16_t* buffer) {
      drop_left(k0);
      u32x4 pieces[kSplitPieces];
      split4(left_raw[0], pieces, 0, split_weights);
      split4(left_raw[1], pieces, 4, split_weights);
#pragma unroll
      for (int p = 0; p < kSplitPieces; ++p) *reinterpret_cast<u32x4*>(buffer + p * kPlane + stage_left_at) = pieces[p];
    };
    auto stage_right = [&](uint32_t k0, int run, uint16_t* buffer) {
      drop_right(k0, run);
      u32x4 pieces[kSplitPieces];
      const float* x = right_raw + run * 8;
      split4(f32x4{x[0], x[1], x[2], x[3]}, pieces, 0, split_weights);
      split4(f32x4{x[4], x[5], x[6], x[7]}, pieces, 4, split_weights);
      uint16_t* at = buffer + BM * BK + tile_at(column, k_part / 8 + run);
#pragma unroll
      for (int p = 0; p < kSplitPieces; ++p) *reinterpret_cast<u32x4*>(at + p * kPlane) = pieces[p];
    };
    bf16x8 l[2][kSplitPieces], r[2][NT][kSplitPieces];
    auto fetch_left = [&](const uint16_t* buffer, int part, int p) {
      l[part][p] = *reinterpret_cast<const bf16x8*>(buffer + p * kPlane + tile_at(wave_m + row, part * 2 + half));
    };
    auto fetch_right = [&](const uint16_t* buffer, int part, int p) {
#pragma unroll
      for (int u = 0; u < NT; ++u)
        r[part][u][p] = *reinterpret_cast<const bf16x8*>(buffer + p * kPlane + BM * BK + tile_at(wave_n + u * 32 + row, part * 2 + half));
    };
    // after product i of a half: the next half's pieces, those that its first product needs early
    auto fetch_next = [&](int i, const uint16_t* buffer, int part) {
      if (i == 0) {
        fetch_left(buffer, part, 0);
        fetch_right(buffer, part, 0);
        fetch_right(buffer, part, 2);
      }
      if (i == 1) fetch_left(buffer, part, 2);
      if (i == 3) fetch_right(buffer, part, 1);
      if (i == 4) fetch_left(buffer, part, 1);
    };
    f32x16 sums[2][NT];   // the products of the leading pieces; all others
#pragma unroll
    for (int u = 0; u < NT; ++u) sums[0][u] = sums[1][u] = zero16();
    auto multiply = [&](int part, int i) {
#pragma unroll
      for (int u = 0; u < NT; ++u) {
        f32x16& sum = sums[i + 1 < kSplitProducts][u];
        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l[part][kSplitLeft[i]], r[part][u][kSplitRight[i]], sum, 0, 0, 0);
      }
    };
    load_left(0);
#pragma unroll
    for (int run = 0; run < kRuns; ++run) load_right(0, run);
    stage_left(0, lds);
    load_left(BK);
#pragma unroll
    for (int run = 0; run < kRuns; ++run) {
      stage_right(0, run, lds);
      load_right(BK, run);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kSplitProducts; ++i) fetch_next(i, lds, 0);
    // Every tile but the last: the products of its first half run beside the splitting of the next tile into the other
    // buffer, those of the second beside the reads of the next tile's first fragments.
    for (uint32_t tile = 0; tile + 1 < tiles; ++tile) {
      uint16_t* here = lds + (tile & 1) * kBuffer;
      uint16_t* there = lds + (~tile & 1) * kBuffer;
      const uint32_t next = (tile + 1) * BK;
#pragma unroll
      for (int i = 0; i < kSplitProducts; ++i) {
        multiply(0, i);
        fetch_next(i, here, 1);
        if (i == 0) {
          stage_left(next, there);
          load_left(next + BK);
        }
        if (i == 2 || (i == 4 && kRuns > 1)) {
          const int run = i / 2 - 1;
          stage_right(next, run, there);
          load_right(next + BK, run);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < kSplitProducts; ++i) {
        multiply(1, i);
        fetch_next(i, there, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (tile % kTilesToASum == kTilesToASum - 1) {
#pragma unroll
        for (int u = 0; u < NT; ++u) {
          total[u] += sums[0][u] + sums[1][u];
          sums[0][u] = sums[1][u] = zero16();
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kSplitProducts; ++i) {
      multiply(0, i);
      fetch_next(i, lds + (~tiles & 1) * kBuffer, 1);
    }
#pragma unroll
    for (int i = 0; i < kSplitProducts; ++i) multiply(1, i);
#pragma unroll
    for (int u = 0; u < NT; ++u) total[u] += sums[0][u] + sums[1][u];
  }

  bool found = false;
#pragma unroll
  for (int u = 0; u < NT; ++u)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      found |= not_finite(total[u][e]);
      total[u][e] *= kSplitUnscale;
    }
  if (__syncthreads_or(found)) {
    // In float: chains of eight products, added up.
    constexpr int LD = BK + 4;
    float* left_lds = reinterpret_cast<float*>(lds);
    float* right_lds = left_lds + BM * LD;
    static_assert((BM + BN) * LD * 4 <= 2 * kBuffer * 2, "the floats fit where their pieces were");
#pragma unroll
    for (int u = 0; u < NT; ++u) total[u] = zero16();
    for (uint32_t k0 = 0; k0 < a.k; k0 += BK) {
      load_left(k0);
      drop_left(k0);
      *reinterpret_cast<f32x4*>(left_lds + left_row * LD + left_chunk * 8) = left_raw[0];
      *reinterpret_cast<f32x4*>(left_lds + left_row * LD + left_chunk * 8 + 4) = left_raw[1];
#pragma unroll
      for (int run = 0; run < kRuns; ++run) {
        load_right(k0, run);
        drop_right(k0, run);
#pragma unroll
        for (int e = 0; e < 8; ++e) right_lds[column * LD + k_part + run * 8 + e] = right_raw[run * 8 + e];
      }
      __syncthreads();
      for (int k = 0; k < BK; k += 8) {
        const f32x4 l = *reinterpret_cast<const f32x4*>(left_lds + (wave_m + row) * LD + k + 4 * half);
#pragma unroll
        for (int u = 0; u < NT; ++u) {
          const f32x4 r = *reinterpret_cast<const f32x4*>(right_lds + (wave_n + u * 32 + row) * LD + k + 4 * half);
          f32x16 sum = zero16();
#pragma unroll
          for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(l[e], r[e], sum, 0, 0, 0);
          total[u] += sum;
        }
      }
      __syncthreads();
    }
  }

#pragma unroll
  for (int u = 0; u < NT; ++u) {
    const uint32_t out_j = n_tile * BN + wave_n + u * 32 + row;
    if (out_j >= a.n) continue;
    uint32_t out_image, out_pos;
    a.rows_fd.divmod(out_j, out_image, out_pos);
    const uint32_t m0 = m_tile * BM + wave_m + 4 * half;
    float* first = a.workspace + (int64_t)out_image * a.conv_image + out_pos + (int64_t)m0 * a.n_rows;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const uint32_t m = 8 * (e / 4) + e % 4;
      float* cell = first + (int64_t)m * a.n_rows;
      if (m0 + m < a.m) *cell = total[u][e];
    }
  }
}

// ------------------------------------------------------------------------ backward-weights

// partial[split][m][n] = sum over the split's positions of output_gradient[m][p] * unrolled[n][p]:
// both operands have the positions innermost.  The positions of every image are cut into pieces
// of kConvPiece (the last one shorter), a split takes a run of consecutive pieces: the result is
// small (64 x 576 is 9 tiles), the chip is filled by the splits.  A single split adds to the
// weight gradient itself.
// Two groups of WM x WN waves share a tile of positions and take half of it each: twice the
// waves in flight for the same partials, which are added in LDS at the end.
template <int WM, int WN>
__global__ void __launch_bounds__(128 * WM * WN, 2) conv_weight_gradient_kernel(const ConvWeightArgs a) {
  constexpr int BM = 32 * WM, BN = 32 * WN, BK = kConvPiece, LD = BK + 4, THREADS = 128 * WM * WN;
  constexpr int kLeft = BM * BK / 4 / THREADS, kRight = BN * BK / 4 / THREADS;
  __shared__ __attribute__((aligned(16))) float left_lds[2][BM * LD];
  __shared__ __attribute__((aligned(16))) float right_lds[2][BN * LD];
  const uint32_t unit = unit_of_block(blockIdx.x, a.units);
  if (unit >= a.units) return;
  uint32_t split, tile, m_tile, n_tile;
  a.tiles_fd.divmod(unit, split, tile);
  a.n_tiles_fd.divmod(tile, m_tile, n_tile);
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t first_piece = split * a.pieces_per_split;
  const uint32_t piece_end = min(first_piece + a.pieces_per_split, a.pieces);

  // The piece that is loaded: positions [p0, p0 + BK) of an image, as far as it has them.
  // Rows beyond the result repeat the last one and are not stored.
  uint32_t piece = first_piece, image, part;
  a.parts_fd.divmod(piece, image, part);
  uint32_t p0 = part * BK;
  const float* left = a.output_gradient + (int64_t)image * a.out_image;
  const float* right = a.workspace + (int64_t)image * a.conv_image;
  f32x4 left_regs[kLeft], right_regs[kRight];
  auto load_tile = [&] {
#pragma unroll
    for (int i = 0; i < kLeft; ++i) {
      const uint32_t chunk = i * THREADS + tid, m = min(m_tile * BM + chunk / (BK / 4), a.m - 1);
      left_regs[i] = load4(left + (int64_t)m * a.n_rows, p0 + chunk % (BK / 4) * 4, a.n_rows);
    }
#pragma unroll
    for (int i = 0; i < kRight; ++i) {
      const uint32_t chunk = i * THREADS + tid, n = min(n_tile * BN + chunk / (BK / 4), a.n - 1);
      right_regs[i] = load4(right + (int64_t)n * a.n_rows, p0 + chunk % (BK / 4) * 4, a.n_rows);
    }
  };
  auto store_tile = [&](int buffer) {
    if (p0 + BK > a.n_rows) {
      asm volatile("");   // stays a branch: as selects it would cost every tile
#pragma unroll
      for (int i = 0; i < kLeft; ++i)
        left_regs[i] = fix4(left_regs[i], p0 + (i * THREADS + tid) % (BK / 4) * 4, a.n_rows);
#pragma unroll
      for (int i = 0; i < kRight; ++i)
        right_regs[i] = fix4(right_regs[i], p0 + (i * THREADS + tid) % (BK / 4) * 4, a.n_rows);
    }
#pragma unroll
    for (int i = 0; i < kLeft; ++i) {
      const uint32_t chunk = i * THREADS + tid;
      *reinterpret_cast<f32x4*>(&left_lds[buffer][chunk / (BK / 4) * LD + chunk % (BK / 4) * 4]) = left_regs[i];
    }
#pragma unroll
    for (int i = 0; i < kRight; ++i) {
      const uint32_t chunk = i * THREADS + tid;
      *reinterpret_cast<f32x4*>(&right_lds[buffer][chunk / (BK / 4) * LD + chunk % (BK / 4) * 4]) = right_regs[i];
    }
  };

  const uint32_t row = lane & 15, group = lane >> 4;
  const uint32_t k_half = wave / (WM * WN) * (BK / 2);
  const uint32_t wave_m = wave / WN % WM * 32, wave_n = wave % WN * 32;
  double total[2][2][4] = {};
  load_tile();
  store_tile(0);
  __syncthreads();
  int buffer = 0;
  // the 32 positions of a wave's half of a tile are summed in the operands' precision, in two
  // sums of sixteen, and the tiles in double, as the partials are
  auto multiply = [&] {
    f32x4 l4[2][2], r4[2][2], sums[2][2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int at = row * LD + k_half + c * 16 + 4 * group;
        l4[t][c] = *reinterpret_cast<const f32x4*>(&left_lds[buffer][(wave_m + t * 16) * LD + at]);
        r4[t][c] = *reinterpret_cast<const f32x4*>(&right_lds[buffer][(wave_n + t * 16) * LD + at]);
      }
#pragma unroll
    for (int tu = 0; tu <= 4; ++tu) {
      if (tu < 4) {
        auto& to = sums[tu / 2][tu % 2];
        to[0] = zero4();
        to[1] = zero4();
#pragma unroll
        for (int c = 0; c < 2; ++c) product16(l4[tu / 2][c], r4[tu % 2][c], to);
      }
      if (tu > 0) {
        const auto& from = sums[(tu - 1) / 2][(tu - 1) % 2];
        const f32x4 sum = from[0] + from[1];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          double& to = total[(tu - 1) / 2][(tu - 1) % 2][r];
          to += (double)sum[r];
          asm volatile("" : "+v"(to));   // added here, not after the next tile's stores
        }
      }
    }
  };
  for (; piece < piece_end; ++piece) {
    if (piece + 1 < piece_end) {   // else the last piece is loaded again, and not used: no load stands under a condition
      p0 += BK;
      if (p0 >= a.n_rows) {
        p0 = 0;
        left += a.out_image;
        right += a.conv_image;
      }
    }
    load_tile();
    multiply();
    store_tile(buffer ^ 1);
    __syncthreads();
    buffer ^= 1;
  }

  // 16 doubles a lane, behind the loop's last barrier
  double* shared = reinterpret_cast<double*>(&left_lds[0][0]) + (wave % (WM * WN) * 64 + lane) * 16;
  static_assert(2 * BM * LD >= WM * WN * 64 * 16 * 2, "the groups' sums fit the left operand's LDS");
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (k_half) shared[(t * 2 + u) * 4 + r] = total[t][u][r];
  __syncthreads();
  if (k_half) return;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) total[t][u][r] += shared[(t * 2 + u) * 4 + r];

  float* to = a.result + (int64_t)split * a.m * a.n;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const uint32_t n = n_tile * BN + wave_n + u * 16 + row;
    if (n >= a.n) continue;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t m = m_tile * BM + wave_m + t * 16 + 4 * group + r;
        if (m >= a.m) continue;
        float& cell = to[(int64_t)m * a.n + n];
        cell = (float)(a.alpha == 0.0 ? total[t][u][r] : a.alpha * (double)cell + total[t][u][r]);
      }
  }
}

// ------------------------------------------------------ backward-weights, three pieces to a float

// Element `chunk` (of eight positions) of row `row` of a piece in LDS, rows of 64 positions: eight consecutive rows' reads of
// one chunk cover 128 bytes' worth of banks once.
__device__ __forceinline__ uint32_t piece_at(uint32_t row, uint32_t chunk) { return row * kConvPiece + ((chunk ^ row) & 7) * 8; }

// partial[split][m][n] = sum over the split's positions of output_gradient[m][p] * unrolled[n][p]:
// both operands have the positions innermost.  The positions of every image are cut into pieces
// of kConvPiece (the last one shorter), a split takes a run of consecutive pieces: the result is
// small (64 x 576 is 9 tiles), the chip is filled by the splits.  A single split adds to the
// weight gradient itself.
// Two groups of WM x WN waves share a piece and take half of its positions each: twice the
// waves in flight for the same partials, which are added in LDS at the end.  The sums of 64 positions (two pieces) are
// float, those of a run double, as the partials are.
__global__ void __launch_bounds__(512, 2) conv_weight_gradient_split_kernel(const ConvWeightArgs a) {
  constexpr int WM = 2, WN = 2;
  constexpr int BM = 32 * WM, BN = 32 * WN, BK = kConvPiece, THREADS = 128 * WM * WN, kChunks = BK / 8;
  constexpr int UA = BM * kChunks / THREADS, UB = BN * kChunks / THREADS, U = UA + UB;   // runs of eight positions a lane stages
  constexpr int kLeft = 2 * kSplitPieces * BM * BK, kRight = 2 * kSplitPieces * BN * BK;
  __shared__ __attribute__((aligned(16))) uint16_t lds[kLeft + kRight];
  const uint32_t unit = unit_of_block(blockIdx.x, a.units);
  if (unit >= a.units) return;
  uint32_t split, tile, m_tile, n_tile;
  a.tiles_fd.divmod(unit, split, tile);
  a.n_tiles_fd.divmod(tile, m_tile, n_tile);
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t first_piece = split * a.pieces_per_split;
  const uint32_t pieces = min(first_piece + a.pieces_per_split, a.pieces) - first_piece;

  // Rows beyond the result repeat the last one and are not stored.
  auto row_of = [&](int i) { return ((i < UA ? i : i - UA) * THREADS + tid) / kChunks; };
  const uint32_t chunk = tid % kChunks;
  uint32_t row_offset[U];
#pragma unroll
  for (int i = 0; i < U; ++i)
    row_offset[i] = (i < UA ? min(m_tile * BM + row_of(i), a.m - 1) : min(n_tile * BN + row_of(i), a.n - 1)) * a.n_rows;
  // The piece that is loaded: positions [p0, p0 + BK) of an image, as far as it has them.
  uint32_t p0;
  const float* left;
  const float* right;
  auto rewind = [&] {
    uint32_t image, part;
    a.parts_fd.divmod(first_piece, image, part);
    p0 = part * BK;
    left = a.output_gradient + (int64_t)image * a.out_image;
    right = a.workspace + (int64_t)image * a.conv_image;
  };
  auto advance = [&](uint32_t piece) {   // from the piece before `piece`; beyond the last one stays there: no load stands under a condition
    if (piece >= pieces) return;
    p0 += BK;
    if (p0 >= a.n_rows) {
      p0 = 0;
      left += a.out_image;
      right += a.conv_image;
    }
  };
  f32x4 raw[2][U][2];
  auto load = [&](int i, int set) {
    const float* row = (i < UA ? left : right) + row_offset[i];
#pragma unroll
    for (int h = 0; h < 2; ++h) raw[set][i][h] = load4(row, p0 + chunk * 8 + h * 4, a.n_rows);
  };
  auto fix = [&](int i, int set, uint32_t at) {
    if (at + BK <= a.n_rows) return;
    asm volatile("");   // stays a branch: as selects it would cost every piece
#pragma unroll
    for (int h = 0; h < 2; ++h) raw[set][i][h] = fix4(raw[set][i][h], at + chunk * 8 + h * 4, a.n_rows);
  };

  const uint32_t row = lane & 31, half = lane >> 5, group = wave / (WM * WN);
  const uint32_t wave_m = wave / WN % WM * 32, wave_n = wave % WN * 32;
  double total[16] = {};
  bool found = false;
  rewind();
  {
    const SplitWeights weights;
    u32x4 split_pieces[kSplitPieces];
    auto plane = [&](int i, int buffer, int p) {
      return i < UA ? &lds[(buffer * kSplitPieces + p) * BM * BK] : &lds[kLeft + (buffer * kSplitPieces + p) * BN * BK];
    };
    auto stage = [&](int i, int h, int buffer, int set, uint32_t at) {
      if (h == 0) fix(i, set, at);
      split4(raw[set][i][h], split_pieces, 4 * h, weights);
      if (h == 0) return;
#pragma unroll
      for (int p = 0; p < kSplitPieces; ++p)
        *reinterpret_cast<u32x4*>(plane(i, buffer, p) + piece_at(row_of(i), chunk)) = split_pieces[p];
    };
    bf16x8 l[2][kSplitPieces], r[2][kSplitPieces];
    auto fetch = [&](int buffer, int part, int p) {   // positions 32 * group + 16 * part .. + 15
      l[part][p] = *reinterpret_cast<const bf16x8*>(plane(0, buffer, p) + piece_at(wave_m + row, group * 4 + part * 2 + half));
      r[part][p] = *reinterpret_cast<const bf16x8*>(plane(UA, buffer, p) + piece_at(wave_n + row, group * 4 + part * 2 + half));
    };
    f32x16 sums[2] = {zero16(), zero16()};   // the products of the leading pieces; all others
    auto multiply = [&](int part, int i) {
      f32x16& to = sums[i + 1 < kSplitProducts];
      to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l[part][kSplitLeft[i]], r[part][kSplitRight[i]], to, 0, 0, 0);
    };
    uint32_t set_p0[2];   // of the pieces in `raw`
    auto step = [&](uint32_t piece, int buffer, int set) {
#pragma unroll
      for (int i = 0; i < kSplitProducts; ++i) {
        multiply(0, i);
        if (i < kSplitPieces) fetch(buffer, 1, kSplitPieces - 1 - i);
#pragma unroll
        for (int j = i * 2 * U / kSplitProducts; j < (i + 1) * 2 * U / kSplitProducts; ++j) {
          if (j == 0) advance(piece + 3);
          stage(j / 2, j % 2, buffer ^ 1, set, set_p0[set]);
          if (j % 2) load(j / 2, set);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      set_p0[set] = p0;
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < kSplitProducts; ++i) {
        multiply(1, i);
        if (i < kSplitPieces) fetch(buffer ^ 1, 0, kSplitPieces - 1 - i);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
#pragma unroll
    for (int i = 0; i < U; ++i) load(i, 0);
    set_p0[0] = p0;
    advance(1);
    set_p0[1] = p0;
#pragma unroll
    for (int i = 0; i < U; ++i) load(i, 1);
#pragma unroll
    for (int j = 0; j < 2 * U; ++j) stage(j / 2, j % 2, 0, 0, set_p0[0]);
    advance(2);
    set_p0[0] = p0;
#pragma unroll
    for (int i = 0; i < U; ++i) load(i, 0);
    __syncthreads();
#pragma unroll
    for (int p = kSplitPieces - 1; p >= 0; --p) fetch(0, 0, p);
    for (uint32_t piece = 0; piece < pieces; piece += 2) {
      step(piece, 0, 1);
      if (piece + 1 < pieces) step(piece + 1, 1, 0);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float sum = sums[0][e] + sums[1][e];
        found |= not_finite(sum);
        total[e] += (double)sum;
      }
      sums[0] = zero16();
      sums[1] = zero16();
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) total[e] *= (double)kSplitUnscale;
  }

  if (__syncthreads_or(found)) {
    // In float: chains of eight products, added in double.
    constexpr int LD = BK + 4;
    float* left_lds = reinterpret_cast<float*>(lds);
    float* right_lds = left_lds + BM * LD;
    static_assert((BM + BN) * LD * 4 <= (kLeft + kRight) * 2, "the floats fit where their pieces were");
#pragma unroll
    for (int e = 0; e < 16; ++e) total[e] = 0.0;
    rewind();
    for (uint32_t piece = 0; piece < pieces; ++piece) {
#pragma unroll
      for (int i = 0; i < U; ++i) {
        load(i, 0);
        fix(i, 0, p0);
        float* to = (i < UA ? left_lds : right_lds) + row_of(i) * LD + chunk * 8;
        *reinterpret_cast<f32x4*>(to) = raw[0][i][0];
        *reinterpret_cast<f32x4*>(to + 4) = raw[0][i][1];
      }
      __syncthreads();
      for (int k = 0; k < BK / 2; k += 8) {
        f32x16 sum = zero16();
        const f32x4 l = *reinterpret_cast<const f32x4*>(left_lds + (wave_m + row) * LD + group * (BK / 2) + k + 4 * half);
        const f32x4 r = *reinterpret_cast<const f32x4*>(right_lds + (wave_n + row) * LD + group * (BK / 2) + k + 4 * half);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(l[e], r[e], sum, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 16; ++e) total[e] += (double)sum[e];
      }
      advance(piece + 1);
      __syncthreads();
    }
  }

  // 16 doubles a lane, behind the last barrier
  double* shared = reinterpret_cast<double*>(lds) + (wave % (WM * WN) * 64 + lane) * 16;
  static_assert((kLeft + kRight) * 2 >= WM * WN * 64 * 16 * 8, "the groups' sums fit the operands' LDS");
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 16; ++e)
    if (group) shared[e] = total[e];
  __syncthreads();
  if (group) return;
#pragma unroll
  for (int e = 0; e < 16; ++e) total[e] += shared[e];

  float* to = a.result + (int64_t)split * a.m * a.n;
  const uint32_t n = n_tile * BN + wave_n + row;
  if (n >= a.n) return;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const uint32_t m = m_tile * BM + wave_m + 8 * (e / 4) + 4 * half + e % 4;
    if (m >= a.m) continue;
    float& cell = to[(int64_t)m * a.n + n];
    cell = (float)(a.alpha == 0.0 ? total[e] : a.alpha * (double)cell + total[e]);
  }
}

template <bool kForward, int kChains>
void launch_product(hipStream_t s, const ConvProductArgs& a, int bm, dim3 grid) {
  if (bm == 32) hipLaunchKernelGGL((conv_product_kernel<32, kForward, kChains>), grid, dim3(kBlock), 0, s, a);
  else if (bm == 64) hipLaunchKernelGGL((conv_product_kernel<64, kForward, kChains>), grid, dim3(kBlock), 0, s, a);
  else hipLaunchKernelGGL((conv_product_kernel<128, kForward, kChains>), grid, dim3(kBlock), 0, s, a);
}

// What conv_data_few_kernel holds of an output gradient's position.
constexpr int64_t kFewChannels = 64;

// Rows of a tile: as few idle rows as possible, 128 before 64 where both leave the same.
int tile_rows(int64_t m) { return m <= 32 ? 32 : (m + 63) / 64 % 2 ? 64 : 128; }

}  // namespace

namespace cthip {

int64_t conv_product_units(int64_t m, int64_t n) {
  const int bm = tile_rows(m), bn = bm == 128 ? 64 : 128;
  return (m + bm - 1) / bm * ((n + bn - 1) / bn);
}

int64_t conv_product_positions(int64_t m) {
  constexpr int64_t kMostTiles = int64_t(1) << 23;
  static_assert(kMostTiles * kBlock < int64_t(1) << 32, "a launch of 2^32 lanes or more is refused");
  const int bm = tile_rows(m);
  return kMostTiles / ((m + bm - 1) / bm) * (bm == 128 ? 64 : 128);
}

void conv_product(hipStream_t s, ConvProductArgs a, bool forward) {
  const int bm = tile_rows(a.m);
  a.units = (uint32_t)conv_product_units(a.m, a.n);
  a.m_tiles_fd = FastDiv((a.m + bm - 1) / bm);
  const dim3 grid((a.units + kXcds - 1) / kXcds * kXcds);
  // Two chains of eight a tile cost the input gradient's product 4 to 6 % where it has many tiles
  // ([64, 64, 56, 56] under 64 windows of 3 x 3 206 and 195 us); a sum of few tiles needs them.
  constexpr uint32_t kFewTerms = 48;
  if (forward) launch_product<true, 2>(s, a, bm, grid);
  else if (a.k <= kFewTerms) launch_product<false, 2>(s, a, bm, grid);
  else launch_product<false, 1>(s, a, bm, grid);
}

// Forward (k cells): [98, 26, 46, 46] under 164 of 3 x 3 (k 234) 235 us with the float kernel, 179 here, [34, 30, 57, 57]
// under 106 of 5 x 5 (750) 247 and 186, [60, 9, 28, 28] under 181 (81) 29 and 24; a tile has 32 k, which fewer than 64 do not
// fill ([104, 1, 80, 80] under 54, 9 cells, 36 and 61), and blocks of 256 positions need to be enough to fill the chip
// ([20, 17, 17, 17] under 31, 23 blocks, 13 and 16): the more the shorter the sums ([67, 8, 71, 71] under 19 at stride 2, k
// 72, 321 blocks, 15.2 and 17.5; from 384 on 0.84 to 1.0 of the float kernel's time).  Of more than 32 rows two blocks share a
// unit, and short sums are over before a last round of few blocks is ([115, 73, 26, 26] under 104 of 1 x 1, k 73, 602 blocks,
// 25 and 29; 12 of 14 such shapes of 513 to 640 blocks and up to 112 cells 0.96 to 1.14).  Sums of 64 to 80 cells under 1 x 1
// windows over 700 to 1600 blocks of full tiles take longer too (64 cells 1.07 to 1.18, [16, 64, 56, 56] under 256 27 and
// 30.5; 80 up to 1.1; 88 and more 0.84 to 1.05) and stay here for their errors, two thirds of the float kernel's.
// Input gradient (k out channels): with many of them the general split kernel throughout ([32, 256, 14, 14] under 256 103
// and 85, [134, 94, 15, 15] under 145 122 and 107; of 65 to 80, a third tile mostly idle, 0.96 to 1.08 of the float kernel's
// time); with up to 64 the kernel that keeps them in registers where the rows pay for that and the positions fill the chip
// ([64, 64, 56, 56] under 64, 576 rows, 214 and 124, without the roll back; [40, 8, 103, 103] under 33 of 1 x 1, 8 rows, 32
// and 43; [174, 172, 26, 26] under 36 of 1 x 1 at stride 2, 29406 positions, 63 and 68).  Beyond 32 channels it holds 64, and
// takes more than the float kernel over small workspaces (with the roll back: k 41 to 64, 20 to 33 MB 1.07 to 1.2 times as long
// in 13 shapes of 14, 43 MB and more 0.82 to 1.05; k 33 to 40, up to 70 MB 0.98 to 1.15, mostly above 1, 73 MB and more
// 0.91 to 1.02).
bool conv_product_splits(int64_t m, int64_t n, int64_t k, bool forward) {
  if (forward) {
    constexpr int64_t kFewCells = 64, kShortSums = 96, kShortRounds = 112, kFewBlocks = 288, kFullChip = 384, kFullUnits = 512,
                      kMostUneven = 640;
    const int64_t blocks = (m + 63) / 64 * ((n + kPositions - 1) / kPositions);
    const bool uneven = m > 32 && blocks > kFullUnits && blocks <= kMostUneven;
    return k >= kFewCells && blocks >= (k <= kShortSums ? kFullChip : kFewBlocks) && !(k <= kShortRounds && uneven);
  }
  constexpr int64_t kFewRows = 32;   // [104, 1, 50, 50] under 105 of 5 x 5, 25 rows, 37 and 43
  if (k > kFewChannels) return m > kFewRows;
  constexpr int64_t kLeastChannels = 20, kLeastRows = 128, kManyRows = 512, kLeastPositions = 8192, kManyPositions = 65536;
  if (k < kLeastChannels || m < kLeastRows || n < (m >= kManyRows ? kLeastPositions : kManyPositions)) return false;
  constexpr int64_t kHalfOfThem = 32, kMostIdle = 40, kLeastCells = int64_t(10) << 20, kManyCells = int64_t(18) << 20;
  return k <= kHalfOfThem || m * n >= (k <= kMostIdle ? kManyCells : kLeastCells);
}

int64_t conv_split_positions(int64_t m) {
  constexpr int64_t kMostTiles = int64_t(1) << 22;   // of 32 rows and 128 positions, the smallest
  static_assert(kMostTiles * 512 < int64_t(1) << 32, "a launch of 2^32 lanes or more is refused");
  return kMostTiles / ((m + 31) / 32) * 128;
}

// Where the rows of the workspace begin on whole sectors of 64 bytes; others are written to memory in parts, each read first.
// Input gradients then lose ([132, 125, 41, 41] under 22 of 3 x 3, 1521 positions a row, us: 510, past the caches 862), and so
// they do at a stride, where the roll back skips about in the workspace and needs the caches ([109, 41, 80, 80] under 60 of
// 5 x 5 at stride 2: 486 and 641).  Forward passes of 32 rows and more have products enough to hide it: 46 shapes 1.01 to
// 1.41 times as long through the caches ([209, 12, 57, 57] under 51 of 3 x 3, 3249 positions, 116 and 164; [63, 15, 101, 101]
// under 58 135 and 189), but for windows of one cell, whose stores follow each other as fast as they can ([88, 90, 102, 102]
// under 43 201 and 185).  Of fewer rows it is 50 shapes of 0.83 to 1.07 ([65, 27, 63, 63] under 17 of 5 x 5, 3481: 278 and
// 235), but 1.06 to 1.29 in nine where the rows begin on 16 bytes and the gathers take longest, at a stride, or the sums are
// short ([68, 57, 102, 102] under 25 of 3 x 3 at stride 2, 2500: 143 and 185; [164, 8, 88, 88] under 5 of 3 x 3, 7396: 116 and
// 134).
static bool past_the_caches(const ConvProductArgs& a, bool forward) {
  constexpr uint32_t kSector = 16, kPiece = 4, kFullTile = 32, kShortSums = 192;
  if ((int64_t)a.images * a.conv_image * (int64_t)sizeof(float) <= kLastLevelCache) return false;
  const bool whole = a.n_rows % kSector == 0 && reinterpret_cast<uintptr_t>(a.workspace) % (kSector * sizeof(float)) == 0;
  const bool strided = a.sx != 1 || a.sy != 1;
  if (!forward) return whole && !strided;
  if (whole) return true;
  if (a.kw * a.kh == 1) return false;
  return a.m >= kFullTile || (a.n_rows % kPiece == 0 && (strided || a.k <= kShortSums));
}

void conv_product_split(hipStream_t s, ConvProductArgs a, bool forward) {
  const auto grid = [&](uint32_t m_tiles, uint32_t positions) {
    a.units = m_tiles * ((a.n + positions - 1) / positions);
    a.m_tiles_fd = FastDiv(m_tiles);
    return dim3((a.units + kXcds - 1) / kXcds * kXcds);
  };
  const dim3 block(kPositions);
  const bool past = past_the_caches(a, forward);
  if (forward) {
    const uint32_t bm = a.m <= 32 ? 32 : 64;
    const dim3 blocks = grid((a.m + bm - 1) / bm, kPositions);
    if (bm == 32 && past) hipLaunchKernelGGL((conv_forward_kernel<1, true>), blocks, block, 0, s, a);
    else if (bm == 32) hipLaunchKernelGGL((conv_forward_kernel<1, false>), blocks, block, 0, s, a);
    else if (past) hipLaunchKernelGGL((conv_forward_kernel<2, true>), blocks, block, 0, s, a);
    else hipLaunchKernelGGL((conv_forward_kernel<2, false>), blocks, block, 0, s, a);
  } else if (a.k <= kFewChannels) {
    // rows enough to a block to pay for its positions' fragments, blocks enough to fill the chip
    constexpr uint32_t kFullChip = 1024;
    const uint32_t row_tiles = (a.m + 31) / 32, n_tiles = (a.n + kPositions - 1) / kPositions;
    const uint32_t parts = std::min(row_tiles, std::max(1u, (kFullChip + n_tiles - 1) / n_tiles));
    const uint32_t tiles = (row_tiles + parts - 1) / parts;
    a.rows_per_block = tiles * 32;
    const dim3 blocks = grid((row_tiles + tiles - 1) / tiles, kPositions);
    if (a.k <= 32 && past) hipLaunchKernelGGL((conv_data_few_kernel<2, true>), blocks, block, 0, s, a);
    else if (a.k <= 32) hipLaunchKernelGGL((conv_data_few_kernel<2, false>), blocks, block, 0, s, a);
    else if (past) hipLaunchKernelGGL((conv_data_few_kernel<4, true>), blocks, block, 0, s, a);
    else hipLaunchKernelGGL((conv_data_few_kernel<4, false>), blocks, block, 0, s, a);
  } else {
    const int bm = tile_rows(a.m);   // more than 32 rows: 64 or 128
    const dim3 blocks = grid((a.m + bm - 1) / bm, 128);
    if (bm == 64) hipLaunchKernelGGL((conv_data_kernel<64>), blocks, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((conv_data_kernel<128>), blocks, dim3(512), 0, s, a);
  }
}

int64_t conv_weight_tiles(int64_t m, int64_t n) {
  return (m <= 32 ? 1 : (m + 63) / 64) * (n <= 32 ? 1 : (n + 63) / 64);
}

int64_t conv_weight_waves(int64_t m, int64_t n) { return (m <= 32 ? 1 : 2) * (n <= 32 ? 1 : 2) * 2; }

void conv_weight_gradient(hipStream_t s, ConvWeightArgs a, int64_t splits) {
  const bool narrow_m = a.m <= 32, narrow_n = a.n <= 32;
  const uint32_t m_tiles = (a.m + (narrow_m ? 31 : 63)) / (narrow_m ? 32 : 64);
  const uint32_t n_tiles = (a.n + (narrow_n ? 31 : 63)) / (narrow_n ? 32 : 64);
  a.tiles_fd = FastDiv(m_tiles * n_tiles);
  a.n_tiles_fd = FastDiv(n_tiles);
  a.units = m_tiles * n_tiles * (uint32_t)splits;
  const dim3 grid((a.units + kXcds - 1) / kXcds * kXcds);
  // A block of the split kernel begins later (three pieces loaded, one split, before its first product) and takes less for
  // a piece: runs of 7 pieces [1, 64, 56, 56] under 64 of 3 x 3 18.5 -> 16.1 us, of 56 [64, 64, 56, 56] 198 -> 163; of 3
  // [74, 13, 19, 19] under 186 of 5 x 5 at stride 2 21.7 -> 23.9, of 1 [8, 256, 7, 7] under 256 22.3 -> 24.9.  Of its narrow forms
  // the few waves split as long as they multiply ([7, 7, 64, 64] under 32 of 1 x 1 11.6 -> 13.9).
  constexpr uint32_t kLongRun = 6;
  if (!narrow_m && !narrow_n && a.pieces_per_split >= kLongRun)
    hipLaunchKernelGGL(conv_weight_gradient_split_kernel, grid, dim3(512), 0, s, a);
  else if (narrow_m && narrow_n) hipLaunchKernelGGL((conv_weight_gradient_kernel<1, 1>), grid, dim3(128), 0, s, a);
  else if (narrow_m) hipLaunchKernelGGL((conv_weight_gradient_kernel<1, 2>), grid, dim3(256), 0, s, a);
  else if (narrow_n) hipLaunchKernelGGL((conv_weight_gradient_kernel<2, 1>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((conv_weight_gradient_kernel<2, 2>), grid, dim3(512), 0, s, a);
}

}  // namespace cthip
