// ops_conv_mfma.hip -- the three float products of a convolution on the matrix cores
// (v_mfma_f32_16x16x4: the tensors' own 32 bits throughout, 157 TFLOP/s dense).
//
// What bounds them.  For 64 images of 64 x 56 x 56 under 64 windows of 3 x 3 a product is
// 14.8 GFLOP (94 us of matrix cores) around an unrolled matrix of 462 MB (75 us of HBM), so
// a product and the movement of that matrix have to overlap; the library's batched products
// ran at 62 to 94 TFLOP/s with the unrolling as a pass of its own before them.  Measured with the
// library's products and with these, one method called over and over: forward 264 -> 235 us, weight
// gradient 220 -> 178 (its sum over the splits, 5, included), input gradient with the roll back of
// 110 340 -> 317; [128, 16, 28, 28] under 32 windows 33 -> 27, 67 -> 31, 36 -> 35.  Other shapes go
// either way, and the rules of ops_conv.hip draw the lines: over 286 shapes the forward passes take
// 0.3 to 1.1 of the library's time where the call is longer than 20 us, the weight gradients 0.3 to
// 1.3 (above 1.1 only up to 26 us), the input gradients 0.24 to 1.23; shorter kernels up to 2.6, for
// calls that take the host less.  What is left is latency: 3.3 to 3.8 waves a SIMD are resident, and
// the matrix cores of a compute unit are busy for 51 (forward), 60 (weight gradient) and 54 % (input
// gradient) of the time that it is.
//
// Tiles.  A block of four waves owns BM x BN of the result.  Both operands lie in LDS as
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
// Rounding.  The matrix cores round after every product, so the error of a sum grows with the length
// of the chain.  Products are summed in chains of eight (input gradient over more than 48 channels:
// sixteen, eight in the last tile; weight gradient: sixteen, then in double), and these are added up.
// The additions are vector instructions that run while the next products do: chains of 128 took the
// same time.  Error against 64 bits, in units of the library's, geometric means and ranges over 280
// shapes: outputs 0.87 (0.40 to 1.10), input gradients 0.80 (0.33 to 1.04), weight gradients 0.45
// (0.07 to 1.08); those above 1.04 at errors of 3e-8 to 7e-8.  Chains of 128: up to 1.5, 1.3 and 1.6.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "conv_products.h"

using namespace cthip;

namespace {

constexpr int kBlock = 256;
typedef float f32x4 __attribute__((ext_vector_type(4)));

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

template <bool kForward, int kChains>
void launch_product(hipStream_t s, const ConvProductArgs& a, int bm, dim3 grid) {
  if (bm == 32) hipLaunchKernelGGL((conv_product_kernel<32, kForward, kChains>), grid, dim3(kBlock), 0, s, a);
  else if (bm == 64) hipLaunchKernelGGL((conv_product_kernel<64, kForward, kChains>), grid, dim3(kBlock), 0, s, a);
  else hipLaunchKernelGGL((conv_product_kernel<128, kForward, kChains>), grid, dim3(kBlock), 0, s, a);
}

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
  if (narrow_m && narrow_n) hipLaunchKernelGGL((conv_weight_gradient_kernel<1, 1>), grid, dim3(128), 0, s, a);
  else if (narrow_m) hipLaunchKernelGGL((conv_weight_gradient_kernel<1, 2>), grid, dim3(256), 0, s, a);
  else if (narrow_n) hipLaunchKernelGGL((conv_weight_gradient_kernel<2, 1>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((conv_weight_gradient_kernel<2, 2>), grid, dim3(512), 0, s, a);
}

}  // namespace cthip
