// conv_products.h -- what ops_conv.hip hands to the matrix-core products of ops_conv_mfma.hip.
#pragma once

#include "common.h"

namespace cthip {

// The cells of a window that the products keep a mask of.
constexpr int kConvMaskTaps = 32;

// forward:       output[m][j]    = sum over k of weights[m][k] * unrolled[k][j] (+ beta * output[m][j]),
//                                  the unrolled input written to the workspace; m out channels, k cells
// backward-data: workspace[m][j] = sum over k of weights[k][m] * output[k][j]; m cells, k out channels
// over the n positions j of all images, numbered on.
struct ConvProductArgs {
  const float* weights;
  const float* input;
  float* output;
  float* workspace;
  int64_t in_image, out_image, conv_image;
  uint32_t m, n, k, n_rows, images;   // n = images * n_rows
  uint32_t in_plane, in_h, in_w, kw, kh;
  int32_t px, py, sx, sy;
  float beta;
  uint32_t units, rows_per_block;
  FastDiv m_tiles_fd, rows_fd, out_w_fd, taps_fd, kw_fd;
};
void conv_product(hipStream_t s, ConvProductArgs a, bool forward);
// The tiles that such a product has, and the positions that one launch of it may have.
int64_t conv_product_units(int64_t m, int64_t n);
int64_t conv_product_positions(int64_t m);

// The same on the bfloat16 matrix cores, and whether a product is faster there (n positions in all); a launch may have so
// many positions, and its buffers must stay below 2^31 bytes, the input's with the padding in front of its first image.
bool conv_product_splits(int64_t m, int64_t n, int64_t k, bool forward);
int64_t conv_split_positions(int64_t m);
void conv_product_split(hipStream_t s, ConvProductArgs a, bool forward);

// The positions of a piece, the unit in which the weight gradient's sum is split.
constexpr int kConvPiece = 64;

// result[split][m][n] = alpha * result[split][m][n] + sum over the split's positions of
//                       output_gradient[m][p] * unrolled[n][p]
struct ConvWeightArgs {
  const float* output_gradient;
  const float* workspace;
  float* result;                       // the weight gradient of a single split, else partial sums
  double alpha;
  int64_t out_image, conv_image;
  uint32_t m, n, n_rows;
  uint32_t pieces, pieces_per_split;   // of all images; of a split
  uint32_t units;
  FastDiv parts_fd, tiles_fd, n_tiles_fd;   // parts: pieces of one image
};
void conv_weight_gradient(hipStream_t s, ConvWeightArgs a, int64_t splits);
int64_t conv_weight_tiles(int64_t m, int64_t n);   // blocks to a split
int64_t conv_weight_waves(int64_t m, int64_t n);   // waves to a block

}  // namespace cthip
