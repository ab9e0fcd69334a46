// conv_gather.h -- where conv_forward_kernel's gathers read, in floats of a buffer that begins with the first row and column
// of the padding in front of the first image.  Plain C++ outside of hipcc: a host program checks the arithmetic.
#pragma once

#include <cstdint>

#ifndef CT_HD
#define CT_HD inline
#endif

namespace cthip {

CT_HD uint32_t gather_padding(uint32_t in_w, int32_t px, int32_t py) { return (uint32_t)py * in_w + (uint32_t)px; }

CT_HD uint32_t gather_length(uint32_t images, uint32_t in_image, uint32_t padding) { return images * in_image + padding; }

// The first cell of the window whose corner is (iy0, ix0), which may lie in the padding.
CT_HD uint32_t gather_window(uint32_t image, uint32_t in_image, uint32_t in_w, uint32_t padding, int32_t iy0, int32_t ix0) {
  return image * in_image + padding + (uint32_t)iy0 * in_w + (uint32_t)ix0;
}

// From there to a tap.  The scalar part of a buffer address is taken off the buffer's length and must not exceed it.  A tap
// that lies in some image does not (its window begins at zero or later); one that does, the lowest rows of a window that is
// taller than a single image and the padding above it, lies in the padding at every position, and is not read wherever the
// lane's part sends it.
CT_HD uint32_t gather_tap(uint32_t channel, uint32_t ky, uint32_t kx, uint32_t in_plane, uint32_t in_w, uint32_t length) {
  const uint32_t cell = channel * in_plane + ky * in_w + kx;
  return cell < length ? cell : length;
}

}  // namespace cthip
