"""The addresses of the forward convolution's gathers (csrc/conv_gather.h), on the host: every window over images of few rows."""
import pathlib
import subprocess

ROOT = pathlib.Path(__file__).resolve().parent.parent

PROGRAM = r"""
#include "conv_gather.h"
#include <cstdio>
#include <initializer_list>
using namespace cthip;

int main() {
  long taps = 0, clamped = 0;
  for (int in_h = 1; in_h <= 4; ++in_h) for (int in_w : {1, 2, 3, 7}) for (int kh = 1; kh <= 5; ++kh) for (int kw = 1; kw <= 5; ++kw)
  for (int py = 0; py <= 2; ++py) for (int px = 0; px <= 2; ++px) for (int stride = 1; stride <= 2; ++stride)
  for (uint32_t images = 1; images <= 2; ++images) for (uint32_t channels = 1; channels <= 2; ++channels) {
    const int span_h = in_h + 2 * py - kh, span_w = in_w + 2 * px - kw;
    if (span_h < 0 || span_w < 0) continue;
    const uint32_t plane = in_h * in_w, in_image = channels * plane, padding = gather_padding(in_w, px, py);
    const uint32_t length = gather_length(images, in_image, padding);
    for (uint32_t image = 0; image < images; ++image)
    for (int oy = 0; oy <= span_h / stride; ++oy) for (int ox = 0; ox <= span_w / stride; ++ox) {
      const int iy0 = oy * stride - py, ix0 = ox * stride - px;
      const uint32_t from = gather_window(image, in_image, in_w, padding, iy0, ix0);
      for (uint32_t c = 0; c < channels; ++c) for (int ky = 0; ky < kh; ++ky) for (int kx = 0; kx < kw; ++kx) {
        const int iy = iy0 + ky, ix = ix0 + kx;
        const bool inside = iy >= 0 && iy < in_h && ix >= 0 && ix < in_w;
        const uint32_t tap = gather_tap(c, ky, kx, plane, in_w, length);
        const bool right = !inside || (from < length && from + tap == padding + image * in_image + c * plane + iy * in_w + ix);
        if (tap > length || !right) {
          printf("image %dx%d of %u, channel %u, window %dx%d, padding %d,%d, stride %d, at %d,%d, tap %d,%d: %u of %u\n", in_h, in_w,
                 images, c, kh, kw, py, px, stride, oy, ox, ky, kx, tap, length);
          return 1;
        }
        ++taps;
        clamped += c * plane + ky * in_w + kx > length;
      }
    }
  }
  printf("%ld taps, %ld of them beyond\n", taps, clamped);
  return clamped == 0;
}
"""


def test_no_tap_lies_beyond_the_buffer(tmp_path):
    """Taps of an image are where they should be, and no scalar offset exceeds the buffer's length: also those of single images
    under windows that reach below them, which are there."""
    (tmp_path / "gather.cpp").write_text(PROGRAM)
    exe = tmp_path / "gather"
    res = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", f"-I{ROOT / 'cortex_amd' / 'csrc'}", str(tmp_path / "gather.cpp"),
                          "-o", str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout
