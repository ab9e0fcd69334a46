"""pooling-backward! of the maximum at stride 2 under 2 x 2 and 3 x 3 windows, to the bit against the CPU oracle, where
a row's 16-byte pieces, the parity of the padding and the windows at the edges can go wrong."""
import numpy as np
import pytest

import harness as H
from cortex_amd import capi
from harness import View

pytestmark = pytest.mark.gpu
NP = H.NP_DTYPES


@pytest.fixture()
def P(pair_factory):
    with pair_factory() as pair:
        yield pair


@pytest.mark.parametrize("code", [capi.F32, capi.F64], ids=["float", "double"])
@pytest.mark.parametrize("k,px,py", [(2, 0, 0), (2, 1, 1), (2, 1, 0), (3, 0, 0), (3, 1, 1), (3, 0, 1), (3, 2, 2)])
def test_max_gradient(P, code, k, px, py):
    rng = np.random.default_rng(10 * k + 3 * px + py)
    # widths around one and several pieces, one plane and several to a block, planes beyond a block's LDS (bands)
    for planes, h, w in ((3, 3, 3), (5, 4, 4), (2, 5, 5), (7, 6, 7), (2, 7, 8), (9, 8, 9), (40, 11, 13), (2, 113, 71),
                         (2, 100, 130)):
        for up in (0, 1):       # floor, and ceil: the last windows reach beyond the padded input
            oh, ow = ((n + 2 * p - k + up) // 2 + 1 for n, p in ((h, py), (w, px)))
            if min(oh, ow) < 1:
                continue
            n_in, n_out = planes * h * w, planes * oh * ow
            # few values: ties decide which inputs the gradient reaches
            x = rng.integers(-3, 4, n_in).astype(NP[code])
            x[rng.integers(0, n_in, 2)] = [np.nan, -0.0]
            inp, out = P.buf(x), P.buf(np.zeros(n_out, NP[code]))
            og, ig = (P.buf(rng.standard_normal(n).astype(NP[code])) for n in (n_out, n_in))
            geometry = (H.pool_desc(k, k, px, py, 2, 2, "max"), 1, planes, h, w, oh, ow)
            P.run(H.pooling_forward, View(out, [n_out]), View(inp, [n_in]), *geometry)
            kernel = P.run(H.pooling_backward, View(ig, [n_in]), View(inp, [n_in]), View(out, [n_out]), View(og, [n_out]),
                           *geometry)
            tiles2 = k == 2 and px == py == 0 and (h, w) == (2 * oh, 2 * ow) and w % 4 == 0
            general = code == capi.F64 and k == 2 and w % 2 == 1
            assert kernel == ("pool_backward_tile2" if tiles2 else
                              "pool_backward_band" if general else "pool_backward_stride2"), (kernel, h, w)
            H.assert_bit_exact(ig.download(), ig.host, f"{planes} planes of {h} x {w}, ceil {up}")


def test_wide_planes_of_odd_width_in_double(P):
    """Planes of an odd width whose rows are off the 16-byte grid every other time: the general form from 2^24 elements on
    under 3 x 3 windows, and under 2 x 2 always."""
    k, side = 3, 511
    out_side = (side - k) // 2 + 1
    rng = np.random.default_rng(1)
    for planes, name in ((64, "pool_backward_stride2"), (65, "pool_backward_band")):
        n_in, n_out = planes * side * side, planes * out_side * out_side
        inp, out = P.buf(rng.integers(-3, 4, n_in).astype(np.float64)), P.buf(np.zeros(n_out))
        og, ig = P.buf(rng.integers(-3, 4, n_out).astype(np.float64)), P.buf(rng.integers(-3, 4, n_in).astype(np.float64))
        geometry = (H.pool_desc(k, k, 0, 0, 2, 2, "max"), 1, planes, side, side, out_side, out_side)
        P.run(H.pooling_forward, View(out, [n_out]), View(inp, [n_in]), *geometry)
        kernel = P.run(H.pooling_backward, View(ig, [n_in]), View(inp, [n_in]), View(out, [n_out]), View(og, [n_out]), *geometry)
        assert kernel == name, (kernel, planes)
        H.assert_bit_exact(ig.download(), ig.host, f"{planes} planes of {side} x {side}")
