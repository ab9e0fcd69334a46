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


@pytest.mark.parametrize("code,k,side,planes", [
    (capi.F64, 3, 511, 32), (capi.F64, 3, 511, 33), (capi.F32, 3, 78, 4308), (capi.F32, 3, 78, 4309),
    (capi.F32, 2, 62, 3273), (capi.F32, 2, 62, 3274), (capi.F32, 2, 511, 100), (capi.F32, 2, 511, 101),
    (capi.F64, 2, 510, 50), (capi.F64, 2, 510, 51),
], ids=lambda v: str(v))
def test_rows_off_the_16_byte_grid(P, code, k, side, planes):
    """Both sides of the sizes from which such rows take the general form: 64, 100, 48 and 100 MiB of gradient; and 100 for
    rows on the grid in double under 2 x 2 windows."""
    out_side = (side - k) // 2 + 1
    rng = np.random.default_rng(planes)
    n_in, n_out = planes * side * side, planes * out_side * out_side
    ints = lambda n: rng.integers(-3, 4, n).astype(NP[code])
    inp, out, og, ig = P.buf(ints(n_in)), P.buf(np.zeros(n_out, NP[code])), P.buf(ints(n_out)), P.buf(ints(n_in))
    geometry = (H.pool_desc(k, k, 0, 0, 2, 2, "max"), 1, planes, side, side, out_side, out_side)
    P.run(H.pooling_forward, View(out, [n_out]), View(inp, [n_in]), *geometry)
    kernel = P.run(H.pooling_backward, View(ig, [n_in]), View(inp, [n_in]), View(out, [n_out]), View(og, [n_out]), *geometry)
    limit = 64 if code == capi.F64 and k == 3 else 48 if (k, side) == (2, 62) else 100
    assert kernel == ("pool_backward_stride2" if n_in * NP[code]().itemsize >> 20 < limit else "pool_backward_band"), kernel
    H.assert_bit_exact(ig.download(), ig.host, f"{planes} planes of {side} x {side}")
