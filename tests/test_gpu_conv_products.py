"""The convolution kernels where their splits and tiles can go wrong, against the CPU oracle."""
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


def vec(buf):
    return View(buf, [buf.init.size])


@pytest.mark.parametrize("code", [capi.F32, capi.F64], ids=["float", "double"])
@pytest.mark.parametrize("batch", [7, 8, 9, 23])     # below, at and off the number of slices that share an element
def test_weight_gradient_over_many_images(P, code, batch):
    """Whole numbers: every product and sum is exact, in any order, so the gradient agrees to the bit."""
    rng = np.random.default_rng(batch)
    cin, cout, h, w, k = 3, 5, 6, 7, 3
    desc, n_rows, n_cols = H.conv_desc(cin, cout, k, k, 1, 1, 1, 1), h * w, cin * k * k
    ints = lambda n: rng.integers(-4, 5, n).astype(NP[code])
    inp, weights, og = P.buf(ints(batch * cin * h * w)), P.buf(ints(cout * n_cols)), P.buf(ints(batch * cout * n_rows))
    out, work = P.buf(ints(batch * cout * n_rows)), P.buf(ints(batch * n_rows * n_cols))
    wg = P.buf(ints(cout * n_cols))
    P.run(H.convolution, "forward", vec(out), 0.0, vec(inp), vec(weights), vec(work), desc, batch, h, w, h, w)
    H.assert_bit_exact(out.download(), out.host, "convolution-forward")
    for alpha in (0.0, 2.0):
        P.run(H.convolution, "backward_weights", vec(wg), alpha, vec(og), vec(inp), vec(work), desc, batch, h, w, h, w)
        H.assert_bit_exact(wg.download(), wg.host, f"convolution-backward-weights, alpha {alpha}")
