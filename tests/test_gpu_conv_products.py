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


# (batch, in channels, out channels, height, width, kernel width, kernel height, pad, stride): the edges of the tiles
# (32, 64 and 128 rows, 128 and 64 columns, 16 k, 64 positions of a piece), of a run of sums (128 k), of the mask of taps
# (32), of the rows (4 positions, 4 cells) and of the routes
PRODUCT_CASES = [
    (1, 1, 1, 2, 2, 1, 1, 0, 1),        # 4 positions, 1 cell: the product is the library's
    (1, 1, 3, 1, 3, 1, 1, 0, 1),        # 3 positions
    (3, 4, 2, 2, 2, 1, 1, 0, 1),        # 4 positions, 4 cells
    (2, 5, 31, 7, 9, 3, 1, 0, 1),       # 15 cells, 49 positions of odd alignment
    (2, 16, 32, 8, 8, 1, 1, 0, 1),      # exactly one tile of k, one piece of positions
    (1, 17, 33, 5, 13, 1, 1, 0, 1),     # one more of each: 17 cells, 65 positions, 33 rows
    (1, 7, 64, 9, 7, 3, 3, 1, 1),       # 63 positions and cells
    (5, 3, 65, 11, 10, 3, 3, 1, 2),     # 65 rows, strided, 30 positions
    (2, 14, 130, 9, 8, 3, 3, 1, 1),     # 126 cells: one run; 130 rows in tiles of 64
    (2, 15, 128, 9, 15, 3, 3, 0, 1),    # 135 cells: two runs; tiles of 128 rows
    (1, 21, 9, 6, 6, 3, 3, 1, 1),       # 189 cells: the last short chain
    (1, 22, 9, 6, 6, 3, 3, 1, 1),       # 198 cells, few tiles: the library
    (2, 3, 200, 5, 5, 3, 3, 1, 1),      # the same for backward-data, over 200 out channels
    (1, 2, 4, 27, 19, 5, 5, 2, 1),      # 25 taps, 513 positions: two pieces
    (1, 2, 4, 13, 12, 6, 6, 2, 1),      # 36 taps: no mask
    (64, 23, 6, 40, 40, 3, 3, 1, 1),    # 800 tiles over 207 cells
]


def weight_route(batch, m, n, n_rows):
    """The kernels of the weight gradient of [m, n] over n_rows positions an image."""
    pieces, products = batch * -(-n_rows // 64), max(1, min(64, n_rows // 4096))
    fit = max(batch * products, (1 << 20) // (4 * m * n))
    tiles = (1 if m <= 32 else -(-m // 64)) * (1 if n <= 32 else -(-n // 64))
    want = 1 if pieces <= 3 else max(1, min(512 // tiles, fit, pieces))
    run = -(-pieces // want)
    splits = -(-pieces // run)
    waves = tiles * splits * 2 * (1 if m <= 32 else 2) * (1 if n <= 32 else 2)
    narrow = m <= 32 or n <= 32
    if n_rows < 4 or (n_rows > 128 and run > 1 and tiles // (2 if narrow else 1) > 64):
        return "gemm+conv_sum_partials"
    if n_rows > 400 and (waves < 1400 or (narrow or n_rows % 4) and n_rows > 2048) and run > max(4, n_rows // 200):
        return "gemm+conv_sum_partials"
    return "conv_weight_gradient" + ("+conv_sum_partials" if splits > 1 else "")


def tiles_of(m, n):
    rows = 32 if m <= 32 else 64 if -(-m // 64) % 2 else 128
    return -(-m // rows) * -(-n // (64 if rows == 128 else 128))


def forward_route(batch, m, k, n_rows, taps):
    """The kernels of an output of m channels over k cells."""
    tiles = tiles_of(m, batch * n_rows)
    ours = k <= 192 or (tiles >= 768 and (k < 576 or m < 128))
    return "conv_product" if ours and k >= 4 and taps <= 32 else "conv_unroll+gemm"


def data_route(batch, m, k, n_rows):
    """The kernels of the input gradient of m cells over k out channels."""
    n = batch * n_rows
    tiles = tiles_of(m, n)
    if k <= 64 or (k <= 160 and tiles < 256):
        ours = True
    elif m >= 192 and (500 if k <= 256 or m >= 3000 else 1000) <= n_rows <= 4096:
        ours = False
    else:
        ours = tiles >= (400 if m <= 96 else 768) or (n_rows <= 128 and tiles >= 250)
    return "conv_product+conv_roll" if ours else "gemm+conv_roll"


# The same for the weight gradient's routes and splits
WEIGHT_CASES = [
    (2, 128, 250, 9, 8, 3, 3, 1, 1),    # 72 tiles, two splits of two pieces, 72 positions
    (2, 128, 250, 9, 15, 3, 3, 1, 1),   # 72 tiles, two splits of three pieces, 135 positions: the library
    (1, 128, 250, 7, 7, 3, 3, 1, 1),    # 72 tiles, one piece
    (1, 406, 520, 5, 5, 3, 3, 1, 1),    # 522 tiles, one piece
    (3, 2, 5, 8, 8, 3, 3, 1, 1),        # three pieces: one split
    (4, 2, 5, 8, 8, 3, 3, 1, 1),        # four of them: four splits
    (1, 20, 64, 13, 13, 3, 3, 1, 1),    # three pieces of one image, the last one of 41 positions
    (3, 64, 64, 40, 40, 3, 3, 1, 1),    # seven splits of eleven pieces: the library
    (2, 60, 3, 48, 48, 3, 3, 1, 1),     # 36 splits of two pieces of images of 2304 positions, few rows
    (5, 200, 3, 48, 48, 3, 3, 1, 1),    # the same with fourteen: the library
    (4, 16, 10, 60, 60, 3, 3, 1, 1),    # four of 3600
    (200, 5, 40, 46, 46, 3, 3, 1, 1),   # 200 splits of 34 pieces of images of 2116 positions
    (200, 5, 40, 47, 47, 3, 3, 1, 1),   # of 2209, off the 16-byte grid: the library
    (1, 64, 64, 56, 56, 3, 3, 1, 1),    # seven splits of seven pieces of one image
    (6, 200, 128, 11, 9, 1, 1, 0, 1),   # six splits of two pieces, an image each
    (7, 160, 128, 11, 9, 3, 3, 1, 1),   # seven partial products of 46 tiles
]

# The same for the output's routes
FORWARD_CASES = [
    (62, 64, 6, 40, 40, 3, 3, 1, 1),    # 576 cells over 775 tiles, few out channels
    (32, 63, 128, 39, 40, 3, 3, 1, 1),  # 567 cells over 780 tiles
    (32, 64, 128, 39, 40, 3, 3, 1, 1),  # 576 cells: the library
]

# The same for the input gradient's routes
DATA_CASES = [
    (2, 3, 160, 5, 5, 3, 3, 1, 1),      # one tile over 160 out channels
    (2, 3, 161, 5, 5, 3, 3, 1, 1),      # over 161: the library
    (1, 2, 5, 12, 11, 8, 5, 2, 1),      # 40 taps
    (70, 6, 64, 26, 26, 3, 3, 1, 1),    # 370 tiles over 64 out channels
    (70, 6, 65, 26, 26, 3, 3, 1, 1),    # over 65: the library
    (48, 11, 65, 26, 26, 3, 3, 1, 1),   # 507 tiles of 99 cells: the library
    (40, 9, 65, 36, 36, 3, 3, 1, 1),    # 810 tiles over 65 out channels
    (41, 5, 65, 35, 36, 3, 3, 1, 1),    # 404 tiles of 45 cells
    (31, 112, 70, 8, 8, 3, 3, 1, 1),    # 248 tiles over 70 out channels
    (32, 112, 70, 8, 8, 3, 3, 1, 1),    # 256, images of 64 positions
    (32, 112, 70, 12, 11, 3, 3, 1, 1),  # 528, of 132: the library
    (17, 25, 65, 25, 24, 3, 3, 1, 1),   # 225 cells, 600 positions: the library
    (26, 22, 260, 27, 37, 3, 3, 1, 1),  # 782 tiles of 198 cells over 260 out channels, 999 positions
    (26, 22, 260, 25, 40, 3, 3, 1, 1),  # of 1000: the library
    (5, 333, 260, 25, 20, 3, 3, 1, 1),  # 940 tiles of 2997 cells, 500 positions
    (5, 334, 260, 25, 20, 3, 3, 1, 1),  # of 3006: the library
]


@pytest.mark.parametrize("case", PRODUCT_CASES + WEIGHT_CASES + FORWARD_CASES + DATA_CASES, ids=lambda c: "x".join(map(str, c)))
def test_products_at_the_edges_of_their_tiles(P, case):
    batch, cin, cout, h, w, kw, kh, pad, stride = case
    check_products(P, batch, cin, cout, h, w, kw, kh, pad, pad, stride, stride)


# (batch, in channels, out channels, height, width, kernel width, kernel height, pad x and y, stride x and y): windows,
# paddings and strides that differ between the directions, decoded from one number of a cell
@pytest.mark.parametrize("case", [
    (3, 5, 20, 9, 14, 3, 2, 1, 0, 2, 1),
    (3, 5, 20, 14, 9, 2, 5, 0, 2, 1, 3),
    (2, 3, 40, 17, 11, 7, 4, 3, 1, 2, 3),
    (2, 2, 70, 8, 21, 8, 4, 0, 3, 3, 1),    # 32 taps
    (2, 2, 70, 21, 8, 3, 11, 2, 5, 1, 2),   # 33: no mask
    (4, 9, 33, 13, 7, 1, 5, 0, 4, 1, 1),
], ids=lambda c: "x".join(map(str, c)))
def test_products_under_rectangular_windows(P, case):
    check_products(P, *case)


def check_products(P, batch, cin, cout, h, w, kw, kh, px, py, sx, sy):
    """Whole numbers whose sums stay below 2^24: exact in any order, so everything agrees to the bit."""
    oh, ow = (h + 2 * py - kh) // sy + 1, (w + 2 * px - kw) // sx + 1
    n_rows, n_cols = oh * ow, cin * kw * kh
    desc = H.conv_desc(cin, cout, kw, kh, px, py, sx, sy)
    geometry = (desc, batch, h, w, oh, ow)
    rng = np.random.default_rng(batch + cin + cout + h + w + kw + kh + px + sx)
    ints = lambda n: rng.integers(-2, 3, n).astype(np.float32)
    inp, weights, og = P.buf(ints(batch * cin * h * w)), P.buf(ints(cout * n_cols)), P.buf(ints(batch * cout * n_rows))
    out, wg, ig = P.buf(ints(batch * cout * n_rows)), P.buf(ints(cout * n_cols)), P.buf(ints(batch * cin * h * w))
    work = P.buf(np.full(batch * n_rows * n_cols + 5, 7.0, np.float32))

    def unrolled(what):
        n = batch * n_rows * n_cols
        got = work.download()
        H.assert_bit_exact(np.ascontiguousarray(got[:n].reshape(batch, n_cols, n_rows).transpose(0, 2, 1)),
                           work.host[:n].reshape(batch, n_rows, n_cols), what)
        assert np.all(got[n:] == 7.0), what

    for alpha in (0.0, 2.0):
        kernel = P.run(H.convolution, "forward", vec(out), alpha, vec(inp), vec(weights), vec(work), *geometry)
        assert kernel == forward_route(batch, cout, n_cols, n_rows, kw * kh), kernel
        H.assert_bit_exact(out.download(), out.host, f"convolution-forward, alpha {alpha}")
        unrolled("unrolled input")
    for alpha in (0.0, 2.0):
        kernel = P.run(H.convolution, "backward_weights", vec(wg), alpha, vec(og), vec(inp), vec(work), *geometry)
        assert kernel == weight_route(batch, cout, n_cols, n_rows), kernel
        H.assert_bit_exact(wg.download(), wg.host, f"convolution-backward-weights, alpha {alpha}")
    kernel = P.run(H.convolution, "backward_data", vec(ig), 0.0, vec(og), vec(weights), vec(work), *geometry)
    assert kernel == data_route(batch, n_cols, cout, n_rows), kernel
    H.assert_bit_exact(ig.download(), ig.host, "convolution-backward-data")
    unrolled("unrolled gradient")


@pytest.mark.parametrize("shift", [0, 5])
def test_forward_over_its_own_input(P, shift):
    """An output that is the input, or shares some of it: the input is unrolled whole before any of the output is stored
    (over 9 cells the product would otherwise be the kernel's that gathers the input as it goes)."""
    batch, c, side, k = 1, 1, 40, 3
    n = c * side * side
    desc, geometry = H.conv_desc(c, c, k, k, 1, 1, 1, 1), (1, side, side, side, side)
    rng = np.random.default_rng(4 + shift)
    ints = lambda m: rng.integers(-4, 5, m).astype(np.float32)
    both, weights, work = P.buf(ints(n + shift)), P.buf(ints(c * k * k)), P.buf(ints(n * k * k))
    inp, out = View(both, [n]), View(both, [n], offset=shift)
    kernel = P.run(H.convolution, "forward", out, 2.0, inp, vec(weights), vec(work), desc, *geometry)
    assert kernel == "conv_unroll+gemm", kernel
    H.assert_bit_exact(both.download(), both.host, "convolution-forward")


def rounding_error(a, b, chain):
    """The 2-norm of the error of a @ b against 64 bits, and that of the same product summed in float, rounded after every
    product, in chains of so many products that are added up one after the other."""
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    exact = a64 @ b64
    total = np.zeros(exact.shape, np.float32)
    for k0 in range(0, a.shape[1], chain):
        acc = np.zeros(exact.shape, np.float32)
        for k in range(k0, min(k0 + chain, a.shape[1])):
            acc = (acc.astype(np.float64) + a64[:, k, None] * b64[k]).astype(np.float32)
        total = (total + acc).astype(np.float32)
    return exact, np.linalg.norm(total - exact)


# (batch, in channels, out channels, side): sums over 54, 144 and 45 cells; 40, 112 and 100 out channels; 64, 225 and 441
# positions of an image
@pytest.mark.parametrize("case", [(4, 6, 40, 8), (2, 16, 112, 15), (1, 5, 100, 21)], ids=lambda c: "x".join(map(str, c)))
def test_products_round_as_short_chains_do(P, case):
    """The error of a product is that of a sum in short chains, whatever the number of its terms: chains of 16 products
    (32 for the weight gradient) leave at least as large an error.  The 2-norms are over a thousand sums or more, whose own
    spread is then below 5 %."""
    batch, cin, cout, side = case
    n_rows, n_cols = side * side, cin * 9
    desc, geometry = H.conv_desc(cin, cout, 3, 3, 1, 1, 1, 1), (batch, side, side, side, side)
    rng = np.random.default_rng(side)
    normal = lambda n: rng.standard_normal(n).astype(np.float32)
    inp, weights, og = P.buf(normal(batch * cin * n_rows)), P.buf(normal(cout * n_cols)), P.buf(normal(batch * cout * n_rows))
    out, wg, ig = P.buf(normal(batch * cout * n_rows)), P.buf(normal(cout * n_cols)), P.buf(normal(batch * cin * n_rows))
    work = P.buf(np.zeros(batch * n_rows * n_cols, np.float32))
    w = weights.init.reshape(cout, n_cols)
    across = lambda buf, rows: np.concatenate(list(buf.reshape(batch, rows, n_rows)), axis=1)

    kernel = P.run(H.convolution, "forward", vec(out), 0.0, vec(inp), vec(weights), vec(work), desc, *geometry)
    assert kernel == "conv_product", kernel
    unrolled = across(work.download(), n_cols)
    exact, bound = rounding_error(w, unrolled, 16)
    assert np.linalg.norm(across(out.download(), cout) - exact) <= 1.05 * bound, "convolution-forward"

    kernel = P.run(H.convolution, "backward_weights", vec(wg), 0.0, vec(og), vec(inp), vec(work), desc, *geometry)
    assert kernel.startswith("conv_weight_gradient"), kernel
    gradient = across(og.init, cout)
    exact, bound = rounding_error(gradient, np.ascontiguousarray(unrolled.T), 32)
    assert np.linalg.norm(wg.download().reshape(cout, n_cols) - exact) <= 1.05 * bound, "convolution-backward-weights"

    kernel = P.run(H.convolution, "backward_data", vec(ig), 0.0, vec(og), vec(weights), vec(work), desc, *geometry)
    assert kernel == "conv_product+conv_roll", kernel
    exact, bound = rounding_error(np.ascontiguousarray(w.T), gradient, 16)
    assert np.linalg.norm(across(work.download(), n_cols) - exact) <= 1.05 * bound, "unrolled gradient"


@pytest.mark.parametrize("code", [capi.F32, capi.F64], ids=["float", "double"])
@pytest.mark.parametrize("cout", [95, 96, 97])      # 97280, 98304 and 99328 weights: the sum shares elements below 98304
def test_weight_gradient_sum_over_many_weights(P, code, cout):
    """Whole numbers: exact in any order."""
    batch, cin, side = 9, 1024, 3
    desc, geometry = H.conv_desc(cin, cout, 1, 1, 0, 0, 1, 1), (batch, side, side, side, side)
    rng = np.random.default_rng(cout)
    ints = lambda n: rng.integers(-4, 5, n).astype(NP[code])
    n_rows = side * side
    inp, weights, og = P.buf(ints(batch * cin * n_rows)), P.buf(ints(cout * cin)), P.buf(ints(batch * cout * n_rows))
    out, work, wg = P.buf(ints(batch * cout * n_rows)), P.buf(ints(batch * n_rows * cin)), P.buf(ints(cout * cin))
    P.run(H.convolution, "forward", vec(out), 0.0, vec(inp), vec(weights), vec(work), desc, *geometry)
    for alpha in (0.0, 2.0):
        P.run(H.convolution, "backward_weights", vec(wg), alpha, vec(og), vec(inp), vec(work), desc, *geometry)
        H.assert_bit_exact(wg.download(), wg.host, f"convolution-backward-weights, alpha {alpha}")


def test_weight_gradient_over_its_own_operand(P):
    """A weight gradient stored over the output gradient that it is formed from: one split, which otherwise stores its
    result as soon as a block has it, here goes through scratch memory."""
    cin, cout, side = 40, 100, 8
    n_cols, n_rows = cin * 9, side * side
    desc, geometry = H.conv_desc(cin, cout, 3, 3, 1, 1, 1, 1), (1, side, side, side, side)
    rng = np.random.default_rng(5)
    ints = lambda n: rng.integers(-4, 5, n).astype(np.float32)
    both, inp, work = P.buf(ints(cout * n_cols)), P.buf(ints(cin * n_rows)), P.buf(ints(n_rows * n_cols))
    out, weights = P.buf(ints(cout * n_rows)), P.buf(ints(cout * n_cols))
    P.run(H.convolution, "forward", vec(out), 0.0, vec(inp), vec(weights), vec(work), desc, *geometry)
    og = View(both, [cout * n_rows])
    kernel = P.run(H.convolution, "backward_weights", vec(both), 0.0, og, vec(inp), vec(work), desc, *geometry)
    assert kernel == "conv_weight_gradient+conv_sum_partials", kernel
    gradient = both.init[:cout * n_rows].reshape(cout, n_rows).astype(np.float64)
    unrolled = work.download().reshape(n_cols, n_rows).astype(np.float64)
    H.assert_bit_exact(both.download(), (gradient @ unrolled.T).astype(np.float32).reshape(-1), "convolution-backward-weights")


# (batch, in channels, out channels, side, window, stride): the float products that are formed in three pieces to a float, and
# others beside the lines: 64 cells or more over 288 blocks of 256 positions, up to 96 cells over 384; 20 to 64 out channels over
# 128 rows or more, beyond 32 of them in workspaces of 42 MB and more; more than 64; runs of six pieces of positions or more.
# Remainders of 32 cells, 32 rows, 16 channels and 256 positions.
SPLIT_CASES = [
    (46, 8, 33, 40, 3, 1),      # 72 cells, 288 blocks: the float kernel
    (62, 8, 33, 40, 3, 1),      # 388, images of 1600 positions: a block spans two
    (190, 7, 64, 23, 3, 1),     # 63 cells: the float kernel; 393 blocks of 100510 positions
    (150, 7, 64, 23, 3, 1),     # 310 of 79350
    (150, 11, 65, 23, 3, 1),    # 99 cells: the last tile of three; 65 rows: two tiles; 620 blocks: the float kernel
    (170, 11, 65, 23, 3, 1),    # 704
    (30, 4, 31, 50, 5, 1),      # 100 cells of 25 taps, one tile of rows, 294 blocks
    (41, 15, 20, 40, 3, 1),     # 135 rows over 20 channels and 65600 positions
    (40, 15, 20, 40, 3, 1),     # 64000 positions: the float kernel
    (7, 57, 33, 36, 3, 1),      # 513 rows over 33 channels and 9072 positions, 19 MB: the float kernel
    (36, 57, 33, 36, 3, 1),     # 46656, 96 MB
    (2, 57, 64, 68, 3, 1),      # 9248 positions, 64 channels, 19 MB: the float kernel
    (5, 57, 64, 68, 3, 1),      # 23120, 47 MB, in several runs of rows
    (3, 33, 66, 20, 1, 1),      # 33 rows over 66 channels
    (5, 20, 200, 19, 3, 2),     # 180 rows over 200
    (6, 15, 129, 33, 3, 1),     # 135 rows over 129 channels, weight gradient over six long runs
]


@pytest.mark.parametrize("case", SPLIT_CASES, ids=lambda c: "x".join(map(str, c)))
def test_products_in_pieces_at_the_edges_of_their_tiles(P, case):
    batch, cin, cout, side, k, stride = case
    check_products(P, batch, cin, cout, side, side, k, k, k // 2, k // 2, stride, stride)


# The output formed in pieces over a single image of one or two rows: the window reaches below it (test_conv_gather.py has the
# arithmetic).  Those cells are zero, also in the unrolled input.
@pytest.mark.parametrize("case", [
    (1, 8, 5, 1, 100000, 3, 3, 1, 1, 1, 1),
    (1, 4, 5, 2, 40000, 5, 5, 2, 2, 1, 1),
    (1, 16, 5, 1, 100000, 1, 5, 0, 2, 1, 1),
    (2, 8, 5, 1, 50000, 3, 3, 1, 1, 1, 1),
], ids=lambda c: "x".join(map(str, c)))
def test_products_in_pieces_over_low_images(P, case):
    check_products(P, *case)


@pytest.mark.parametrize("case", [
    (64, 12, 33, 103, 3, 1),     # rows of 10609 positions
    (160, 20, 5, 100, 3, 2),     # of 2500, few rows, at a stride
    (48, 16, 24, 104, 3, 1),     # of 10816, whole sectors: the input gradient too, rolled back from the end
], ids=lambda c: "x".join(map(str, c)))
def test_workspaces_beyond_the_last_level_cache(P, case):
    """Unrolled matrices of more than 256 MiB go past the caches, those of half of the images do not: all of it agrees to the bit
    (a position's sum does not depend on the images around it)."""
    batch, cin, cout, side, k, stride = case
    out_side = (side + 2 * (k // 2) - k) // stride + 1
    n_rows, n_cols, part = out_side ** 2, cin * k * k, batch // 2
    cells = n_rows * n_cols
    assert part * cells * 4 < 256 << 20 < batch * cells * 4 and in_pieces(part, cout, n_cols, n_rows, k * k)[0]
    desc, geometry = H.conv_desc(cin, cout, k, k, k // 2, k // 2, stride, stride), (side, side, out_side, out_side)
    rng = np.random.default_rng(cin)
    normal = lambda n: H.Buf(rng.standard_normal(n).astype(np.float32), gpu=True)
    x, w, g = normal(batch * cin * side * side), normal(cout * n_cols), normal(batch * cout * n_rows)
    zeros = lambda n: [H.Buf(np.zeros(n, np.float32), gpu=True) for _ in range(2)]
    out, ig, work = zeros(batch * cout * n_rows), zeros(batch * cin * side * side), zeros(batch * cells)
    try:
        for which, to, per_image, source, source_image in (("forward", out, cout * n_rows, x, cin * side * side),
                                                           ("backward_data", ig, cin * side * side, g, cout * n_rows)):
            H.convolution(P.hip, which, vec(to[0]), 0.0, vec(source), vec(w), vec(work[0]), desc, batch, *geometry)
            for first in (0, part):
                some = lambda buf, n: View(buf, [part * n], offset=first * n)
                H.convolution(P.hip, which, some(to[1], per_image), 0.0, some(source, source_image), vec(w), some(work[1], cells), desc,
                              part, *geometry)
            H.assert_bit_exact(to[0].download(), to[1].download(), which)
            H.assert_bit_exact(work[0].download(), work[1].download(), "unrolled, " + which)
    finally:
        for buf in (x, w, g, *out, *ig, *work):
            buf.free()


def in_pieces(batch, m, k, n_rows, taps):
    """Whether the output of m channels over k cells, its weight gradient and its input gradient are formed in pieces."""
    n = batch * n_rows
    blocks = -(-m // 64) * -(-n // 256)
    forward = forward_route(batch, m, k, n_rows, taps) == "conv_product" and k >= 64 and blocks >= (384 if k <= 96 else 288)
    forward = forward and not (k <= 112 and m > 32 and 512 < blocks <= 640)
    pieces, fit = batch * -(-n_rows // 64), max(batch * max(1, min(64, n_rows // 4096)), (1 << 20) // (4 * m * k))
    want = 1 if pieces <= 3 else max(1, min(512 // (-(-m // 64) * -(-k // 64)), fit, pieces))
    weights = weight_route(batch, m, k, n_rows).startswith("conv_weight") and min(m, k) > 32 and -(-pieces // want) >= 6
    data = k > 32 if m > 64 else m >= 20 and k >= 128 and n >= (8192 if k >= 512 else 65536)
    data = data and (not 32 < m <= 64 or k * n >= (18 if m <= 40 else 10) << 20)
    return forward, weights, data_route(batch, k, m, n_rows) == "conv_product+conv_roll" and data


@pytest.mark.parametrize("cout", [31, 33])     # one tile of rows and two
@pytest.mark.parametrize("positive", [False, True])
def test_outputs_in_pieces_round_as_short_chains_do(P, cout, positive):
    """Of either sign and of one, whose sums grow with every product: the error of an output formed in pieces is no larger than
    that of chains of eight products, the float kernel's."""
    batch, cin, side, k = 30, 20, 50, 3
    n_rows, n_cols = side * side, cin * k * k
    desc, geometry = H.conv_desc(cin, cout, k, k, 1, 1, 1, 1), (batch, side, side, side, side)
    rng = np.random.default_rng(cout)
    values = lambda n: (rng.random(n) if positive else rng.standard_normal(n)).astype(np.float32)
    inp, weights, out = P.buf(values(batch * cin * n_rows)), P.buf(values(cout * n_cols)), P.buf(np.zeros(batch * cout * n_rows, np.float32))
    work = P.buf(np.zeros(batch * n_rows * n_cols, np.float32))
    assert in_pieces(batch, cout, n_cols, n_rows, k * k)[0]
    H.convolution(P.hip, "forward", vec(out), 0.0, vec(inp), vec(weights), vec(work), desc, *geometry)
    unrolled = work.download()[:n_cols * n_rows].reshape(n_cols, n_rows)     # of the first image
    exact, bound = rounding_error(weights.init.reshape(cout, n_cols), unrolled, 8)
    assert np.linalg.norm(out.download()[:cout * n_rows].reshape(cout, n_rows) - exact) <= bound


@pytest.mark.parametrize("case", SPLIT_CASES, ids=lambda c: "x".join(map(str, c)))
def test_which_products_are_formed_in_pieces(P, case):
    """Sums of one product of two floats and zeros: the float kernels and the library round it once.  The pieces leave out up to
    2^-24 of it, and of the thousands of sums here some are rounded the other way."""
    batch, cin, cout, side, k, stride = case
    out_side = (side + 2 * (k // 2) - k) // stride + 1
    n_rows, n_cols = out_side ** 2, cin * k * k
    desc, geometry = H.conv_desc(cin, cout, k, k, k // 2, k // 2, stride, stride), (batch, side, side, out_side, out_side)
    rng = np.random.default_rng(cin + cout)
    normal = lambda *n: rng.standard_normal(n).astype(np.float32)
    at = lambda n, below: rng.integers(0, below, n)
    inp, work = P.buf(normal(batch * cin * side * side)), P.buf(normal(batch * n_rows * n_cols))
    out, wg, ig = P.buf(normal(batch * cout * n_rows)), P.buf(normal(cout * n_cols)), P.buf(normal(batch * cin * side * side))

    cell, one = at(cout, n_cols), normal(cout)
    w = np.zeros((cout, n_cols), np.float32)
    w[np.arange(cout), cell] = one
    H.convolution(P.hip, "forward", vec(out), 0.0, vec(inp), vec(P.buf(w)), vec(work), desc, *geometry)
    unrolled = work.download().reshape(batch, n_cols, n_rows)
    got = [np.any(out.download().reshape(batch, cout, n_rows) != unrolled[:, cell] * one[None, :, None])]

    image, position = at(cout, batch), at(cout, n_rows)
    g = np.zeros((batch, cout, n_rows), np.float32)
    g[image, np.arange(cout), position] = one
    H.convolution(P.hip, "backward_weights", vec(wg), 0.0, vec(P.buf(g)), vec(inp), vec(work), desc, *geometry)
    got.append(np.any(wg.download().reshape(cout, n_cols) != unrolled[image, :, position] * one[:, None]))

    channel, w, ones = at(batch * n_rows, cout).reshape(batch, n_rows), normal(cout, n_cols), normal(batch, n_rows)
    g = np.zeros((batch, cout, n_rows), np.float32)
    np.put_along_axis(g, channel[:, None], ones[:, None], axis=1)
    H.convolution(P.hip, "backward_data", vec(ig), 0.0, vec(P.buf(g)), vec(P.buf(w)), vec(work), desc, *geometry)
    got.append(np.any(work.download().reshape(batch, n_cols, n_rows) != w.T[:, channel].transpose(1, 0, 2) * ones[:, None]))
    assert tuple(map(bool, got)) == in_pieces(batch, cout, n_cols, n_rows, k * k)


# Each kernel of the products in pieces: the output over 33 and over 31 channels, the weight gradient, the input gradient over
# 20, 33, 66 and 65 channels (the last two in tiles of 64 and of 128 rows); and one that is formed in floats throughout
@pytest.mark.parametrize("case", [(62, 8, 33, 40, 3), (30, 4, 31, 50, 5), (41, 15, 20, 40, 3), (36, 57, 33, 36, 3),
                                  (3, 33, 66, 20, 1), (150, 11, 65, 23, 3), (6, 15, 129, 33, 3), (5, 20, 200, 19, 3)], ids=lambda c: "x".join(map(str, c)))
def test_products_in_pieces_at_the_ends_of_the_number_range(P, case):
    """An infinity, a NaN and floats that the pieces do not hold, in the weights and in both gradients' operands: the blocks
    that meet them form their sums again from the floats.  Where the oracle's sums are finite the bar is 1e-5 of the sums of
    magnitudes; elsewhere the classes agree."""
    batch, cin, cout, side, k = case
    n_rows, n_cols = side * side, cin * k * k
    desc, geometry = H.conv_desc(cin, cout, k, k, k // 2, k // 2, 1, 1), (batch, side, side, side, side)
    rng = np.random.default_rng(cin)
    normal = lambda n: rng.standard_normal(n).astype(np.float32)
    x, w, g = normal(batch * cin * n_rows), normal(cout * n_cols), normal(batch * cout * n_rows)
    x[5], x[3 * n_rows + 3], w[3], w[n_cols + 1], g[11], g[2 * n_rows + 1] = np.inf, 1e35, np.nan, -1e36, -np.inf, 3e35
    inp, weights, og = P.buf(x), P.buf(w), P.buf(g)
    out, wg, ig = P.buf(normal(batch * cout * n_rows)), P.buf(normal(cout * n_cols)), P.buf(normal(batch * cin * n_rows))
    work = P.buf(np.zeros(batch * n_rows * n_cols, np.float32))
    ordinary = lambda v: np.where(np.isfinite(v) & (np.abs(v) < 1e30), v, 0).astype(np.float64)
    largest = lambda v: np.abs(ordinary(v)).max()
    # of the sums over the positions: by Cauchy and Schwarz, of the channels' norms
    norm = lambda v, channels: np.sqrt((ordinary(v).reshape(batch, channels, n_rows) ** 2).sum(axis=(0, 2))).max()

    def check(buf, scale, what):
        got, want = buf.download().astype(np.float64), buf.host.astype(np.float64)
        plain = np.isfinite(want) & (np.abs(want) < 1e30)
        assert np.array_equal(np.isnan(got), np.isnan(want)), what
        assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)]), what
        big = np.isfinite(want) & ~plain
        assert np.all(np.abs(got[big] - want[big]) <= 1e-5 * np.abs(want[big])), what
        assert np.all(np.abs(got[plain] - want[plain]) <= 1e-5 * scale), what
        assert not np.all(np.isnan(want)) and plain.any(), what

    P.run(H.convolution, "forward", vec(out), 0.0, vec(inp), vec(weights), vec(work), desc, *geometry)
    check(out, largest(x) * largest(w) * n_cols, "convolution-forward")
    P.run(H.convolution, "backward_weights", vec(wg), 0.0, vec(og), vec(inp), vec(work), desc, *geometry)
    check(wg, norm(g, cout) * norm(x, cin), "convolution-backward-weights")
    P.run(H.convolution, "backward_data", vec(ig), 0.0, vec(og), vec(weights), vec(work), desc, *geometry)
    check(ig, largest(g) * largest(w) * cout * k * k, "convolution-backward-data")


@pytest.mark.parametrize("exponent", [-118, -126, -133, -142])
def test_products_in_pieces_of_small_operands(P, exponent):
    """Floats of 24 bits around the least normal one, under weights near 2^100: the remainders that the pieces are cut from are
    denormal.  The oracle sums in double; bar: 1e-6 of the sum of magnitudes."""
    batch, cin, cout, side, k = 62, 8, 33, 40, 3
    n_rows, n_cols = side * side, cin * k * k
    desc, geometry = H.conv_desc(cin, cout, k, k, 1, 1, 1, 1), (batch, side, side, side, side)
    rng = np.random.default_rng(-exponent)
    full = lambda n, e: np.ldexp(rng.choice([-1.0, 1.0], n) * rng.integers(1 << 23, 1 << 24, n), e - 23).astype(np.float32)
    inp, weights = P.buf(full(batch * cin * n_rows, exponent)), P.buf(full(cout * n_cols, 100))
    out = P.buf(np.zeros(batch * cout * n_rows, np.float32))
    work = P.buf(np.zeros(batch * n_rows * n_cols, np.float32))
    assert in_pieces(batch, cout, n_cols, n_rows, k * k)[0]
    P.run(H.convolution, "forward", vec(out), 0.0, vec(inp), vec(weights), vec(work), desc, *geometry)
    unrolled = np.abs(work.download().reshape(batch, n_cols, n_rows)).astype(np.float64)
    scale = np.matmul(np.abs(weights.init.reshape(cout, n_cols)).astype(np.float64), unrolled).reshape(-1)
    assert np.all(np.abs(out.download().astype(np.float64) - out.host) <= 1e-6 * scale)
