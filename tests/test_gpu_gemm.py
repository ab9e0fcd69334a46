"""gemm! of float matrices at the edges of its tiles and of its number range, against the CPU oracle."""
import ctypes as C
import threading

import numpy as np
import pytest

import harness as H
from harness import View

pytestmark = pytest.mark.gpu


@pytest.fixture()
def P(pair_factory):
    with pair_factory() as pair:
        yield pair


def run(P, a, b, c, ta, tb, m, n, k, alpha=1.0, beta=0.0):
    """c [m, ldc] = alpha * op(a) op(b) + beta * c on both sides; the kernels that ran, the result, the oracle's."""
    ba, bb, bc = P.buf(a), P.buf(b), P.buf(c)
    va, vb, vc = (View(x, [x.init.size]) for x in (ba, bb, bc))
    kernel = P.run(H.gemm, vc, c.shape[1], ta, tb, alpha, va, m, k, a.shape[1], vb, n, b.shape[1], beta)
    return kernel, bc.download().reshape(c.shape), bc.host.reshape(c.shape)


def operands(make, m, n, k, ta, tb, pad=0):
    return (make((k, m + pad) if ta else (m, k + pad)), make((n, k + pad) if tb else (k, n + pad)), make((m, n + pad)))


# tiles are 32, 64 or 128 a side and hold 32 k, in pairs; sixteen waves of the small kernel take 512 k between them
EDGES = [(1, 1, 1), (3, 2, 5), (31, 33, 31), (32, 32, 32), (33, 31, 33), (64, 65, 63), (63, 64, 65), (130, 60, 97), (65, 40, 512),
         (40, 65, 513), (5, 7, 545), (10, 128, 1100), (700, 520, 40), (513, 700, 33), (770, 1030, 66), (513, 385, 700),
         (1040, 1025, 129), (1025, 1040, 290), (2050, 1100, 130), (300, 500, 1100), (130, 70, 3000), (1152, 1030, 550)]


# the small kernel: tiles of 16 x 16, whose eight waves take 256 k between them, in one run, in two and a remainder, and with
# partial sums; of 32 x 32 over more of them
EDGES += [(16, 16, 256), (15, 17, 255), (17, 15, 257), (33, 16, 511), (1, 49, 513), (47, 1, 288), (10, 30, 2600), (640, 450, 255),
          (650, 430, 257), (417, 801, 480)]


@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("size", EDGES, ids=str)
def test_whole_numbers_are_exact(P, size, ta, tb):
    """Whole numbers whose sums stay below 2^24: every product and sum is exact in any order."""
    m, n, k = size
    rng = np.random.default_rng(m + n + k)
    a, b, c = operands(lambda s: rng.integers(-7, 8, s).astype(np.float32), m, n, k, ta, tb, pad=(m + k) % 3)
    for alpha, beta in ((1.0, 0.0), (2.0, -1.0)):
        kernel, got, want = run(P, a, b, c, ta, tb, m, n, k, alpha, beta)
        assert kernel.startswith("gemm_"), kernel
        H.assert_bit_exact(got, want, f"{size} ta={ta} tb={tb} alpha={alpha} ({kernel})")


KERNELS = {(40, 40, 100): "gemm_small", (10, 20, 3700): "gemm_medium_pair+gemm_sum", (640, 640, 50): "gemm_medium",
           (900, 900, 400): "gemm_medium_pair", (2048, 2048, 256): "gemm_large", (64, 2048, 4096): "gemm_medium_pair+gemm_sum",
           (1024, 1536, 2048): "gemm_large+gemm_sum", (2000, 2000, 20): "rocblas_gemm", (650, 450, 255): "gemm_small"}


@pytest.mark.parametrize("size", KERNELS, ids=str)
def test_error_is_below_a_plain_sum_s(P, size):
    """The 2-norm of the error against 64 bits stays below that of the plain float sum, rounded after every product; the
    kernel that ran is the one that the sizes call for.  The plain sum rounds k times at the size of the sum so far; the
    large products here once for 8 k, the five small ones, 2^-8 of them, as often each, and what is left out is below 2^-24 of
    a product, a sixth of that on average and of either sign: an eighth of the roundings and a third of the error, of which
    half is asked for."""
    m, n, k = size
    rng = np.random.default_rng(k)
    a, b, c = operands(lambda s: rng.standard_normal(s).astype(np.float32), m, n, k, False, True)
    kernel, got, _ = run(P, a, b, c, False, True, m, n, k)
    assert kernel == KERNELS[size], kernel
    some = slice(0, 10)   # of the rows: two hundred sums or more
    a64, b64 = a[some].astype(np.float64), b.astype(np.float64)
    exact, plain = a64 @ b64.T, np.zeros((len(a64), n), np.float32)
    for i in range(k):
        plain = (plain + a64[:, i, None] * b64[None, :, i]).astype(np.float32)
    if kernel != "rocblas_gemm":
        assert np.linalg.norm(got[some] - exact) <= 0.5 * np.linalg.norm(plain - exact)


@pytest.mark.parametrize("size", [(40, 50, 32), (640, 640, 50), (900, 900, 400), (2048, 2048, 256)], ids=str)
def test_what_is_left_out_is_below_its_bound(P, size):
    """Every operand 1 + 2^-8 - 2^-17, whose pieces are 1, 2^-8 and -2^-17: the three products that are left out are the most
    that they can be, 0.99 * 2^-24 of a product, and of one sign.  The large products are ones, whose sums are exact.  Bar, in
    2^-24 of the result: 1 for what is left out, 5 k / 8 roundings of the small sums, 2^-7 of the large one, and one each
    where the two sums, those of two groups of waves and the scale meet."""
    m, n, k = size
    x = np.float32(1 + 2.0 ** -8 - 2.0 ** -17)
    a, b = np.full((m, k), x), np.full((n, k), x)
    kernel, got, _ = run(P, a, b, np.zeros((m, n), np.float32), False, True, m, n, k)
    assert kernel in ("gemm_small", "gemm_medium", "gemm_medium_pair", "gemm_large"), kernel
    exact = k * float(x) ** 2
    assert np.all(np.abs(got.astype(np.float64) - exact) <= (4 + 5 * k / 8 / 128) * 2.0 ** -24 * exact), kernel


@pytest.mark.parametrize("size", [(40, 50, 100), (640, 640, 50), (900, 900, 400), (2048, 2048, 256), (64, 2048, 4096), (650, 450, 255)],
                         ids=str)
def test_the_ends_of_the_number_range(P, size):
    """Infinities, NaN, and floats and results beyond what the pieces hold: the block forms its sums again from the floats.
    The oracle sums in double and rounds once; bar: 1e-5 of the sum of magnitudes and, where that is
    denormal, half of the least float for each of the k products, which are rounded to multiples of it; classes alike."""
    m, n, k = size
    rng = np.random.default_rng(m)
    a, b, c = operands(lambda s: rng.standard_normal(s).astype(np.float32), m, n, k, False, True)
    a[1, 3], a[2, k - 1], a[3, 0], a[4, 5], a[5, :] = np.inf, -np.inf, np.nan, 3e38, 1e-42
    a[6, :] = 1e-30
    b[2, :], b[3, 1], b[4, :] = 0.0, 1e37, 1e38
    a[7, :] *= 1e20
    b[6, :] *= 1e18
    kernel, got, want = run(P, a, b, c, False, True, m, n, k)
    scale = np.abs(np.where(np.isfinite(a), a, 0).astype(np.float64)) @ np.abs(b.astype(np.float64)).T
    sure = scale <= 1e38   # sums of finite products that come near the largest float may pass it on the way
    special = ~np.isfinite(want)
    assert np.array_equal(np.isnan(got)[sure], np.isnan(want)[sure]), kernel
    assert np.array_equal(got[sure & special & ~np.isnan(want)], want[sure & special & ~np.isnan(want)]), kernel
    fine = sure & ~special
    assert np.all(np.abs(got[fine].astype(np.float64) - want[fine]) <= 1e-5 * scale[fine] + k * 2.0 ** -150), kernel


@pytest.mark.parametrize("size", [(1, 1), (5, 1435), (100, 39), (500, 500)], ids=str)
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
def test_outer_products_are_the_floats_products(P, size, ta, tb):
    """One product to a result: rounded once, as float multiplication rounds it, also where it is denormal or overflows."""
    m, n = size
    rng = np.random.default_rng(m)
    a, b, c = operands(lambda s: rng.standard_normal(s).astype(np.float32), m, n, 1, ta, tb)
    a.reshape(-1)[::7] *= 1e-25
    a.reshape(-1)[3::11] *= 1e25
    b.reshape(-1)[::5] *= 1e-18
    b.reshape(-1)[2::13] *= 1e18
    kernel, got, _ = run(P, a, b, c, ta, tb, m, n, 1)
    assert kernel == "gemm_small", kernel
    with np.errstate(over="ignore"):
        want = a.reshape(m, 1) * b.reshape(1, n) + np.float32(0)   # a sum begins at +0
    H.assert_bit_exact(got, want, kernel)


@pytest.mark.parametrize("size", [(40, 50, 100), (640, 640, 64), (650, 450, 255)], ids=str)
@pytest.mark.parametrize("exponent", [-118, -126, -133, -142])
def test_small_operands(P, exponent, size):
    """Floats of 24 bits around the least normal one, by floats near 2^100: the remainders that the pieces are cut from are
    denormal.  The oracle sums in double; bar: 1e-6 of the sum of magnitudes."""
    m, n, k = size
    rng = np.random.default_rng(m)
    full = lambda s, e: np.ldexp(rng.choice([-1.0, 1.0], s) * rng.integers(1 << 23, 1 << 24, s), e - 23).astype(np.float32)
    a, b = full((m, k), exponent), full((n, k), 100)
    kernel, got, want = run(P, a, b, np.zeros((m, n), np.float32), False, True, m, n, k)
    assert kernel.startswith("gemm_"), kernel
    scale = np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64)).T
    assert np.all(np.abs(got.astype(np.float64) - want) <= 1e-6 * scale), kernel


@pytest.mark.parametrize("exponent", [-135, -100, 60])
def test_scaled_operands_scale_the_result(P, exponent):
    """Multiplying an operand by a power of two multiplies the result, to the bit, as long as neither leaves the floats:
    also where the operand's last bits are denormal (whole numbers below 2^8 keep them)."""
    m, n, k = 70, 50, 90
    rng = np.random.default_rng(7)
    a, b, c = operands(lambda s: rng.integers(-120, 121, s).astype(np.float32), m, n, k, False, True)
    _, want, _ = run(P, a, b, c, False, True, m, n, k)
    kernel, got, _ = run(P, np.ldexp(a, exponent).astype(np.float32), b, c, False, True, m, n, k)
    H.assert_bit_exact(got, np.ldexp(want, exponent).astype(np.float32), kernel)


def test_a_result_over_its_own_operand_is_the_library_s(P):
    m = 48
    rng = np.random.default_rng(8)
    a = P.buf(rng.integers(-4, 5, m * m).astype(np.float32))
    b, c = P.buf(rng.integers(-4, 5, m * m).astype(np.float32)), P.buf(np.zeros(2 * m * m, np.float32))
    v = lambda x: View(x, [x.init.size])
    assert P.run(H.gemm, v(c), m, False, False, 1.0, v(a), m, m, m, v(b), m, m, 0.0) == "gemm_small"
    H.gemm(P.hip, v(a), m, False, False, 1.0, v(a), m, m, m, v(b), m, m, 0.0)
    from cortex_amd import capi
    assert capi.last_kernel() == "rocblas_gemm"


def test_two_threads_on_one_stream():
    """Products with partial sums, of two sizes, from two threads on one stream: the launches of one call stay together."""
    from cortex_amd import capi
    stream = C.c_void_p()
    capi.call("ct_set_device", 0)
    capi.call("ct_set_debug_sync", 0)
    capi.call("ct_stream_create", C.byref(stream))
    errors, calls = [], 300
    start = threading.Barrier(2)

    def work(m, n, k):
        try:
            capi.call("ct_set_device", 0)
            rng = np.random.default_rng(m)
            host = [rng.integers(-3, 4, s).astype(np.float32) for s in ((m, k), (n, k), (m, n))]
            a, b, c = (H.Buf(h, gpu=True) for h in host)
            others = [H.Buf(np.zeros((m, n), np.float32), gpu=True) for _ in range(9)]
            start.wait()
            for i in range(calls):
                to = c if i % 10 == 0 else others[i % 10 - 1]
                capi.call("ct_gemm", stream, to.dev, n, 0, 1, 1.0, a.dev, m, k, k, b.dev, n, k, 0.0, capi.F32)
                assert capi.last_kernel().endswith("+gemm_sum")
            capi.call("ct_stream_sync", stream)
            want = host[0] @ host[1].T
            for x in [c] + others:
                assert np.array_equal(x.download().reshape(m, n), want)
                x.free()
            a.free()
            b.free()
        except BaseException as e:     # the other thread is not left at the barrier
            start.abort()
            errors.append(e)

    try:
        threads = [threading.Thread(target=work, args=size) for size in ((10, 20, 3700), (64, 2048, 4096))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors
    finally:
        capi.call("ct_stream_destroy", stream)
        capi.call("ct_set_debug_sync", 1)
