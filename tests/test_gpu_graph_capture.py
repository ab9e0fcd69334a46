"""The library's calls recorded into a HIP graph and replayed.

A caller whose step is a fixed sequence of small calls (the reference's own networks: batches of 128 x 784)
can record the sequence once with hipStreamBeginCapture on the stream it hands to the library and replay it
with one launch per step.  That needs every recorded call to do nothing but launch kernels on that stream:
no allocation, no wait, no memset node (scratch reserved ahead, debug-sync mode off).  The test records a bias
add, a bias gradient, a column reduction cut into row segments (two launches through the stream's scratch),
the same through the entry point that allocates nothing, a softmax, a one-launch batch-normalization update
and an Adam step, replays the graph three times with new inputs and eager work on the stream in between, and
compares every replay, bit for bit, with the same calls made eagerly on the same inputs.
"""
import ctypes as C

import numpy as np
import pytest

from cortex_amd import capi

pytestmark = pytest.mark.gpu

HIP_STREAM_CAPTURE_MODE_THREAD_LOCAL = 1


def hip_runtime():
    rt = C.CDLL("libamdhip64.so")
    for name, argtypes in (("hipStreamBeginCapture", [C.c_void_p, C.c_int]),
                           ("hipStreamEndCapture", [C.c_void_p, C.POINTER(C.c_void_p)]),
                           ("hipGraphInstantiate", [C.POINTER(C.c_void_p), C.c_void_p, C.c_void_p, C.c_void_p, C.c_size_t]),
                           ("hipGraphLaunch", [C.c_void_p, C.c_void_p]),
                           ("hipGraphExecDestroy", [C.c_void_p]),
                           ("hipGraphDestroy", [C.c_void_p]),
                           ("hipGraphGetNodes", [C.c_void_p, C.c_void_p, C.POINTER(C.c_size_t)])):
        fn = getattr(rt, name)
        fn.argtypes = argtypes
        fn.restype = C.c_int
    return rt


class Dev:
    def __init__(self, host: np.ndarray):
        self.host = np.ascontiguousarray(host).reshape(-1)
        p = C.c_void_p()
        capi.call("ct_malloc", C.byref(p), max(1, self.host.nbytes))
        self.ptr = p.value
        self.upload(self.host, None)

    def upload(self, host: np.ndarray, stream):
        host = np.ascontiguousarray(host).reshape(-1)
        assert host.nbytes == self.host.nbytes
        capi.call("ct_memcpy_async", self.ptr, host.ctypes.data, host.nbytes, capi.COPY_H2D, stream)
        capi.call("ct_stream_sync", stream)

    def download(self, stream) -> np.ndarray:
        out = np.empty_like(self.host)
        capi.call("ct_stream_sync", stream)
        capi.call("ct_memcpy_async", out.ctypes.data, self.ptr, out.nbytes, capi.COPY_D2H, stream)
        capi.call("ct_stream_sync", stream)
        return out

    def free(self):
        capi.call("ct_free", self.ptr)


def dims(shape, strides=None):
    if strides is None:
        strides, m = [], 1
        for s in reversed(shape):
            strides.insert(0, m)
            m *= s
    return capi.make_dims(shape, strides)


def test_a_recorded_step_replays_to_the_eager_results():
    rt = hip_runtime()
    capi.call("ct_set_device", 0)
    capi.call("ct_set_debug_sync", 0)
    stream = C.c_void_p()
    capi.call("ct_stream_create", C.byref(stream))
    capi.call("ct_stream_reserve_scratch", stream, 4 << 20, 4 << 20)
    batch, pixels, classes = 128, 784, 10
    rows, cols = 4096, 2048            # a column reduction above the size one launch over narrow strips takes
    rng = np.random.default_rng(41)
    f32 = np.float32
    act = Dev(rng.standard_normal(batch * pixels).astype(f32))
    bias = Dev(rng.standard_normal(pixels).astype(f32))
    logits = Dev(rng.standard_normal(batch * classes).astype(f32))
    big = Dev(rng.standard_normal(rows * cols).astype(f32))
    stats = [Dev(rng.uniform(0.5, 1.5, pixels).astype(f32)) for _ in range(6)]
    params, grads = Dev(rng.standard_normal(pixels * 16).astype(f32)), Dev(rng.standard_normal(pixels * 16).astype(f32))
    m, v = Dev(np.zeros(pixels * 16, f32)), Dev(np.full(pixels * 16, 1e-6, f32))
    # every output twice: one set for the eager calls, one for the graph's
    outs = {side: {"added": Dev(np.zeros(batch * pixels, f32)), "grad": Dev(np.zeros(pixels, f32)),
                   "colsum": Dev(np.zeros(cols, f32)), "colmax": Dev(np.zeros(cols, f32)),
                   "soft": Dev(np.zeros(batch * classes, f32)), "norm": Dev(np.zeros(batch * pixels, f32))}
            for side in ("eager", "graph")}
    state = {side: {"params": Dev(params.host), "m": Dev(m.host), "v": Dev(v.host),
                    "bmean": Dev(np.zeros(pixels, f32)), "bvar": Dev(np.zeros(pixels, f32)),
                    "rmean": Dev(stats[2].host), "rvar": Dev(stats[3].host)} for side in ("eager", "graph")}
    d_act, d_row, d_grad = dims([batch, pixels]), dims([pixels]), dims([batch, pixels], [0, 1])
    d_logits = dims([batch, classes])
    d_cols_view, d_cols_out = dims([cols, rows], [1, cols]), dims([cols, 1])
    ref = C.byref

    def step(side):
        o, st = outs[side], state[side]
        capi.call("ct_binary_op", stream, o["added"].ptr, ref(d_act), act.ptr, ref(d_act), 1.0, bias.ptr, ref(d_row), 1.0,
                  batch * pixels, capi.BINARY_OPS["+"], capi.F32)
        capi.call("ct_binary_accum", stream, o["grad"].ptr, ref(d_grad), 1.0, o["added"].ptr, ref(d_act), 1.0, batch * pixels,
                  capi.BINARY_OPS["+"], 0, 1, capi.F32)
        capi.call("ct_unary_reduce", stream, o["colsum"].ptr, ref(d_cols_out), 1.0, big.ptr, ref(d_cols_view),
                  capi.REDUCE_OPS["sum"], capi.F32)
        capi.call("ct_unary_reduce_noalloc", stream, o["colmax"].ptr, ref(d_cols_out), 1.0, big.ptr, ref(d_cols_view),
                  capi.REDUCE_OPS["max"], capi.F32)
        capi.call("ct_softmax_eltwise", stream, o["soft"].ptr, ref(d_logits), logits.ptr, ref(d_logits), capi.F32)
        capi.call("ct_batch_normalize_update_and_apply_eltwise", stream, o["norm"].ptr, act.ptr, st["bmean"].ptr, st["bvar"].ptr,
                  st["rmean"].ptr, st["rvar"].ptr, 0.9, stats[4].ptr, stats[5].ptr, 1e-3, batch, pixels, capi.F32)
        capi.call("ct_adam_step", stream, capi.F32, 1e-3, 0.9, 0.999, 1e-8, 0.9, 0.999, 1.0, grads.ptr, st["params"].ptr,
                  st["m"].ptr, st["v"].ptr, pixels * 16)

    everything = []
    try:
        step("graph")          # once eagerly: kernels are loaded and scratch is in place before anything is recorded
        for name in ("params", "m", "v", "rmean", "rvar"):
            state["graph"][name].upload(state["eager"][name].host, stream)
        capi.call("ct_memset", stream, outs["graph"]["grad"].ptr, capi.F32, 0.0, pixels)
        capi.call("ct_stream_sync", stream)
        assert rt.hipStreamBeginCapture(stream, HIP_STREAM_CAPTURE_MODE_THREAD_LOCAL) == 0
        try:
            step("graph")
        finally:
            graph = C.c_void_p()
            ended = rt.hipStreamEndCapture(stream, C.byref(graph))
        assert ended == 0 and graph.value, f"the capture did not end cleanly (hipError {ended})"
        n_nodes = C.c_size_t(0)
        assert rt.hipGraphGetNodes(graph, None, C.byref(n_nodes)) == 0
        assert n_nodes.value >= 9, n_nodes.value      # seven calls, two of them two launches
        graph_exec = C.c_void_p()
        assert rt.hipGraphInstantiate(C.byref(graph_exec), graph, None, None, 0) == 0
        for replay in range(3):
            # new inputs, written by eager work on the same stream between the replays
            act.upload(rng.standard_normal(batch * pixels).astype(f32), stream)
            big.upload(rng.standard_normal(rows * cols).astype(f32), stream)
            logits.upload(rng.standard_normal(batch * classes).astype(f32), stream)
            grads.upload(rng.standard_normal(pixels * 16).astype(f32), stream)
            step("eager")
            capi.call("ct_stream_sync", stream)
            assert rt.hipGraphLaunch(graph_exec, stream) == 0
            capi.call("ct_stream_sync", stream)
            for name in outs["eager"]:
                a, b = outs["eager"][name].download(stream), outs["graph"][name].download(stream)
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (replay, name)
            for name in state["eager"]:
                a, b = state["eager"][name].download(stream), state["graph"][name].download(stream)
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (replay, name)
        assert np.any(outs["graph"]["colsum"].download(stream) != 0)
        assert rt.hipGraphExecDestroy(graph_exec) == 0
        assert rt.hipGraphDestroy(graph) == 0
    finally:
        capi.call("ct_stream_sync", stream)
        for group in (outs["eager"], outs["graph"], state["eager"], state["graph"]):
            everything.extend(group.values())
        everything.extend([act, bias, logits, big, params, grads, m, v] + stats)
        for t in everything:
            t.free()
        capi.call("ct_stream_destroy", stream)
        capi.call("ct_set_debug_sync", 1)


class Recorded:
    """What `step` puts on `stream`, as a graph that can be launched again and again."""

    def __init__(self, rt, stream, step):
        self.rt, self.stream, self.graph, self.exec = rt, stream, C.c_void_p(), C.c_void_p()
        assert rt.hipStreamBeginCapture(stream, HIP_STREAM_CAPTURE_MODE_THREAD_LOCAL) == 0
        try:
            step()
        finally:
            ended = rt.hipStreamEndCapture(stream, C.byref(self.graph))
        assert ended == 0 and self.graph.value, f"the capture did not end cleanly (hipError {ended})"
        assert rt.hipGraphInstantiate(C.byref(self.exec), self.graph, None, None, 0) == 0

    def replay(self):
        assert self.rt.hipGraphLaunch(self.exec, self.stream) == 0
        capi.call("ct_stream_sync", self.stream)

    def destroy(self):
        capi.call("ct_stream_sync", self.stream)
        assert self.rt.hipGraphExecDestroy(self.exec) == 0 and self.rt.hipGraphDestroy(self.graph) == 0


@pytest.fixture()
def fresh():
    """A stream without scratch, debug-sync mode off, and a list of tensors that are given back."""
    capi.call("ct_set_device", 0)
    capi.call("ct_set_debug_sync", 0)
    stream, tensors = C.c_void_p(), []
    capi.call("ct_stream_create", C.byref(stream))

    def tensor(host):
        tensors.append(Dev(host))
        return tensors[-1]

    yield stream, tensor
    capi.call("ct_stream_sync", stream)
    for t in tensors:
        t.free()
    capi.call("ct_stream_destroy", stream)
    capi.call("ct_set_debug_sync", 1)


def product(stream, c, a, b, m, n, k):
    """c [m, n] = a [m, k] b [n, k]^T; the kernels that were launched."""
    capi.call("ct_gemm", stream, c.ptr, n, 0, 1, 1.0, a.ptr, m, k, k, b.ptr, n, k, 0.0, capi.F32)
    return capi.last_kernel()


def whole(rng, *shape):
    return rng.integers(-3, 4, shape).astype(np.float32)


def test_recorded_products_and_reductions_outlive_a_larger_eager_product(fresh):
    """A product with partial sums and a split reduction, recorded with the scratch that a first eager call left; then eager
    products that need many times the scratch, between the replays.  Whole numbers: every sum is exact."""
    stream, tensor = fresh
    capi.call("ct_stream_reserve_scratch", stream, 1 << 20, 0)
    rng = np.random.default_rng(3)
    m, n, k, rows, cols = 10, 20, 3700, 4096, 2048
    a, b, c = tensor(whole(rng, m, k)), tensor(whole(rng, n, k)), tensor(whole(rng, m, n))
    x, total = tensor(whole(rng, rows, cols)), tensor(whole(rng, cols))
    sizes = [(768, 1024, 4096), (2048, 3072, 4096)]
    large = [(tensor(whole(rng, q, s)), tensor(whole(rng, p, s)), tensor(np.zeros((q, p), np.float32)), (q, p, s)) for q, p, s in sizes]

    def step():
        assert product(stream, c, a, b, m, n, k).endswith("+gemm_sum")
        capi.call("ct_unary_reduce", stream, total.ptr, C.byref(dims([cols, 1])), 1.0, x.ptr, C.byref(dims([cols, rows], [1, cols])),
                  capi.REDUCE_OPS["sum"], capi.F32)

    step()      # the kernels are loaded
    capi.call("ct_stream_sync", stream)
    recorded = Recorded(hip_runtime(), stream, step)
    for replay in range(5):
        host_a, host_x = whole(rng, m, k), whole(rng, rows, cols)
        a.upload(host_a, stream)
        x.upload(host_x, stream)
        if replay:
            p, q, r, size = large[replay % 2]
            assert product(stream, r, p, q, *size).endswith("+gemm_sum")
        recorded.replay()
        assert np.array_equal(c.download(stream).reshape(m, n), host_a @ b.host.reshape(n, k).T), replay
        assert np.array_equal(total.download(stream), host_x.sum(axis=0)), replay
        if replay:
            rows_of = slice(0, 7)
            want = p.host.reshape(size[0], size[2])[rows_of] @ q.host.reshape(size[1], size[2]).T
            assert np.array_equal(r.download(stream).reshape(size[:2])[rows_of], want), replay
    recorded.destroy()


def test_a_product_recorded_without_scratch_does_without(fresh):
    """The same product keeps no partial sums where a capture finds no scratch, and its result is as exact."""
    stream, tensor = fresh
    rng = np.random.default_rng(4)
    m, n, k = 10, 20, 3700
    a, b, c = tensor(whole(rng, m, k)), tensor(whole(rng, n, k)), tensor(whole(rng, m, n))
    kernels = []
    product(stream, c, a, b, m, n, 30)      # the library is loaded; no scratch needed
    recorded = Recorded(hip_runtime(), stream, lambda: kernels.append(product(stream, c, a, b, m, n, k)))
    assert kernels[0].startswith("gemm_") and not kernels[0].endswith("+gemm_sum"), kernels
    for replay in range(3):
        host = whole(rng, m, k)
        a.upload(host, stream)
        recorded.replay()
        assert np.array_equal(c.download(stream).reshape(m, n), host @ b.host.reshape(n, k).T), replay
        assert product(stream, c, a, b, m, n, k).endswith("+gemm_sum")
        assert np.array_equal(c.download(stream).reshape(m, n), host @ b.host.reshape(n, k).T), replay
    recorded.destroy()


@pytest.mark.parametrize("recorded_rows,reserved", [(262144, 4600 << 10), (262144, 0), (270000, 0)])     # more than 262144: the library's
def test_a_recorded_sort_of_labels_keeps_its_scratch(fresh, recorded_rows, reserved):
    """Updates of rows chosen by labels, recorded on scratch that holds the library's sort of the labels (16 bytes an entry) and
    may not hold the kernels' own (18): eager calls of 262144 between the replays leave that block where it is.  Whole numbers."""
    stream, tensor = fresh
    classes, counts = 5000, (recorded_rows, 262144)
    if reserved:
        capi.call("ct_stream_reserve_scratch", stream, 0, reserved)
    rng = np.random.default_rng(5)
    most = max(counts)
    labels, y = tensor(rng.integers(0, classes, most).astype(np.int32)), tensor(whole(rng, most))
    sums = [tensor(np.zeros(classes, np.float32)) for _ in range(2)]
    rows = [capi.make_dims([n, 1], [1, 1], [labels.ptr, None]) for n in counts]

    def add(side):
        n, plain = counts[side], dims([counts[side], 1])
        capi.call("ct_memset", stream, sums[side].ptr, capi.F32, 0.0, classes)
        capi.call("ct_binary_accum", stream, sums[side].ptr, C.byref(rows[side]), 1.0, y.ptr, C.byref(plain), 1.0, n,
                  capi.BINARY_OPS["+"], 0, 1, capi.F32)

    add(0)
    capi.call("ct_stream_sync", stream)
    recorded = Recorded(hip_runtime(), stream, lambda: add(0))
    for replay in range(4):
        host_labels, host = rng.integers(0, classes, most).astype(np.int32), whole(rng, most)
        labels.upload(host_labels, stream)
        y.upload(host, stream)
        if replay:
            add(1)
        recorded.replay()
        for side in (0, 1) if replay else (0,):
            n = counts[side]
            want = np.bincount(host_labels[:n], weights=host[:n], minlength=classes).astype(np.float32)
            assert np.array_equal(sums[side].download(stream), want), (replay, side)
    recorded.destroy()
