"""The native half of the front end (``csrc/front.cpp``) against the Python functions that it stands in for."""
import ctypes as C
import importlib.util
import random
import sys

import numpy as np
import pytest

import cortex_amd
from cortex_amd import capi, dimensions as dims, driver

pytestmark = pytest.mark.skipif(dims.front is None, reason="built without Python's headers")


class Index:
    """An index tensor as the algebra sees it."""

    def ecount(self):
        return 3


@pytest.fixture(scope="module")
def python():
    """dimensions.py as it is where nothing native has been built."""
    name, package = "cortex_amd._front", vars(cortex_amd)
    loaded, attribute = sys.modules.get(name), package.pop("_front", None)
    sys.modules[name] = None
    try:
        spec = importlib.util.spec_from_file_location("cortex_amd._dimensions_in_python", dims.__file__)
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
    finally:
        sys.modules[name] = loaded
        if attribute is not None:
            package["_front"] = attribute
    assert module.front is None
    return module


def outcome(f, *args, **named):
    try:
        return f(*args, **named)
    except Exception as e:
        return type(e).__name__, str(e)


EDGES = [
    {"shape": [], "strides": []}, {"shape": [4], "strides": []}, {"shape": [4], "strides": [2]},
    {"shape": (2, 3), "strides": (3, 1)},
    {"shape": [2, 3], "strides": [1]}, {"shape": [0, 3], "strides": [3, 1]}, {"shape": [-2, 3], "strides": [3, 1]},
    {"shape": [True, 3], "strides": [3, 1]}, {"shape": [np.int64(2), 3], "strides": [3, 1]},
    {"shape": [2, 3], "strides": [np.int64(3), 1]}, {"shape": [2, Index()], "strides": [3, 1]},
    {"shape": [1 << 40, 1 << 40], "strides": [1 << 40, 1]}, {"shape": [1 << 70], "strides": [1]},
    {"shape": [2, 3], "strides": [1 << 62, 1]}, {"shape": [2] * 8, "strides": [128, 64, 32, 16, 8, 4, 2, 1]},
    {"shape": [2] * 9, "strides": [256, 128, 64, 32, 16, 8, 4, 2, 1]}, {"shape": [1, 1], "strides": [1, 1]},
    {"shape": [2, 3]}, {"strides": [1]}, {"shape": None, "strides": None}, {"shape": [2.0], "strides": [1]},
]


def drawn(rng):
    shape = [rng.choice([1, 1, 2, 3, 4, 6, rng.randint(0, 9)]) for _ in range(rng.randint(1, 5))]
    strides, step = [], 1
    for s in reversed(shape):
        strides.insert(0, step)
        step *= max(s, 1)
    if rng.random() < 0.4:
        rng.shuffle(strides)
    if rng.random() < 0.3:
        strides = [s * 2 for s in strides]
    return {"shape": shape, "strides": strides}


@pytest.mark.parametrize("name", ["direct_key", "ecount", "shape", "dense", "access_increasing", "dimension_seq_to_max_shape",
                                  "commensurate_dims", "to_2d_shape", "to_batch_shape", "as_2d", "as_batch"])
def test_native_shape_algebra_is_the_python_one(python, name):
    native, plain = getattr(dims, name), getattr(python, name)
    assert native is not plain and type(native) is type(len)
    rng = random.Random(name)
    cases = [(d,) for d in EDGES] + [(drawn(rng),) for _ in range(400)]
    if name in ("direct_key", "dimension_seq_to_max_shape", "commensurate_dims"):
        cases += [(a, b) for a in EDGES for b in EDGES]
        cases += [tuple(drawn(rng) for _ in range(rng.randint(2, 5))) for _ in range(800)] + [()]
    else:
        cases += [(), (EDGES[3], EDGES[3])]
        assert native(dims=EDGES[3]) == plain(dims=EDGES[3])
    for args in cases:
        got, want = outcome(native, *args), outcome(plain, *args)
        if isinstance(want, tuple) and want and want[0] == "TypeError":
            assert got[0] == "TypeError", args
        else:
            assert got == want and type(got) is type(want), args


def test_results_are_fresh():
    d = dims.dimensions([2, 3, 4])
    for f in (dims.shape, dims.as_2d, dims.as_batch, dims.to_2d_shape, dims.dimension_seq_to_max_shape):
        want, got = f(d), f(d)
        (got if isinstance(got, list) else got[next(iter(got))]).clear()
        assert f(d) == want and d["shape"] == [2, 3, 4]


@pytest.mark.parametrize("rank", [1, 2, 8])
def test_dims_are_those_that_ctypes_makes(rank):
    d = dims.dimensions(list(range(2, 2 + rank)))
    got = driver._dims_ref(d)
    assert type(got) is bytes and got == bytes(capi.make_dims(d["shape"], d["strides"], None))


@pytest.mark.parametrize("d", [{"shape": [2, np.int64(3)], "strides": [3, 1]}, {"shape": [2, 3], "strides": [np.int64(3), 1]}])
def test_other_dims_still_go_through_ctypes(d):
    assert bytes(driver._dims_ref(d)._obj) == bytes(capi.make_dims([2, 3], [3, 1], None))


def test_calls_report_what_the_library_reports():
    """A refused call raises the same error by both ways in, and leaves the host running: nothing here reaches a device."""
    if not capi.LIB_PATH.exists():
        pytest.skip("the library is not built")
    capi.lib()
    d = dims.dimensions([2, 2])
    native, by_ctypes = driver._dims_ref(d), C.byref(capi.make_dims(d["shape"], d["strides"], None))
    errors = [outcome(capi.call, "ct_assign_constant", None, None, x, 77, 1.0, 4) for x in (native, by_ctypes)]
    assert errors[0] == errors[1] and errors[0][0] == "CortexHipError"
    for args in ((), (None, None, native), (None, 1.5, native, 4, 1.0, 4)):
        with pytest.raises((TypeError, C.ArgumentError)):
            capi.call("ct_assign_constant", *args)
    with pytest.raises(AttributeError):
        capi.call("ct_no_such_entry")


def test_calls_go_to_the_library_that_is_set(monkeypatch):
    """A library put in the place of the one that was loaded gets every call, those that the native half makes among them."""
    if not capi.LIB_PATH.exists():
        pytest.skip("the library is not built")
    capi.lib()
    refused = ("ct_memset", None, None, capi.F32, 0.0, -1)
    with pytest.raises(capi.CortexHipError):
        capi.call(*refused)

    class Library:
        def ct_memset(self, *args):
            calls.append(args)
            return 0

    calls = []
    with monkeypatch.context() as m:
        m.setattr(capi, "_lib", Library())
        assert capi.call(*refused) is None and calls == [refused[1:]]
    with pytest.raises(capi.CortexHipError):
        capi.call(*refused)
    assert len(calls) == 1


def test_bytes_are_dimensions_only_where_the_entry_point_takes_them(monkeypatch):
    """Bytes in the place of any other pointer are an address, as ctypes has it: the source of a copy, of whatever length."""
    class Library:
        def ct_memcpy_async(self, *args):
            calls.append(args)
            return 0

        def ct_assign(self, stream, dest, dest_dims, *args):
            calls.append((dest, dest_dims._obj.ndim, list(dest_dims._obj.shape[:2])))
            return 0

    calls = []
    monkeypatch.setattr(capi, "_lib", Library())
    for source in (b"", bytes(3), bytes(C.sizeof(capi.CtDims)), bytes(5000)):
        capi.call("ct_memcpy_async", 64, source, len(source), 1, None)
        assert calls.pop() == (64, source, len(source), 1, None)
    packed = bytes(capi.make_dims([4, 5], [5, 1]))
    capi.call("ct_assign", None, 64, packed, 64, packed, capi.F32, 20)
    assert calls.pop() == (64, 2, [4, 5])


@pytest.mark.parametrize("stale", [False, True])
def test_a_build_without_a_host_compiler_leaves_the_front_end_in_python(tmp_path, monkeypatch, capsys, stale):
    from cortex_amd import build

    monkeypatch.setattr(build, "FRONT", tmp_path / build.FRONT.name)
    if stale:
        build.FRONT.touch()
    monkeypatch.setenv("PATH", str(tmp_path))
    build._build_front(force=True)
    assert "g++ is missing" in capsys.readouterr().err and list(tmp_path.iterdir()) == []
