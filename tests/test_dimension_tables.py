"""The shape algebra keeps its results by value where every entry is a plain int; entries of other number types take
the general path.  Both have to agree, on what they return and on what they refuse, and nothing that is kept may be
handed out."""
import random

import numpy as np
import pytest

from cortex_amd import dimensions as dims


def outcome(f, *args):
    try:
        return f(*args)
    except Exception as e:      # noqa: BLE001 (the type and the message are what is compared)
        return type(e), str(e).split("{")[0]


def general(d):
    """The same dimensions with numpy integers: no key, so the general path."""
    out = {"shape": [np.int64(v) for v in d["shape"]], "strides": [np.int64(v) for v in d["strides"]]}
    assert dims.direct_key(out) is None
    return out


def plain(x):
    if isinstance(x, dict):
        return {k: plain(v) for k, v in x.items()}
    return [plain(v) for v in x] if isinstance(x, (list, tuple)) else int(x) if isinstance(x, np.integer) else x


def drawn(rng):
    rank = rng.randint(1, 4)
    shape = [rng.choice([0, 1, 1, 2, 3, 4, 6]) for _ in range(rank)]
    strides, step = [], rng.choice([1, 1, 1, 2])
    for s in reversed(shape):
        strides.insert(0, step)
        step *= max(1, s) * rng.choice([1, 1, 1, 2])
    if rng.random() < 0.3:
        order = rng.sample(range(rank), rank)
        shape, strides = [shape[i] for i in order], [strides[i] for i in order]
    if rng.random() < 0.15:
        strides[rng.randrange(rank)] = 0
    return {"shape": shape, "strides": strides}


@pytest.mark.parametrize("seed", range(4))
def test_kept_results_are_those_of_the_general_path(seed):
    rng = random.Random(seed)
    for _ in range(1500):
        a, b, c = drawn(rng), drawn(rng), drawn(rng)
        target = [rng.choice([1, 2, 3, 4, 6, 12]) for _ in range(rng.randint(1, 3))]
        for _ in range(2):      # the second time from the table
            for f in (dims.dense, dims.access_increasing, dims.ecount, dims.shape):
                assert plain(outcome(f, a)) == plain(outcome(f, general(a))), (f, a)
            for to_shape in (dims.to_2d_shape, dims.to_batch_shape):
                assert plain(outcome(dims.as_matrix, a, to_shape)) == plain(outcome(dims.as_matrix, general(a), to_shape)), a
            assert plain(outcome(dims.in_place_reshape, a, target)) == plain(outcome(dims.in_place_reshape, general(a), target)), (a, target)
            assert plain(outcome(dims.dimension_seq_to_max_shape, a, b, c)) == plain(
                outcome(dims.dimension_seq_to_max_shape, general(a), general(b), general(c))), (a, b, c)
            assert plain(outcome(dims.dimensions, a["shape"])) == plain(outcome(dims.dimensions, general(a)["shape"])), a


def test_results_belong_to_the_caller():
    d = {"shape": [4, 6], "strides": [6, 1]}
    for f in (lambda: dims.in_place_reshape(d, [2, 12]), lambda: dims.as_matrix(d, dims.to_batch_shape),
              lambda: dims.dimensions([4, 6]), lambda: dims.dimension_seq_to_max_shape(d, d)["dimensions"][0]):
        first = f()
        first["shape"][0], first["strides"][0] = 99, 99
        assert f() != first
    info = dims.dimension_seq_to_max_shape(d, d)
    info["max-shape"][0] = 99
    assert dims.dimension_seq_to_max_shape(d, d)["max-shape"] == [4, 6]


def test_truth_values_are_not_taken_for_the_ints_they_equal():
    assert dims.direct_key({"shape": [True, 2], "strides": [2, 1]}) is None


def test_shapes_never_seen_are_worked_out_directly(monkeypatch):
    """A program whose shapes change all the time pays for the tables' keys and entries; the general algebra on top of
    that made it slower than no tables.  Packed tensors of plain ints have to do without it, the first time too."""
    def general(*_):
        raise AssertionError("the general path")

    for name in ("_dimensions", "_dense_of", "_dimension_seq_to_max_shape", "_in_place_reshape"):
        monkeypatch.setattr(dims, name, general)
    rng = random.Random(99)
    for _ in range(50):
        n, c = rng.randint(2, 10 ** 7), rng.randint(2, 10 ** 6)
        d = dims.dimensions([n, 1, c])
        assert d["strides"] == [c, c, 1]
        assert dims.dense(d) and dims.access_increasing(d) and dims.ecount(d) == n * c
        assert dims.in_place_reshape(d, [n * c])["strides"] == [1]
        assert dims.as_matrix(d, dims.to_batch_shape) == {"shape": [n, c], "strides": [c, 1]}
        info = dims.dimension_seq_to_max_shape(d, dims.dimensions([c]))
        assert info == {"max-shape": [n, 1, c], "dimensions": [{"shape": [n, 1, c], "strides": [c, c, 1]},
                                                               {"shape": [1, 1, c], "strides": [c, c, 1]}]}
