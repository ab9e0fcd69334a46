"""Shape / stride algebra of cortex tensors: a Python mirror of
``src/cortex/tensor/dimensions.clj``.

A *dimensions* value is a dict ``{"shape": [...], "strides": [...]}`` with the
slowest-changing dimension first and strides in elements.  A shape entry may be
an index tensor (any object with ``ecount()``) instead of a number; that
dimension is then addressed indirectly (``dimensions.clj:7-9``).

Everything here is host-side integer logic shared by all backends; the device
library re-derives the same address function from the resulting maps.

A program makes the same few shapes' calls over and over, and the algebra was
most of what a small call cost (a bias over 128 x 784: 18.6 us, 8.9 with the
tables; a training step of a digit network, of which the GPU is busy for 85 us:
536 us, 271).  Where every shape entry and stride is a plain
int the results are functions of those values alone and are kept, by value, in
bounded ``lru_cache`` tables; index tensors and other number types are worked
out each time.  Callers get fresh lists: nothing that is kept is handed out.
Shapes that change all the time gain nothing from the tables and pay for their
entries, so the packed tensors among them are worked out without the general
algebra (seven functions of a shape never seen: 38 us without tables, 45 with
tables in front of the general algebra, 15 now; of a shape seen before 7).
Where ``csrc/front.cpp`` is built it answers for plain ints in place of the
tables, which are then reached only by what it hands on; the figures above are
of the Python functions.
"""
from __future__ import annotations

from functools import lru_cache
from typing import List, Optional, Sequence

try:
    from . import _front as front
except ImportError:     # not built: everything below works without it
    front = None

_CACHE_LIMIT = 4096


class DimensionError(ValueError):
    """Stands in for the ``ex-info`` thrown by ``when-not-error``."""

    def __init__(self, message: str, data=None):
        super().__init__(f"{message} {data or {}}")
        self.data = data or {}


def _is_number(x) -> bool:
    return isinstance(x, int) or (hasattr(x, "__index__") and not hasattr(x, "ecount"))


def _entry(shape_entry) -> int:
    """``disambiguate-shape-entry`` (:48-53)."""
    if type(shape_entry) is int:
        return shape_entry
    if _is_number(shape_entry):
        return int(shape_entry)
    return int(shape_entry.ecount())


def disambiguate_shape(shape_vec) -> List[int]:
    return [s if type(s) is int else _entry(s) for s in shape_vec]


def direct_shape(shape) -> bool:
    for s in shape:
        if type(s) is not int and not _is_number(s):
            return False
    return True


def _plain(values) -> bool:
    for v in values:
        if type(v) is not int:
            return False
    return True


def direct_key(*args) -> Optional[tuple]:
    """The shapes and strides of ``args`` as hashable values, or None unless all are plain ints."""
    key = []
    for d in args:
        shp, strides = d["shape"], d["strides"]
        for v in shp:
            if type(v) is not int:
                return None
        for v in strides:
            if type(v) is not int:
                return None
        key.append((tuple(shp), tuple(strides)))
    return tuple(key)


def extend_strides(shape, strides) -> List[int]:
    """``extend-strides`` (:75-92): fills missing leading strides row-major."""
    rev_strides = list(reversed(list(strides or [])))
    rev_shape = list(reversed(disambiguate_shape(shape)))
    out: List[int] = []
    for i in range(len(shape)):
        cur = rev_strides[i] if i < len(rev_strides) else None
        if i == 0:
            out.append(cur if cur is not None else 1)
        else:
            out.append(cur if cur is not None else out[i - 1] * rev_shape[i - 1])
    return list(reversed(out))


def _packed_strides(shape) -> Optional[List[int]]:
    """Row-major strides of a shape of plain ints of at least 1 (which ``dimensions`` always accepts), else None."""
    strides, step = [], 1
    for v in reversed(shape):
        if type(v) is not int or v < 1:
            return None
        strides.append(step)
        step *= v
    strides.reverse()
    return strides


def dimensions(shape, names=None, strides=None) -> dict:
    """``dimensions`` (:95-118)."""
    if strides is None:
        packed = _packed_strides(shape)
        if packed:
            return {"shape": list(shape), "strides": packed, "names": names}
    return _dimensions(shape, names, strides)


def _dimensions(shape, names, strides) -> dict:
    strides = extend_strides(shape, strides)
    pairs = sorted(zip(disambiguate_shape(shape), strides), key=lambda p: -p[1])
    max_stride = max([0] + [p[1] for p in pairs])
    elem_count = 1
    for s, _ in pairs[1:]:
        elem_count *= s
    if not elem_count <= max_stride:
        raise DimensionError("Stride appears to be too small for element count",
                             {"max-stride": max_stride, "elem-count": elem_count, "strides": strides, "shape": list(shape)})
    return {"shape": list(shape), "strides": strides, "names": names}


def ecount(dims) -> int:
    n = 1
    for s in dims["shape"]:
        n *= s if type(s) is int else _entry(s)
    return n


def shape(dims) -> List[int]:
    return disambiguate_shape(dims["shape"])


def to_2d_shape(dims) -> List[int]:
    """``->2d-shape`` (:144-153)."""
    shp = dims["shape"]
    if not shp:
        raise DimensionError("Invalid shape in dimension map", {"shape": shp})
    if len(shp) == 1:
        return [1, _entry(shp[0])]
    if not direct_shape(shp[:-1]):
        raise DimensionError("Index buffers not supported for this operation.")
    n = 1
    for s in shp[:-1]:
        n *= int(s)
    return [n, _entry(shp[-1])]


def to_batch_shape(dims) -> List[int]:
    """``->batch-shape`` (:156-165)."""
    shp = dims["shape"]
    if not shp:
        raise DimensionError("Invalid shape in dimension map", {"shape": shp})
    if len(shp) == 1:
        return [1, _entry(shp[0])]
    if not direct_shape(shp[1:]):
        raise DimensionError("Index buffers not supported for this operation.")
    n = 1
    for s in shp[1:]:
        n *= int(s)
    return [_entry(shp[0]), n]


def dense(dims) -> bool:
    """``dense?`` (:178-191)."""
    key = direct_key(dims)
    return _dense_direct(*key[0]) if key else _dense_of(dims["shape"], dims["strides"])


def _dense_of(shp, strides) -> bool:
    if not direct_shape(shp):
        return False
    if len(shp) == 1:
        return int(strides[0]) == 1
    pairs = [(int(s), int(st)) for s, st in zip(shp, strides) if int(s) != 1]
    pairs.sort(key=lambda p: -p[1])
    if not pairs:
        return False
    rest = 1
    for s, _ in pairs[1:]:
        rest *= s
    return pairs[0][1] == rest


def _dense_plain(shp, strides) -> bool:
    """``_dense_of`` for plain ints: the first of the largest strides steps over all the other elements."""
    if len(shp) == 1:
        return strides[0] == 1
    count, largest, extent = 1, None, 1
    for s, st in zip(shp, strides):
        if s != 1:
            count *= s
            if largest is None or st > largest:
                largest, extent = st, s
    if count == 0:
        return _dense_of(shp, strides)
    return largest is not None and largest * extent == count


_dense_direct = lru_cache(maxsize=_CACHE_LIMIT)(_dense_plain)


def direct(dims) -> bool:
    return direct_shape(dims["shape"])


def indirect(dims) -> bool:
    return not direct(dims)


def access_increasing(dims) -> bool:
    """``access-increasing?`` (:204-211)."""
    if not direct_shape(dims["shape"]):
        return False
    st = dims["strides"]
    for i in range(len(st) - 1):
        if not st[i] >= st[i + 1]:
            return False
    return True


def elem_idx_to_addr(rev_shape, rev_strides, rev_max_shape, arg: int, index_lookup=None) -> int:
    """``elem-idx->addr`` (:226-252).  ``index_lookup(entry, i)`` reads element
    ``i`` of an index tensor; it is only needed for indirect shapes."""
    offset = 0
    for i in range(len(rev_shape)):
        next_max = int(rev_max_shape[i])
        entry = rev_shape[i]
        next_dim = _entry(entry)
        shape_idx = arg % next_dim
        arg //= next_max
        if _is_number(entry):
            offset += int(rev_strides[i]) * shape_idx
        else:
            offset += int(rev_strides[i]) * int(index_lookup(entry, shape_idx))
    return offset


def max_extend_strides(shp, strides, max_count: int) -> List[int]:
    """``max-extend-strides`` (:280-300)."""
    shp = disambiguate_shape(shp)
    mi = 0
    for i in range(1, len(shp)):
        if strides[i] > strides[mi]:
            mi = i
    stride_val = strides[mi] * shp[mi]
    return [stride_val] * (max_count - len(strides)) + list(strides)


@lru_cache(maxsize=_CACHE_LIMIT)
def _max_shape_direct(key: tuple) -> tuple:
    max_count = 0
    for shp, strides in key:
        if len(shp) != len(strides) or not shp:
            _dimension_seq_to_max_shape([{"shape": list(s), "strides": list(st)} for s, st in key])   # says what is wrong
        max_count = max(max_count, len(shp))
    max_shape, extended = [0] * max_count, []
    for shp, strides in key:
        pad = max_count - len(shp)
        if pad:
            mi = strides.index(max(strides))
            strides = (strides[mi] * shp[mi],) * pad + strides
            shp = (1,) * pad + shp
        for i, v in enumerate(shp):
            if v > max_shape[i]:
                max_shape[i] = v
        extended.append((shp, strides))
    return tuple(max_shape), tuple(extended)


@lru_cache(maxsize=_CACHE_LIMIT)
def commensurate(key: tuple) -> bool:
    """Whether every dimension of every entry of a ``direct_key`` divides the largest (``tensor.clj:592-604``)."""
    max_shape, extended = _max_shape_direct(key)
    return not any(mx % s != 0 for shp, _ in extended for mx, s in zip(max_shape, shp))


def dimension_seq_to_max_shape(*args) -> dict:
    """``dimension-seq->max-shape`` (:326-353)."""
    key = direct_key(*args)
    if key is None:
        return _dimension_seq_to_max_shape(args)
    max_shape, extended = _max_shape_direct(key)
    return {"max-shape": list(max_shape), "dimensions": [{"shape": list(s), "strides": list(st)} for s, st in extended]}


def _dimension_seq_to_max_shape(args) -> dict:
    for a in args:
        if len(a["shape"]) != len(a["strides"]):
            raise DimensionError("Some dimensions have different shape and stride counts", {"args": list(args)})
    max_count = max([0] + [len(a["shape"]) for a in args])
    strides = [max_extend_strides(a["shape"], a["strides"], max_count) for a in args]
    shapes = [[1] * (max_count - len(a["shape"])) + list(a["shape"]) for a in args]
    max_shape = [max([0] + [disambiguate_shape(s)[i] for s in shapes]) for i in range(max_count)]
    return {"max-shape": max_shape,
            "dimensions": [{"shape": s, "strides": st} for s, st in zip(shapes, strides)]}


def minimize(dims) -> dict:
    """``minimize`` (:356-383): strip size-1 dimensions, merge packed neighbours."""
    stripped = [(s, st) for s, st in zip(dims["shape"], dims["strides"]) if not (_is_number(s) and int(s) == 1)]
    if not stripped:
        return {"shape": [1], "strides": [1]}
    rev = list(reversed(stripped))
    out = [rev[0]]
    for (cur_shp, cur_stride), (last_shp, last_stride) in zip(rev[1:], rev[:-1]):
        if _is_number(last_shp) and int(cur_stride) == int(last_shp) * int(last_stride):
            str_shp, str_str = out[-1]
            out[-1] = (int(str_shp) * int(cur_shp), str_str)
        else:
            out.append((cur_shp, cur_stride))
    out.reverse()
    return {"shape": [s for s, _ in out], "strides": [st for _, st in out]}


def _reshape_plain(key: tuple, new_shape: tuple) -> tuple:
    (shp, strides), = key
    packed = _packed_strides(new_shape)
    if packed and shp and len(shp) == len(strides):
        # most tensors are packed, and their reshape is the packed one
        old = new = 1
        for s in shp:
            old *= s
        for s in new_shape:
            new *= s
        last = strides[0]
        for st in strides:
            if st > last:
                break
            last = st
        else:
            if new <= old and _dense_plain(shp, strides):
                return tuple(packed)
    return tuple(_in_place_reshape({"shape": list(shp), "strides": list(strides)}, list(new_shape))["strides"])


_reshaped_strides = lru_cache(maxsize=_CACHE_LIMIT)(_reshape_plain)


def in_place_reshape(existing_dims, new_shape: Sequence[int]) -> dict:
    """``in-place-reshape`` (:386-470)."""
    new_shape = list(new_shape)
    key = direct_key(existing_dims)
    if key is None or not _plain(new_shape):
        return _in_place_reshape(existing_dims, new_shape)
    return {"shape": new_shape, "strides": list(_reshaped_strides(key, tuple(new_shape)))}


def _in_place_reshape(existing_dims, new_shape: List[int]) -> dict:
    new_dims = dimensions(new_shape)
    if not ecount(new_dims) <= ecount(existing_dims):
        raise DimensionError("Reshaped dimensions are larger than tensor",
                             {"tensor-ecount": ecount(existing_dims), "reshape-ecount": ecount(new_dims)})
    if access_increasing(existing_dims) and dense(existing_dims):
        return {"shape": new_shape, "strides": extend_strides(new_shape, [])}
    if access_increasing(existing_dims):
        existing = minimize(existing_dims)
        info = [[int(s), int(st)] for s, st in zip(reversed(existing["shape"]), reversed(existing["strides"]))]
        old_count = len(info)
        max_old_idx = old_count - 1
        rev_shape = list(reversed(new_shape))
        rev_new_strides: List[int] = []
        new_idx = old_idx = 0
        while new_idx < len(new_shape):
            old_dim, old_stride = info[min(old_idx, max_old_idx)]
            new_dim = int(rev_shape[new_idx])
            if not (old_idx < old_count or new_dim == 1):
                raise DimensionError("Ran out of old shape dimensions",
                                     {"old-idx": old_idx, "rev-new-strides": rev_new_strides, "new-dim": new_dim})
            if new_dim == 1:
                last = rev_new_strides[-1] if rev_new_strides else 1
                prev = rev_shape[new_idx - 1] if new_idx >= 1 else 1
                rev_new_strides.append(int(last) * int(prev))
                new_idx += 1
            elif old_dim == new_dim:
                rev_new_strides.append(old_stride)
                new_idx += 1
                old_idx += 1
            elif old_dim < new_dim:
                raise DimensionError("Cannot combine dimensions across padded boundaries",
                                     {"old-dim": old_dim, "new-dim": new_dim})
            else:
                if old_dim % new_dim != 0:
                    raise DimensionError("New dimension not commensurate with old dimension",
                                         {"old-dim": old_dim, "new-dim": new_dim})
                info[old_idx] = [old_dim // new_dim, old_stride * new_dim]
                rev_new_strides.append(old_stride)
                new_idx += 1
        return {"shape": new_shape, "strides": extend_strides(new_shape, list(reversed(rev_new_strides)))}
    raise DimensionError("Cannot (at this point) in-place-reshape transposed or indirect dimensions")


@lru_cache(maxsize=_CACHE_LIMIT)
def _matrix_direct(key: tuple, to_shape) -> tuple:
    (shp, strides), = key
    new_shape = tuple(to_shape({"shape": list(shp), "strides": list(strides)}))
    return new_shape, _reshape_plain(key, new_shape)


def as_matrix(dims, to_shape) -> dict:
    """``in_place_reshape`` to ``to_shape(dims)``, one of ``to_2d_shape`` and ``to_batch_shape``."""
    key = direct_key(dims)
    if key is None:
        return in_place_reshape(dims, to_shape(dims))
    shp, strides = _matrix_direct(key, to_shape)
    return {"shape": list(shp), "strides": list(strides)}


def as_2d(dims) -> dict:
    return as_matrix(dims, to_2d_shape)


def as_batch(dims) -> dict:
    return as_matrix(dims, to_batch_shape)


def commensurate_dims(*args) -> bool:
    """Whether the dimensions are plain ints and every one divides the largest: what is not is for the general rules."""
    key = direct_key(*args)
    return key is not None and commensurate(key)


def transpose(dims, reorder_vec: Sequence[int]) -> dict:
    """``transpose`` (:473-484): permutes shape and strides; no data moves."""
    shp, strides = dims["shape"], dims["strides"]
    if len(set(reorder_vec)) != len(shp):
        raise DimensionError("Every dimension must be represented in the reorder vector",
                             {"shape": shp, "reorder-vec": list(reorder_vec)})
    return {"shape": [shp[i] for i in reorder_vec], "strides": [strides[i] for i in reorder_vec]}


ALL = "all"


def select(dims, *args) -> dict:
    """``select`` (:487-569).  Each argument is ``ALL``, a number, an increasing
    list of indexes (a contiguous range) or an index tensor.  Returns
    ``{"dimensions": ..., "elem-offset": n}``."""
    data_shp = shape(dims)
    if len(data_shp) != len(args):
        raise DimensionError("arg count must match shape count", {"shape": data_shp, "args": list(args)})
    shp, strides = dims["shape"], dims["strides"]
    rev_shape = list(reversed(shp))
    rev_strides = list(reversed(strides))
    conv = []
    for dim, arg in zip(shp, args):
        if isinstance(arg, str) and arg == ALL:
            conv.append(range(_entry(dim)))
        elif isinstance(arg, (list, tuple, range)):
            arg = list(arg)
            if not all(arg[i] < arg[i + 1] for i in range(len(arg) - 1)):
                raise DimensionError("Argument is not monotonicly increasing", {"argument": arg})
            if not _entry(dim) > max([0] + arg):
                raise DimensionError("Argument out of range of dimension", {"dimension": dim, "argument": arg})
            conv.append(arg)
        elif _is_number(arg):
            conv.append(int(arg))
        elif hasattr(arg, "ecount"):
            if len(arg.shape()) != 1:
                raise DimensionError("Index arguments must be vectors", {"arg-shape": arg.shape()})
            conv.append(arg)
        else:
            raise DimensionError("argument to select of incorrect type", {"arg": arg})
    rev_args = list(reversed(conv))
    products = []
    for item in rev_shape:
        products.append(_entry(item) * (products[-1] if products else 1))
    first_elem_idx = 0
    for arg, prev in zip(rev_args, [None] + products):
        if isinstance(arg, int):
            start = arg
        elif isinstance(arg, (list, range)):
            start = arg[0]
        else:
            start = 0  # indirect indexing: relative index 0
        first_elem_idx += (prev or 1) * start
    elem_addr = elem_idx_to_addr(rev_shape, rev_strides, rev_shape, first_elem_idx,
                                 index_lookup=lambda entry, i: 0)
    kept = [(a, st) for a, st in zip(rev_args, rev_strides) if not isinstance(a, int)]
    new_strides = list(reversed([st for _, st in kept]))
    new_shape = list(reversed([len(a) if isinstance(a, (list, range)) else a for a, _ in kept]))
    return {"dimensions": {"shape": new_shape, "strides": new_strides}, "elem-offset": elem_addr}


if front is not None:
    # The same functions in native code (csrc/front.cpp) where every entry is a plain int; they hand on to the ones above
    # what is not.  A bias over 128 x 784 from Python: 6.4 us a call, 9.1 without; a digit network's training step: 170, 241.
    direct_key, ecount, shape, dense, access_increasing, dimension_seq_to_max_shape, commensurate_dims, to_2d_shape, \
        to_batch_shape, as_2d, as_batch = (front.stand_in(f) for f in (
            direct_key, ecount, shape, dense, access_increasing, dimension_seq_to_max_shape, commensurate_dims, to_2d_shape,
            to_batch_shape, as_2d, as_batch))
