"""What the front-end works out per call and keeps by value: strides, products, packed descriptors, scalars."""
import ctypes
import warnings

import numpy as np
import pytest

from honeycrisp_amd import _lib
from honeycrisp_amd.backend import HIPBackend
from honeycrisp_amd.descriptors import BroadcastStrides, DType, product, stridesForShape
from honeycrisp_amd.tensor import Tensor


def view(shape):
    return Tensor(dataHandle=object(), shape=shape, dtype=DType.float32)


@pytest.mark.parametrize("shape,new,strides", [
    ([3, 4], [3, 4], [4, 1]), ([1, 4], [3, 4], [0, 1]), ([4], [2, 3, 4], [0, 0, 1]), ([3, 1, 5], [3, 7, 5], [5, 0, 1]),
    ([], [2], [0]), ([0, 4], [0, 4], [4, 1]), ([2, 0], [2, 0], [0, 1]), ([1, 1], [1, 1], [1, 1])])
def test_expanded_strides(shape, new, strides):
    for kind in (int, np.int64):      # (sizes may be numpy's: what is kept holds Python's)
        made = view([kind(n) for n in shape]).expandStrides([kind(n) for n in new])
        assert made.shape == new and made.strides == strides
        assert all(type(n) is int for n in made.shape + made.strides)
        plain = BroadcastStrides(new, strides)
        assert (made.dataCount, made.isNoOp) == (plain.dataCount, plain.isNoOp)
        made.shape.append(7)          # (the caller's own lists)
        made.strides.clear()


def test_expansions_that_are_refused():
    for _ in range(2):
        with pytest.raises(AssertionError, match="axis 1 cannot expand"):
            view([3, 4]).expandStrides([3, 8])
        with pytest.raises(AssertionError, match="shorter shape"):
            view([3, 4]).expandStrides([4])


def test_products_and_strides():
    assert product([]) == 1 and product([3, 0, 5]) == 0
    wide = [np.int64(1 << 40), np.int64(1 << 40)]
    assert product(wide) == 1 << 80 and type(product(wide)) is int
    # one pass, without warnings: iterators, factors beyond 64 bits, unsigned and narrow integers among Python's
    assert product(iter([3, 4])) == product(np.int64(n) for n in (3, 4)) == 12
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert product(wide) == 1 << 80 and product([np.int64(3), 1 << 70]) == 3 << 70
        assert product(np.array([1 << 40, 1 << 40])) == 1 << 80 and product([np.int8(100), 100]) == product([np.uint64(100), np.int64(100)]) == 10000
    rng = np.random.default_rng(0)
    for _ in range(50):
        shape = [int(n) for n in rng.integers(0, 5, size=rng.integers(0, 7))]
        assert stridesForShape(shape) == [int(np.prod(shape[i + 1:], dtype=np.int64)) for i in range(len(shape))]


def test_packed_descriptors():
    packed = _lib.packed_strides((2, 3), (0, 1))._obj
    assert packed.ndim == 2 and list(packed.shape)[:2] == [2, 3] and list(packed.strides)[:2] == [0, 1]
    with pytest.raises(ValueError, match="at most 8 axes"):
        _lib.packed_strides((1,) * 9, (1,) * 9)


@pytest.mark.parametrize("value", [0.1, -0.0, 1e-46, 16777217.0, 3.4028235e38, 7, True, np.float32(0.1), np.float64(0.1), np.int64(3)])
def test_scalars_round_once(value):
    f, i = HIPBackend._scalar(value, DType.float32)
    want = np.float32(value)
    assert np.float32(ctypes.c_float(f).value).tobytes() == want.tobytes() and i == 0
    if abs(value) < 2 ** 62:
        assert HIPBackend._scalar(value, DType.int64)[1].value == int(value)
