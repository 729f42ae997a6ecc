"""argsort of 32-bit keys by digits: every number of entries per lane, full and partial, values of every kind, both orders, along both axes."""
import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType
from honeycrisp_amd.tensor import Tensor
from recorded_kernels import kernels_of

pytestmark = pytest.mark.gpu


def keys_of(x):
    """The order that the sort uses: of the bits, -0 like +0, NaN by its sign at either end."""
    with np.errstate(invalid="ignore"):
        u = (x.astype(np.float32) + np.float32(0)).view(np.uint32)
    return np.where(u >> 31, ~u, u | np.uint32(1 << 31))


@pytest.mark.parametrize("dtype", [DType.float32, DType.float16], ids=lambda d: d.name)
@pytest.mark.parametrize("lines,length", [(2, 128), (2, 129), (3, 255), (256, 256), (257, 256), (5, 257), (2, 511), (256, 512), (1, 513), (2, 1023), (2, 1024), (2, 1025),
                                          (2, 2048), (2, 2049), (3, 3000), (2, 4095), (2, 4096), (3, 4097), (2, 8191), (1, 50257)])
def test_argsort_by_digits(hip_backend, capfd, dtype, lines, length):
    rng = np.random.default_rng(lines * length)
    bits = rng.integers(0, 1 << (8 * dtype.byteSize), size=(lines, length)).astype(np.uint32 if dtype == DType.float32 else np.uint16)
    anything = bits.view(dtype.numpy)                                     # (every exponent, both signs, infinities and NaN)
    with np.errstate(over="ignore"):
        usual = (rng.standard_normal((lines, length)) * 3).astype(dtype.numpy)
    special = rng.choice(np.array([0.0, -0.0, 1.0, -1.0, np.inf, -np.inf, 65504.0, 6e-8, -6e-8], dtype.numpy), size=(lines, length))
    few = np.full((lines, length), 2.5, dtype.numpy)
    few[:, length // 2] = -1
    with hip_backend.use():
        kernel = kernels_of(hip_backend, capfd, lambda t=Tensor(data=usual): t.argsort(1))[0]
        assert ("_wide_" in kernel or "_radix_" in kernel) == (128 < length and lines * -(-length // 4096) <= 256), kernel
        for x in (anything, usual, special, few):
            for descending in (False, True):
                key = keys_of(x)
                want = np.argsort(~key if descending else key, axis=1, kind="stable")
                assert np.array_equal(Tensor(data=x).argsort(1, descending=descending, stable=True).numpy(), want)
                assert np.array_equal(Tensor(data=np.ascontiguousarray(x.T)).argsort(0, descending=descending, stable=True).numpy(), want.T)
