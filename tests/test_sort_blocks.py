"""argsort with as many sorting blocks as compute units and more: blocks of 1024 and of 256 lanes, each with every number of
entries per lane."""
import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType
from honeycrisp_amd.tensor import Tensor
from recorded_kernels import kernels_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [DType.float32, DType.float16, DType.int64], ids=lambda d: d.name)
@pytest.mark.parametrize("lines,length", [(300, 513), (300, 1025), (300, 2049), (300, 4096), (257, 600), (256, 600), (256, 1024), (256, 1025), (256, 2048),
                                          (256, 2049), (128, 4097), (130, 4097), (90, 8193)])
def test_argsort_of_many_lines(hip_backend, capfd, dtype, lines, length):
    rng = np.random.default_rng(lines + length)
    x = rng.integers(-200, 200, size=(lines, length)).astype(dtype.numpy)   # (many equal keys: their order is the indices')
    with hip_backend.use():
        t = Tensor(data=x)
        blocks = lines * -(-length // 4096)
        first = kernels_of(hip_backend, capfd, lambda: t.argsort(1, stable=True))[0]
        assert ("_wide_" in first) == (blocks <= hip_backend.deviceInfo()["compute_units"]), first
        for descending in (False, True):
            got = Tensor(data=x).argsort(1, descending=descending, stable=True).numpy()
            assert np.array_equal(got, np.argsort(-x if descending else x, axis=1, kind="stable"))
