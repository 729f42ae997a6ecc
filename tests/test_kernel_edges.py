"""Sizes at which kernels change over: edges of tiles and runs, remainders, the smallest and the largest of a
path's range, each against the CPU oracle (or a 64-bit computation where the oracle rounds differently)."""
import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType
from honeycrisp_amd.tensor import Tensor
from test_hip_parity import check_exact, rand

pytestmark = pytest.mark.gpu

F32, F16, I64 = DType.float32, DType.float16, DType.int64


@pytest.mark.parametrize("dtype", [F32, F16, I64], ids=["f32", "f16", "i64"])
@pytest.mark.parametrize("shape", [(3, 2), (2, 255), (2, 257), (2, 513), (2, 1024), (2, 2047), (2, 4095), (2, 4099),
                                   (1, 65536), (1, 65537), (3, 70001)], ids=str)
def test_argsort_at_the_ends_of_runs(hip_backend, oracle_backend, dtype, shape):
    """1 .. 16 entries per lane, the last run of a line of any length, one and two passes of 16-way
    merging; few distinct values, so that equal keys meet in every pair of runs and the order of
    their indices decides."""
    rng = np.random.default_rng(shape[1])
    x = rng.integers(-40, 41, size=shape)
    x = x if dtype == I64 else x.astype(dtype.numpy)
    for descending in (False, True):
        check_exact(hip_backend, oracle_backend, lambda: Tensor(data=x).argsort(1, descending=descending, stable=True))
    if dtype != I64:
        f = rand(rng, shape, dtype)
        f[0, :2] = [np.inf, -np.inf]
        check_exact(hip_backend, oracle_backend, lambda: Tensor(data=f).argsort(1))
