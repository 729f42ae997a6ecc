"""Row scatters whose lists one launch makes: ends of its loops, more rows than a workgroup holds, indices read through strides, and the other way
past its number of destinations. Whole numbers: every sum is exact."""
import numpy as np
import pytest

from honeycrisp_amd.tensor import Tensor
from recorded_kernels import kernels_of

pytestmark = pytest.mark.gpu


# (2 indices per lane: 2048 in a step, eight steps in a round; 32 destinations per workgroup, then 33; one or few destinations take more rows
# than the 8192 that wait in LDS)
@pytest.mark.parametrize("n,rows", [(1, 1), (2, 1), (3, 70000), (2047, 8192), (2049, 8193), (16384, 31), (16385, 33), (18431, 8192), (8193, 1), (20001, 40),
                                    (40001, 1024), (300, 262144), (300, 262145)])
def test_scatter_of_rows(hip_backend, capfd, n, rows):
    rng = np.random.default_rng(n + rows)
    ids = rng.integers(0, rows, size=(n,))
    x = rng.integers(-2, 3, size=(n, 256)).astype(np.float32)
    with hip_backend.use():
        sources, index = Tensor(data=x), Tensor(data=ids)
        kernels = kernels_of(hip_backend, capfd, lambda: sources.scatter(0, rows, index))
        got = sources.scatter(0, rows, index).numpy()
    assert ("hc_scatter_rows_lists" in kernels) == (rows <= 262144) and ("hc_scatter_rows_count" in kernels) == (rows > 262144)
    touched = np.unique(ids)
    want = np.zeros((touched.size, 256), np.float32)
    np.add.at(want, np.searchsorted(touched, ids), x)
    assert np.array_equal(got[touched], want)
    got[touched] = 0
    assert not got.any()


@pytest.mark.parametrize("outer,n,rows", [(3, 1000, 50), (70, 40, 300)])
def test_scatter_along_an_inner_axis(hip_backend, outer, n, rows):
    """Destinations of several outer slices, indices of one slice for all of them and of their own."""
    rng = np.random.default_rng(outer)
    x = rng.integers(-2, 3, size=(outer, n, 256)).astype(np.float32)
    for shape in ((1, n, 1), (outer, n, 1)):
        ids = rng.integers(0, rows, size=shape)
        with hip_backend.use():
            got = Tensor(data=x).scatter(1, rows, Tensor(data=ids)).numpy()
        want = np.zeros((outer, rows, 256), np.float32)
        np.add.at(want, (np.arange(outer)[:, None], np.broadcast_to(ids, (outer, n, 1))[..., 0]), x)
        assert np.array_equal(got, want)
