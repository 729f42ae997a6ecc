"""Row scatters whose lists one launch makes: ends of its loops, more rows than a workgroup holds, indices read through strides, and the other way
past its number of destinations. Whole numbers: every sum is exact."""
import numpy as np
import pytest

from honeycrisp_amd.descriptors import BroadcastData, BroadcastStrides, DType, ScatterGatherIndices
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


# (up to 24576 rows here, whose indices are read one at a time: both sides of that)
@pytest.mark.parametrize("outer,n,rows", [(3, 1000, 50), (70, 40, 300), (24, 1024, 40), (24, 1025, 40)])
def test_scatter_along_an_inner_axis(hip_backend, capfd, outer, n, rows):
    """Destinations of several outer slices, indices of one slice for all of them and of their own."""
    rng = np.random.default_rng(outer)
    x = rng.integers(-2, 3, size=(outer, n, 256)).astype(np.float32)
    for shape in ((1, n, 1), (outer, n, 1)):
        ids = rng.integers(0, rows, size=shape)
        with hip_backend.use():
            sources, index = Tensor(data=x), Tensor(data=ids)
            kernels = kernels_of(hip_backend, capfd, lambda: sources.scatter(1, rows, index))
            got = sources.scatter(1, rows, index).numpy()
        assert ("hc_scatter_rows_lists" in kernels) == (outer * n <= 24576) != ("hc_scatter_rows_count" in kernels)
        want = np.zeros((outer, rows, 256), np.float32)
        np.add.at(want, (np.arange(outer)[:, None], np.broadcast_to(ids, (outer, n, 1))[..., 0]), x)
        assert np.array_equal(got, want)


@pytest.mark.parametrize("n", [24576, 24577])
def test_indices_read_through_strides(hip_backend, capfd, n):
    """One slice, one index for all rows: not the dense reading, and its limit."""
    x = np.ones((n, 256), np.float32)
    with hip_backend.use():
        sources = Tensor(data=x)
        index_data, strides = Tensor(data=np.array([3])).data, BroadcastStrides([n, 256], [0, 0])
        call = lambda: hip_backend.scatter(sources.data, ScatterGatherIndices([5, 256], 0, BroadcastData(strides, index_data)), DType.float32)
        kernels = kernels_of(hip_backend, capfd, call)
        got = Tensor(dataHandle=call(), shape=[5, 256], dtype=DType.float32).numpy()
    assert ("hc_scatter_rows_lists" in kernels) == (n <= 24576) != ("hc_scatter_rows_count" in kernels)
    want = np.zeros((5, 256), np.float32)
    want[3] = n
    np.testing.assert_array_equal(got, want)
