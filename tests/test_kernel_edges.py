"""Sizes at which kernels change over: edges of tiles and runs, remainders, the smallest and the largest of a
path's range, each against the CPU oracle (or a 64-bit computation where the oracle rounds differently)."""
import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType, ElemwiseOp
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


@pytest.mark.parametrize("dtype", [F32, I64], ids=["f32", "i64"])
@pytest.mark.parametrize("length", [4096 * 3 + 257, 65536 + 4097])
def test_argsort_of_runs_that_overlap_unevenly(hip_backend, oracle_backend, dtype, length):
    """Keys of some runs of 4096 lie between two neighbouring entries of others, and a line that is sorted already; nine
    lines, of which the first eight go to an XCD each, along rows and along columns."""
    rng = np.random.default_rng(length)
    run = np.arange(length) // 4096
    x = rng.integers(-30000, 30001, size=(9, length)) * np.where(run % 3 == 0, 1000, 1)
    x[1] = np.sort(x[1])
    x = x.astype(dtype.numpy)
    for descending in (False, True):
        check_exact(hip_backend, oracle_backend, lambda: Tensor(data=x).argsort(1, descending=descending, stable=True))
    columns = np.ascontiguousarray(x.T)
    check_exact(hip_backend, oracle_backend, lambda: Tensor(data=columns).argsort(0))


@pytest.mark.parametrize("dtype", [F32, F16], ids=["f32", "f16"])
@pytest.mark.parametrize("shape", [(3, 1), (5, 7), (70, 128), (3, 256), (3, 260), (2, 1024), (2, 1028), (3, 2048), (2, 2056),
                                   (2, 8192), (2, 8196), (2, 16384), (2, 16392), (1, 32771)], ids=str)
def test_gradients_of_rows_at_the_ends_of_the_registers(hip_backend, dtype, shape):
    """logSoftmax, its gradient and normalizeGrad: 1, 8 and 64 lanes and a block per row, held in registers or streamed."""
    rng = np.random.default_rng(shape[1])
    x, g = rand(rng, shape, dtype), rand(rng, shape, dtype)
    x64, g64 = x.astype(np.float64), g.astype(np.float64)
    n = shape[1]
    logp = x64 - np.log(np.exp(x64).sum(1, keepdims=True))
    c = x64 - x64.mean(1, keepdims=True)
    shifted = (c * c).mean(1, keepdims=True) + 1e-3
    want = {"logSoftmax": logp, "logSoftmaxGrad": g64 - g64.sum(1, keepdims=True) * np.exp(logp),
            "normalizeGrad": (g64 - g64.mean(1, keepdims=True)) / np.sqrt(shifted)
            - c * (c * g64).sum(1, keepdims=True) / shifted ** 1.5 / n}
    with hip_backend.use():
        xt, gt = Tensor(data=x), Tensor(data=g)
        dims = xt.reduceDims(1)
        got = {"logSoftmax": hip_backend.logSoftmax(xt.data, dims, dtype),
               "logSoftmaxGrad": hip_backend.logSoftmaxGrad(xt.data, gt.data, dims, dtype),
               "normalizeGrad": hip_backend.normalizeGrad(xt.data, gt.data, dims, 1e-3, dtype)}
        got = {name: Tensor(dataHandle=d, shape=list(shape), dtype=dtype).numpy() for name, d in got.items()}
    # a handful of roundings of values no larger than the largest input or result (sums of n terms: sqrt(n) / 16 more);
    # normalizeGrad divides by a deviation of sqrt(1e-3) where a row has one element, and rounds its sums to the type
    eps = 2.0 ** -11 if dtype == F16 else 2.0 ** -24
    for name, value in want.items():
        if name == "normalizeGrad":
            size = max(np.abs(value).max(), np.abs(g64).max(), (np.abs(g64) / np.sqrt(shifted)).max())
        else:
            size = max(np.abs(value).max(), np.abs(x64).max(), np.abs(g64).max(), np.abs(g64.sum(1)).max() if dtype == F32 else 0)
        assert np.abs(got[name] - value).max() <= 16 * eps * size * max(1, np.sqrt(n) / 16), name


@pytest.mark.parametrize("dtype", [F32, F16], ids=["f32", "f16"])
def test_gelu_gradient_over_its_range(hip_backend, dtype):
    """The tails, zero, and values whose cube and square leave the range of the type."""
    x = np.concatenate([np.linspace(-12, 12, 100003), [0.0, -0.0, 300.0, -300.0, 60000.0, -60000.0]]).astype(dtype.numpy)
    u = 0.797884561 * x.astype(np.float64) + 0.035677408145115 * x.astype(np.float64) ** 3
    up, down = 1 / (1 + np.exp(np.minimum(-2 * u, 700))), 1 / (1 + np.exp(np.minimum(2 * u, 700)))
    want = 2 * x.astype(np.float64) * up * down * (0.797884561 + 0.107032224435345 * x.astype(np.float64) ** 2) + up
    with hip_backend.use():
        xt = Tensor(data=x)
        d = hip_backend.elemwise(xt.data, ElemwiseOp.geluApproxGrad, None, x.size, dtype)
        got = Tensor(dataHandle=d, shape=[x.size], dtype=dtype).numpy().astype(np.float64)
    # fp16: one rounding of the result (2^-11 relative, 2^-25 among subnormals); fp32: u of size |u| rounded to 2^-24 moves
    # the result by |u| * 2^-24 of x^2, and 1 - tanh^2 loses what is below 2^-24
    bound = np.abs(want) * 2.0 ** -10.9 + 2.0 ** -25 if dtype == F16 else np.abs(want) * 2.0 ** -20 + 2.0 ** -20
    assert (np.abs(got - want) <= bound).all()
    y = np.array([np.nan, np.inf, -np.inf], dtype=dtype.numpy)
    with hip_backend.use():
        d = hip_backend.elemwise(Tensor(data=y).data, ElemwiseOp.geluApproxGrad, None, 3, dtype)
        assert np.isnan(Tensor(dataHandle=d, shape=[3], dtype=dtype).numpy()).all()


@pytest.mark.parametrize("dtype", [F32, F16, I64], ids=["f32", "f16", "i64"])
@pytest.mark.parametrize("vecs,rows", [(64, 65535), (64, 65536), (256, 16383), (256, 16384), (256, 16385)])
def test_gather_and_scatter_of_rows_around_64_mib(hip_backend, dtype, vecs, rows):
    """Results of 64 MiB and more pass the caches: gather of `rows` rows (a quarter and all of a wave's vectors), scatter whose
    sources and result come to as much. Small whole numbers: every sum is exact in every type."""
    rng = np.random.default_rng(rows)
    width, buckets = vecs * 16 // dtype.byteSize, 301
    table = rng.integers(-3, 4, size=(buckets, width)).astype(dtype.numpy)
    ids = rng.integers(0, buckets, size=(rows,))
    ids[: rows // 2] = np.arange(rows // 2) % 7          # half of the sources meet in a few rows
    x = rng.integers(-1, 2, size=(rows - buckets, 8)).astype(dtype.numpy)
    with hip_backend.use():
        got = Tensor(data=table).gather(0, Tensor(data=ids)).numpy()
        assert got.tobytes() == table[ids].tobytes()
        wide = np.tile(x, (1, width // 8))
        summed = Tensor(data=wide).scatter(0, buckets, Tensor(data=ids[: rows - buckets])).numpy()
    want = np.zeros((buckets, 8))
    np.add.at(want, ids[: rows - buckets], x.astype(np.float64))
    assert np.abs(want).max() < 2048                     # (fp16 holds whole numbers up to 2048)
    np.testing.assert_array_equal(summed, np.tile(want.astype(dtype.numpy), (1, width // 8)))


@pytest.mark.parametrize("dtype", [F32, F16], ids=["f32", "f16"])
@pytest.mark.parametrize("shape", [(1, 32768), (1, 32769), (8, 50257), (3, 65536 + 8), (511, 32772)], ids=str)
def test_log_softmax_of_few_long_rows(hip_backend, dtype, shape):
    """Rows cut into pieces: whole and broken vectors, a last piece of any length, two pieces a row up to one per 1024 elements;
    masked pieces (-infinity) count nothing, a NaN anywhere and a row of -infinity only give NaN."""
    rng = np.random.default_rng(shape[1])
    x = rand(rng, shape, dtype)
    x[0, : shape[1] - 1500] = -np.inf
    x64 = x.astype(np.float64)
    m = x64.max(1, keepdims=True)
    want = x64 - m - np.log(np.exp(x64 - m).sum(1, keepdims=True))
    with hip_backend.use():
        got = Tensor(data=x).logSoftmax().numpy().astype(np.float64)
        # the sum's and the logarithm's last bits, one rounding of log(sum) + max, one of the difference
        eps = np.finfo(dtype.numpy).eps
        finite = np.isfinite(want)
        assert np.array_equal(got[~finite], want[~finite])
        assert np.abs(got - want)[finite].max() <= 2 * eps * np.abs(want[finite]).max() + 4e-6
        y = x.copy()
        y[0, shape[1] // 2] = np.nan
        assert np.isnan(Tensor(data=y).logSoftmax().numpy()[0]).all()
        y[0] = -np.inf
        assert np.isnan(Tensor(data=y).logSoftmax().numpy()[0]).all()


@pytest.mark.parametrize("shape", [(1, 4096), (3, 65 * 1024), (2, 64 * 1024 + 1), (1, 256 * 1024), (1, 257 * 1024), (1, 260 * 1024 + 3)], ids=str)
def test_running_sums_of_segmented_rows(hip_backend, oracle_backend, shape):
    """Rows of 4 to 260 segments: around 64 (a round of a segment's own scan of the totals) and around 256 (past which a launch of its
    own scans them); whole numbers, so every order of the sums gives the same."""
    rng = np.random.default_rng(shape[1])
    x = rng.integers(-2, 3, size=shape)
    for exclusive in (False, True):
        for reverse in (False, True):
            for values in (x, x.astype(np.float32)):
                check_exact(hip_backend, oracle_backend,
                            lambda: Tensor(data=values).cumulativeSum(1, exclusive=exclusive, reverse=reverse))
