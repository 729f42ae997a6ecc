"""Running sums and products of rows that a workgroup takes: ends of lanes, tiles and groups of both sizes of block, rows at any element, every direction.
Values whose sums and products are exact, so that every order of them gives the same bits."""
import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType
from honeycrisp_amd.tensor import Tensor
from recorded_kernels import kernels_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,longest", [(DType.float32, 57344), (DType.float16, 49152), (DType.int64, 24576)], ids=lambda v: getattr(v, "name", v))
@pytest.mark.parametrize("rows,n", [(3, 256), (3, 257), (2048, 300), (2049, 300), (2049, 512), (2, 1023), (2, 1024), (2, 1025), (511, 1027), (512, 1027), (2, 4095),
                                    (2, 4097), (2, 8193), (600, 8195), (1, 16385), (2, 32767), (2, 32769), (1, "longest"), (1, "longer"), (63, 60001), (128, 60001)])
def test_running_sums_and_products_of_rows(hip_backend, capfd, dtype, longest, rows, n):
    n = {"longest": longest, "longer": longest + 1}.get(n, n)
    rng = np.random.default_rng(rows + n)
    # sums of 0 and +-1 that stay within a hundred or so of zero (fp16 holds whole numbers up to 2048); products of signs and halves and twos in turn
    steps = rng.integers(0, 2, size=(rows, (n + 1) // 2)) * rng.choice([-1, 1], size=(rows, 1))
    x = np.stack([steps, -steps], axis=2).reshape(rows, -1)[:, :n]
    factors = np.where(rng.random((rows, n)) < 0.5, -1.0, 1.0) * np.where(np.arange(n) % 9 == 4, 2.0, np.where(np.arange(n) % 9 == 7, 0.5, 1.0))
    if dtype == DType.int64:
        x, factors = x * (1 << 40), np.sign(factors)
    with hip_backend.use():
        t, f = Tensor(data=x.astype(dtype.numpy), dtype=dtype), Tensor(data=factors.astype(dtype.numpy), dtype=dtype)
        kernels = kernels_of(hip_backend, capfd, lambda: t.cumulativeSum(1))
        block = n > 256 and (n >= 512 or rows <= 2048) and (n <= longest or rows >= (128 if dtype == DType.int64 else 64))
        assert kernels[-1].split("_")[3] == ("rowblock" if block else "rows") and (not block or ("_wide_" in kernels[-1]) == (n > 1024 and rows < 512)), kernels
        for reverse in (False, True):
            for exclusive in (False, True):
                for source, value, op, first in ((t, x, np.cumsum, 0), (f, factors, np.cumprod, 1)):
                    want = op(value[:, ::-1] if reverse else value, axis=1)
                    if exclusive:
                        want = np.concatenate([np.full((rows, 1), first), want[:, :-1]], axis=1)
                    want = (want[:, ::-1] if reverse else want).astype(dtype.numpy)
                    call = source.cumulativeSum if source is t else source.cumulativeProd
                    assert np.array_equal(call(1, exclusive=exclusive, reverse=reverse).numpy(), want), (reverse, exclusive, first)


def test_running_sums_of_ordinary_values(hip_backend):
    rng = np.random.default_rng(0)
    x = rng.standard_normal((5, 40000)).astype(np.float32)
    with hip_backend.use():
        got = Tensor(data=x).cumulativeSum(1).numpy().astype(np.float64)
    want = np.cumsum(x.astype(np.float64), axis=1)
    # a value passes through 4 additions in a lane, 6 in a wave, 4 among waves, 10 tiles and a few more, each rounding a sum of magnitudes at most
    assert (np.abs(got - want) <= 32 * 2.0 ** -24 * np.cumsum(np.abs(x).astype(np.float64), axis=1)).all()
