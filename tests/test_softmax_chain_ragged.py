"""[* s] [+ mask] -> logSoftmax [-> exp] over rows that are no whole number of 16-byte vectors: one kernel in a recording and under
batching, and the bits of the separate launches."""
import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType
from honeycrisp_amd.tensor import Tensor
from test_capture_fusion import check

pytestmark = pytest.mark.gpu


# (fp32: 8 lanes up to 128 elements, a wave up to 1024; fp16: a wave from 257 to 2048. Ends of the teams and of their strides.)
@pytest.mark.parametrize("dtype,rows,t", [(DType.float32, r, t) for r, t in [(3, 9), (5, 63), (33, 127), (2, 129), (7, 201), (3, 254), (2, 1021), (2, 1023)]] +
                         [(DType.float16, r, t) for r, t in [(2, 257), (7, 300), (3, 1001), (2, 2047)]],
                         ids=lambda v: v.name if isinstance(v, DType) else str(v))
def test_ragged_attention_softmax_becomes_one_kernel(hip_backend, dtype, rows, t):
    rng = np.random.default_rng(rows + t)
    with hip_backend.use():
        values = rng.standard_normal((rows, t, t)) * 4
        values[0, 0, t // 2] = np.inf                # a row of NaN, as from the separate launches
        values[0, 1, :] = -np.inf                    # ... and one of nothing but -infinity
        values[0, 2, 1] = -np.inf
        scores = Tensor(data=values.astype(np.float32), dtype=dtype)
        mask = Tensor(data=np.where(np.tril(np.ones((t, t))) > 0, 0.0, -1e4).astype(np.float32), dtype=dtype)
        check(hip_backend, lambda: (scores * 0.125 + mask).softmax(), removed=3)
        check(hip_backend, lambda: (mask + scores * 0.125).softmax(), removed=3)
        check(hip_backend, lambda: (scores * 0.125).logSoftmax(), removed=1)
        check(hip_backend, lambda: (scores + mask).softmax(), removed=2)
        check(hip_backend, lambda: scores.softmax(), removed=1)


def test_ragged_rows_that_are_left_alone(hip_backend):
    rng = np.random.default_rng(3)
    with hip_backend.use():
        for shape, dtype in (((9, 5), DType.float32), ((4, 1025), DType.float32), ((4, 2049), DType.float16), ((6, 101), DType.float16)):
            x = Tensor(data=rng.standard_normal(shape).astype(np.float32), dtype=dtype)
            check(hip_backend, lambda: (x * 0.5).softmax(), removed=0)
