"""GELU and its gradient of every fp16 value, against 64 bits."""
import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType, ElemwiseOp
from honeycrisp_amd.tensor import Tensor

pytestmark = pytest.mark.gpu


def test_gelu_of_every_half(hip_backend):
    x = np.arange(65536, dtype=np.uint16).view(np.float16)
    with hip_backend.use():
        got = Tensor(data=x).gelu().numpy()
        d = hip_backend.elemwise(Tensor(data=x).data, ElemwiseOp.geluApproxGrad, None, x.size, DType.float16)
        grad = Tensor(dataHandle=d, shape=[x.size], dtype=DType.float16).numpy()
    finite = np.isfinite(x)
    f = x[finite].astype(np.float64)
    u2 = 2 * (0.797884561 * f + 0.035677408145115 * f**3)
    up, down = 1 / (1 + np.exp(np.minimum(-u2, 700))), 1 / (1 + np.exp(np.minimum(u2, 700)))
    # one rounding to fp16 (2^-11 relative, 2^-25 among subnormals); the exponent, |u| up to 12 where the result is not yet zero, carries
    # a few roundings of 2^-24 of itself; the value is f / 2 times 1 + tanh u, where tanh u was rounded to 2^-24
    for value, want, tanh in ((got, f * up, np.abs(f) * 2.0 ** -25), (grad, 2 * f * up * down * (0.797884561 + 0.107032224435345 * f**2) + up, 0)):
        assert (np.abs(value[finite].astype(np.float64) - want) <= np.abs(want) * 2.0 ** -10.9 + 2.0 ** -25 + tanh).all()
    assert got[x == np.inf][0] == np.inf and np.isnan(got[x == -np.inf]).all() and np.isnan(got[np.isnan(x)]).all()
    assert np.isnan(grad[~finite]).all()
