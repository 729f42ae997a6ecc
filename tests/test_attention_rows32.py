"""fp16 attention over rows of any whole number of 16-byte vectors and heads of 32, 64 and 128: one launch whose replays
return the bits of the separate launches, at the ends of the 32-row blocks, the chunks of values and the row teams."""
import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType
from honeycrisp_amd.tensor import Tensor
from test_capture_fusion import check

pytestmark = pytest.mark.gpu

F16 = DType.float16
# (heads, T, head width): one vector; 8 lanes per row up to 256 scores; a wave above, one to four vectors per lane
SHAPES = [(300, 16, 32), (256, 24, 64), (130, 40, 64), (130, 64, 32), (100, 72, 128), (40, 248, 64), (32, 256, 128), (33, 264, 64),
          (16, 512, 32), (17, 512, 128), (9, 1000, 64), (8, 1024, 64), (8, 1032, 32), (8, 1536, 64), (4, 2048, 64)]


@pytest.mark.parametrize("heads,t,hd", SHAPES, ids=str)
def test_attention_of_any_row_length(hip_backend, heads, t, hd):
    rng = np.random.default_rng(heads + t + hd)
    with hip_backend.use():
        q, k, v = (Tensor(data=rng.standard_normal((heads, t, hd)).astype(np.float32), dtype=F16) for _ in range(3))
        causal = np.tril(np.ones((t, t))) > 0
        mask = Tensor(data=np.where(causal, 0.0, -1e4).astype(np.float32), dtype=F16)
        never = Tensor(data=np.where(causal, 0.0, -np.inf).astype(np.float32), dtype=F16)

        def attention(scale=0.125, mask=mask, log=False):
            s = Tensor.batchedMatmul(q, False, k, True, False)
            if scale:
                s = s * scale
            if mask is not None:
                s = s + mask
            return Tensor.batchedMatmul(s.logSoftmax() if log else s.softmax(), False, v, False, False)

        check(hip_backend, attention, removed=3 + 2)
        check(hip_backend, lambda: attention(scale=0.3, mask=never), removed=3 + 2)   # (no fp16 value; exponentials of -infinity)
        check(hip_backend, lambda: attention(mask=None), removed=2 + 2)
        check(hip_backend, lambda: attention(scale=None, log=True), removed=1 + 2)


def test_attention_of_swapped_heads(hip_backend):
    """Heads that are an inner axis of [B, T, H, hd], read and written through strides."""
    B, T, H, hd = 6, 200, 8, 64
    rng = np.random.default_rng(1)
    with hip_backend.use():
        q, k, v = (Tensor(data=rng.standard_normal((B, T, H * hd)).astype(np.float32), dtype=F16) for _ in range(3))

        def attention():
            heads = [x.reshape([B, T, H, hd]).swap(1, 2) for x in (q, k, v)]
            p = (Tensor.batchedMatmul(heads[0], False, heads[1], True, False) * 0.125).softmax()
            return Tensor.batchedMatmul(p, False, heads[2], False, False).swap(1, 2).reshape([B, T, H * hd])

        check(hip_backend, attention, removed=4 + 2 + 2)


def test_attention_that_leaves_compute_units_idle_stays_apart(hip_backend):
    """Fewer blocks of 32 rows than compute units: scale, logSoftmax and exp merge, the products stay."""
    rng = np.random.default_rng(2)
    with hip_backend.use():
        q, k, v = (Tensor(data=rng.standard_normal((3, 200, 64)).astype(np.float32), dtype=F16) for _ in range(3))

        def attention():
            p = (Tensor.batchedMatmul(q, False, k, True, False) * 0.125).softmax()
            return Tensor.batchedMatmul(p, False, v, False, False)

        check(hip_backend, attention, removed=2)


# One workgroup per compute unit: heads of 128 above T = 512, and of 64 above 1024 where the rounds of blocks fill the device to less
# than 0.75 on average (288 and 520 blocks against 588). The separate launches are faster there.
@pytest.mark.parametrize("heads,t,hd,merged", [(16, 520, 128, False), (5, 2048, 128, False), (6, 1536, 64, False), (13, 1280, 64, False),
                                               (16, 512, 128, True), (8, 1128, 32, True), (14, 1344, 64, True)], ids=str)
def test_attention_with_one_workgroup_per_compute_unit(hip_backend, heads, t, hd, merged):
    rng = np.random.default_rng(4)
    with hip_backend.use():
        q, k, v = (Tensor(data=rng.standard_normal((heads, t, hd)).astype(np.float32), dtype=F16) for _ in range(3))

        def attention():
            p = (Tensor.batchedMatmul(q, False, k, True, False) * 0.125).softmax()
            return Tensor.batchedMatmul(p, False, v, False, False)

        check(hip_backend, attention, removed=2 + (2 if merged else 0))
