"""Head swaps around batched products whose rows start at any alignment (sequence lengths that are no whole number of 16-byte
vectors): read and written through the strides, as with aligned rows, and the bits of the separate launches."""
import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType
from honeycrisp_amd.tensor import Tensor
from test_capture_fusion import check

pytestmark = pytest.mark.gpu


def attention(q, k, v, B, T, H, hd):
    heads = lambda x: x.reshape([B, T, H, hd]).swap(1, 2)
    probs = (Tensor.batchedMatmul(heads(q), False, heads(k), True, False) * 0.125).softmax()
    return Tensor.batchedMatmul(probs, False, heads(v), False, False).swap(1, 2).reshape([B, T, H * hd])


def qkv(rng, B, T, H, hd, dtype):
    return [Tensor(data=rng.standard_normal((B, T, H * hd)).astype(np.float32), dtype=dtype) for _ in range(3)]


# (T one below and above a tile and a K-slice, one row; one level of batch and two; heads narrower than a tile.)
@pytest.mark.parametrize("dtype", [DType.float32, DType.float16], ids=["f32", "f16"])
@pytest.mark.parametrize("B,T,H,hd", [(3, 201, 8, 64), (2, 33, 3, 40), (1, 77, 4, 64), (2, 63, 2, 128), (2, 65, 5, 8), (1, 333, 3, 64), (5, 17, 4, 32)])
def test_ragged_head_swaps_fold_into_the_batched_products(hip_backend, dtype, B, T, H, hd):
    rng = np.random.default_rng(B + T + H)
    chain = 2 if dtype == DType.float32 or 2 * T > 512 else 0      # scale, logSoftmax, exp -> 1
    with hip_backend.use():
        q, k, v = qkv(rng, B, T, H, hd, dtype)
        check(hip_backend, lambda: attention(q, k, v, B, T, H, hd), removed=4 + chain)


@pytest.mark.parametrize("dtype", [DType.float32, DType.float16], ids=["f32", "f16"])
def test_rows_that_end_within_a_vector_stay_copies(hip_backend, dtype):
    """Heads of 30: what the last 16 bytes of a head's row reach into is checked for the copy, not for the tensor behind it."""
    rng = np.random.default_rng(30)
    with hip_backend.use():
        q, k, v = qkv(rng, 2, 40, 4, 30, dtype)
        check(hip_backend, lambda: attention(q, k, v, 2, 40, 4, 30), removed=2)
