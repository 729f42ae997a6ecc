"""fp16 products whose tile leaves compute units without a block because a smaller one needs a nearly empty further round."""
from ctypes import c_void_p

import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType

pytestmark = pytest.mark.gpu

GUARD = 64


@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)], ids=["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("shape", [
    # 64 x 64 and 128 x 64 tiles in two rounds against one round of 128 x 64, 128 x 128, 256 x 128: whole tiles, remainders
    # of M, of N and of K, rows at every alignment, either side of K = 512 and 1024
    (512, 512, 3456), (504, 513, 3440), (1536, 768, 2304), (1531, 600, 2301), (768, 1024, 3072), (1992, 1096, 913), (2048, 511, 1536),
    (1848, 1904, 2245), (1032, 520, 504)])
def test_tiles_that_leave_compute_units_idle(hip_backend, shape, layout):
    M, K, N = shape
    (ta, tb), hip = layout, hip_backend
    rng = np.random.default_rng(M + K + N)
    a = (rng.standard_normal((M, K)) / np.sqrt(K)).astype(np.float16)
    b = rng.standard_normal((K, N)).astype(np.float16)
    guard = (np.arange(M * N + 2 * GUARD) % 7).astype(np.float16)
    out, da, db = hip.upload(guard), hip.upload(np.ascontiguousarray(a.T) if ta else a), hip.upload(np.ascontiguousarray(b.T) if tb else b)
    hip._check(hip._lib.hc_matmul(hip._ctx, int(DType.float16), 1, c_void_p(da.ptr), int(ta), c_void_p(db.ptr), int(tb), 0, M, K, N,
                                  c_void_p(out.ptr + GUARD * 2)))
    host = out.onCPU().view(np.float16)
    assert np.array_equal(host[:GUARD], guard[:GUARD]) and np.array_equal(host[GUARD + M * N:], guard[GUARD + M * N:]), "wrote outside C"
    exact = a.astype(np.float64) @ b.astype(np.float64)
    # K roundings of fp32 partial sums of at most the sum of magnitudes, then one to fp16
    bound = (K + 8) * 2.0 ** -23 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)) + 2.0 ** -11 * np.abs(exact) + 2.0 ** -24
    assert (np.abs(host[GUARD:GUARD + M * N].reshape(M, N).astype(np.float64) - exact) <= bound).all()
