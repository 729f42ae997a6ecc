"""fp16 products whose tile leaves compute units without a block because a smaller one needs a nearly empty further round."""
from ctypes import c_void_p

import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType
from recorded_kernels import kernels_of

pytestmark = pytest.mark.gpu

GUARD = 64


@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)], ids=["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("shape,tile", [
    # 64 x 64 and 128 x 64 tiles in two rounds against one round of 128 x 64, 128 x 128, 256 x 128: whole tiles, remainders
    # of M, of N and of K, rows at every alignment, either side of K = 512 and 1024 (and of the margins: 1.556 times the score
    # of the full tile, 1.214, 1.279; the last shape has too few tiles of any kind)
    ((512, 512, 3456), "128x64"), ((504, 513, 3440), "128x64"), ((1536, 768, 2304), "128x128"), ((1531, 600, 2301), "128x128"),
    ((768, 1024, 3072), "128x128"), ((1992, 1096, 913), "128x64"), ((2048, 511, 1536), "128x64"), ((1848, 1904, 2245), "256x128"),
    ((1032, 520, 504), "64x64")], ids=lambda v: v if isinstance(v, str) else "%dx%dx%d" % v)
def test_tiles_that_leave_compute_units_idle(hip_backend, capfd, shape, tile, layout):
    M, K, N = shape
    (ta, tb), hip = layout, hip_backend
    rng = np.random.default_rng(M + K + N)
    a = (rng.standard_normal((M, K)) / np.sqrt(K)).astype(np.float16)
    b = rng.standard_normal((K, N)).astype(np.float16)
    guard = (np.arange(M * N + 2 * GUARD) % 7).astype(np.float16)
    out, da, db = hip.upload(guard), hip.upload(np.ascontiguousarray(a.T) if ta else a), hip.upload(np.ascontiguousarray(b.T) if tb else b)
    call = lambda: hip._check(hip._lib.hc_matmul(hip._ctx, int(DType.float16), 1, c_void_p(da.ptr), int(ta), c_void_p(db.ptr), int(tb), 0, M, K, N,
                                                 c_void_p(out.ptr + GUARD * 2)))
    kernels = kernels_of(hip, capfd, call)
    assert len(kernels) == 1 and "_%s_" % tile in kernels[0], kernels
    call()
    host = out.onCPU().view(np.float16)
    assert np.array_equal(host[:GUARD], guard[:GUARD]) and np.array_equal(host[GUARD + M * N:], guard[GUARD + M * N:]), "wrote outside C"
    exact = a.astype(np.float64) @ b.astype(np.float64)
    # K roundings of fp32 partial sums of at most the sum of magnitudes, then one to fp16
    bound = (K + 8) * 2.0 ** -23 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)) + 2.0 ** -11 * np.abs(exact) + 2.0 ** -24
    assert (np.abs(host[GUARD:GUARD + M * N].reshape(M, N).astype(np.float64) - exact) <= bound).all()
