"""Products with few tiles, whose waves split K (gemm_ks.hip): every tile, layout and element alignment at the ends of
tiles, of 64-byte blocks of K, of the waves' shares and of the loads in flight, against 64-bit sums."""
from ctypes import c_void_p

import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType

pytestmark = pytest.mark.gpu

F32, F16 = DType.float32, DType.float16
GUARD = 64
TILES = [(F16, "16x32"), (F32, "16x32"), (F32, "32x32"), (F32, "32x64")]
# (M, K, N): K below a piece, a block, a wave's block; one block for some of the waves; with a remainder; more than two rounds of loads
SHAPES = [(1, 1, 1), (1, 64, 64), (5, 7, 3), (15, 31, 31), (16, 32, 32), (17, 33, 33), (16, 100, 40), (31, 256, 63), (32, 255, 64),
          (33, 257, 65), (48, 512, 136), (16, 2560, 32), (3, 2561, 37), (16, 4099, 72)]


def product(hip, dtype, a, b, ta, tb):
    """a [M, K] x b [K, N] by hc_matmul from the storage orders (ta, tb), with guards around the result."""
    (M, K), N = a.shape, b.shape[1]
    es = a.itemsize
    guard = (np.arange(M * N + 2 * GUARD) % 7).astype(a.dtype)
    out, da, db = hip.upload(guard), hip.upload(np.ascontiguousarray(a.T) if ta else a), hip.upload(np.ascontiguousarray(b.T) if tb else b)
    hip._check(hip._lib.hc_matmul(hip._ctx, int(dtype), 1, c_void_p(da.ptr), int(ta), c_void_p(db.ptr), int(tb), 0, M, K, N,
                                  c_void_p(out.ptr + GUARD * es)))
    host = out.onCPU().view(a.dtype)
    assert np.array_equal(host[:GUARD], guard[:GUARD]) and np.array_equal(host[GUARD + M * N:], guard[GUARD + M * N:]), "wrote outside C"
    return host[GUARD:GUARD + M * N].reshape(M, N)


@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)], ids=["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("dtype,tile", TILES, ids=lambda v: getattr(v, "name", v))
def test_products_whose_waves_split_k(hip_backend, switch, dtype, tile, layout):
    rng = np.random.default_rng(len(tile) + 2 * layout[0] + layout[1])
    for M, K, N in SHAPES:
        print(dtype.name, tile, layout, M, K, N, flush=True)
        a = (rng.standard_normal((M, K)) / np.sqrt(K)).astype(dtype.numpy)
        b = rng.standard_normal((K, N)).astype(dtype.numpy)
        exact = a.astype(np.float64) @ b.astype(np.float64)
        # K roundings of fp32 partial sums of at most the sum of magnitudes, then one to the tensor type
        bound = (K + 8) * 2.0 ** -23 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
        if dtype == F16:
            bound += 2.0 ** -11 * np.abs(exact) + 2.0 ** -24
        switch.setenv("HCHIP_GEMM_KERNEL", "ks")
        switch.setenv("HCHIP_GEMM_TILE", tile)
        got = product(hip_backend, dtype, a, b, *layout)
        assert (np.abs(got.astype(np.float64) - exact) <= bound).all()
        if M > 1 and N > 1:
            # what lies behind a row's or a column's last k is the next one's first: an infinity there stays there
            a[1, 0] = np.inf
            b[0, 1] = np.inf
            got = product(hip_backend, dtype, a, b, *layout)
            clean = np.ones((M, N), bool)
            clean[1], clean[:, 1] = False, False
            assert np.isfinite(got[clean]).all() and (np.abs(got[clean].astype(np.float64) - exact[clean]) <= bound[clean]).all()
            assert not np.isfinite(got[~clean]).any()


@pytest.mark.parametrize("dtype,shapes", [
    # (either side of each line of the rule: 128 and 129 tiles of 64 x 64, K = 127 and 128; 16 rows and 17, 64 and 65
    # tiles of 16 x 32, 192 and 193, K = 1024 and above)
    (F32, [(64, 128, 8192), (64, 127, 4096), (64, 128, 8256), (512, 130, 1024), (300, 200, 260)]),
    (F16, [(16, 24, 8192), (16, 24, 8224), (17, 127, 200), (128, 256, 256), (128, 256, 320), (96, 1025, 1001), (96, 1024, 1025), (33, 2048, 2000)]),
], ids=["f32", "f16"])
def test_products_at_the_lines_of_the_rule(hip_backend, switch, dtype, shapes):
    """Whatever kernel the rule picks, the result is within the bound of the 64-bit sums and within twice of it of the tiled kernels'."""
    rng = np.random.default_rng(5)
    for M, K, N in shapes:
        print(dtype.name, M, K, N, flush=True)
        a = (rng.standard_normal((M, K)) / np.sqrt(K)).astype(dtype.numpy)
        b = rng.standard_normal((K, N)).astype(dtype.numpy)
        exact = a.astype(np.float64) @ b.astype(np.float64)
        bound = (K + 8) * 2.0 ** -23 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
        if dtype == F16:
            bound += 2.0 ** -11 * np.abs(exact) + 2.0 ** -24
        got = product(hip_backend, dtype, a, b, False, False)
        assert (np.abs(got.astype(np.float64) - exact) <= bound).all()
        switch.setenv("HCHIP_GEMM_TILE", "64x64")
        tiled = product(hip_backend, dtype, a, b, False, False)
        switch.delenv("HCHIP_GEMM_TILE")
        assert (np.abs(tiled.astype(np.float64) - got.astype(np.float64)) <= 2 * bound).all()
