"""Products with few tiles, whose waves split K (gemm_ks.hip): every tile, layout and element alignment at the ends of
tiles, of 64-byte blocks of K, of the waves' shares and of the loads in flight, against 64-bit sums."""
import functools
from ctypes import c_void_p

import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType
from honeycrisp_amd.tensor import Tensor
from recorded_kernels import kernels_of
from test_capture_fusion import check

pytestmark = pytest.mark.gpu

F32, F16 = DType.float32, DType.float16
SHORT = {F32: "f32", F16: "f16"}
GUARD = 64
TILES = [(F16, "16x32"), (F32, "16x32"), (F32, "32x32"), (F32, "32x64")]
# (M, K, N): K below a piece, a block, a wave's block; one block for some of the waves; with a remainder; more than two rounds of loads
SHAPES = [(1, 1, 1), (1, 64, 64), (5, 7, 3), (15, 31, 31), (16, 32, 32), (17, 33, 33), (16, 100, 40), (31, 256, 63), (32, 255, 64),
          (33, 257, 65), (48, 512, 136), (16, 2560, 32), (3, 2561, 37), (16, 4099, 72)]


def product(hip, dtype, a, b, ta, tb, capfd=None):
    """a [M, K] x b [K, N] by hc_matmul from the storage orders (ta, tb), with guards around the result. With `capfd`: the
    result and the names of the kernels that the same call puts into a recording."""
    (M, K), N = a.shape, b.shape[1]
    es = a.itemsize
    guard = (np.arange(M * N + 2 * GUARD) % 7).astype(a.dtype)
    # (the pieces of 16 bytes that are fetched may end behind an operand; without room there another kernel takes the call)
    store = lambda x, transposed: hip.upload(np.concatenate([(x.T if transposed else x).ravel(), np.full(16, np.inf, x.dtype)]))
    out, da, db = hip.upload(guard), store(a, ta), store(b, tb)
    call = lambda: hip._check(hip._lib.hc_matmul(hip._ctx, int(dtype), 1, c_void_p(da.ptr), int(ta), c_void_p(db.ptr), int(tb), 0, M, K, N,
                                                 c_void_p(out.ptr + GUARD * es)))
    if capfd is not None:
        return product(hip, dtype, a, b, ta, tb), kernels_of(hip, capfd, call)
    call()
    host = out.onCPU().view(a.dtype)
    assert np.array_equal(host[:GUARD], guard[:GUARD]) and np.array_equal(host[GUARD + M * N:], guard[GUARD + M * N:]), "wrote outside C"
    return host[GUARD:GUARD + M * N].reshape(M, N)


@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)], ids=["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("dtype,tile", TILES, ids=lambda v: getattr(v, "name", v))
def test_products_whose_waves_split_k(hip_backend, switch, capfd, dtype, tile, layout):
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
        got, kernels = product(hip_backend, dtype, a, b, *layout, capfd=capfd)
        whole = K % (64 // a.itemsize) == 0 and N % (16 // a.itemsize) == 0 and (M % (16 // a.itemsize) == 0 or not layout[0])
        modes = ("m" if layout[0] and M > 1 else "k") + ("k" if layout[1] or N == 1 else "n")     # (a single row or column runs along K)
        assert kernels == ["hc_gemm_%s_ks_%s_%s%s" % (SHORT[dtype], tile, modes, "" if whole else "_e")]
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
    # (either side of each line of the rule: 128 and 129 tiles of 64 x 64, K = 127 and 128; 16 rows and 17, K of one slice and above,
    # 256 tiles of 16 x 32 and 257, 64 and more, 192 and 193, K = 1024 and above)
    (F32, [(64, 128, 8192, "32x64"), (64, 127, 4096, None), (64, 128, 8256, None), (512, 130, 1024, "32x64"), (300, 200, 260, "16x32"),
           (300, 200, 450, "32x32")]),
    (F16, [(16, 24, 8192, None), (16, 24, 8224, None), (16, 72, 8192, "16x32"), (16, 72, 8224, None), (17, 127, 200, None), (128, 256, 256, "16x32"), (128, 256, 320, None),
           (128, 192, 256, None), (96, 1025, 1001, "16x32"), (96, 1024, 1025, "16x32"), (96, 1025, 1025, None), (33, 2048, 2000, "16x32")]),
], ids=["f32", "f16"])
def test_products_at_the_lines_of_the_rule(hip_backend, switch, capfd, dtype, shapes):
    """The rule picks the kernel on either side of its lines; whichever it is, the result is within the bound of the 64-bit sums and
    within twice of it of the tiled kernels'."""
    rng = np.random.default_rng(5)
    for M, K, N, tile in shapes:
        print(dtype.name, M, K, N, flush=True)
        a = (rng.standard_normal((M, K)) / np.sqrt(K)).astype(dtype.numpy)
        b = rng.standard_normal((K, N)).astype(dtype.numpy)
        exact = a.astype(np.float64) @ b.astype(np.float64)
        bound = (K + 8) * 2.0 ** -23 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
        if dtype == F16:
            bound += 2.0 ** -11 * np.abs(exact) + 2.0 ** -24
        got, kernels = product(hip_backend, dtype, a, b, False, False, capfd=capfd)
        assert len(kernels) == 1 and ("_ks_%s_" % tile in kernels[0] if tile else "_ks_" not in kernels[0]), (M, K, N, kernels)
        assert (np.abs(got.astype(np.float64) - exact) <= bound).all()
        switch.setenv("HCHIP_GEMM_TILE", "64x64")
        tiled, kernels = product(hip_backend, dtype, a, b, False, False, capfd=capfd)
        switch.delenv("HCHIP_GEMM_TILE")
        assert len(kernels) == 1 and "_64x64_" in kernels[0], kernels
        assert (np.abs(tiled.astype(np.float64) - got.astype(np.float64)) <= 2 * bound).all()


@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)], ids=["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("dtype,tile", TILES, ids=lambda v: getattr(v, "name", v))
def test_merged_operations_of_products_whose_waves_split_k(hip_backend, switch, capfd, dtype, tile, layout):
    """The second build of the kernels (*_m): every operation that a recording merges into a product, alone and in lists, and groups of
    products over one input, with the bits of the separate launches. Whole blocks of K and remainders, M and N off the tiles."""
    kernel = "hc_gemm_%s_ks_%s_%s%s" % (SHORT[dtype], tile, "m" if layout[0] else "k", "k" if layout[1] else "n")
    ta, tb = layout
    rng = np.random.default_rng(3)
    switch.setenv("HCHIP_GEMM_KERNEL", "ks")
    switch.setenv("HCHIP_GEMM_TILE", tile)
    t = lambda *shape: Tensor(data=rng.standard_normal(shape).astype(np.float32), dtype=dtype)
    # (K a whole number of 16-byte pieces where an operand runs along it; M where A does not)
    shapes = [(64, 128, 64, ""), (40 if ta else 33, 136, 72, "_e"), (72 if ta else 45, 1000, 200, "_e"), (8, 320, 136, "")]
    if ta and not tb:
        shapes.append((40, 131, 72, "_e"))
    with hip_backend.use():
        for M, K, N, edge in shapes:
            print(kernel, M, K, N, flush=True)
            x, res = t(K, M) if ta else t(M, K), t(M, N)
            ws = [t(N, K) if tb else t(K, N) for _ in range(4)]
            rows = [t(N) for _ in range(4)]
            wide = Tensor(data=rng.standard_normal((N,)).astype(np.float32))      # (a parameter in fp32, cast at call time)
            one = lambda i=0: Tensor.matmul(x, ta, ws[i], tb, False)
            programs = [(lambda: one() + rows[0], 1), (lambda: one() + res, 1), (lambda: one().gelu(), 1), (lambda: (one() + rows[0]).gelu(), 2),
                        (lambda: res + (one() + rows[0]), 2), (lambda: ((one() + rows[0]) + res) + rows[1], 3), (lambda: ((one() + rows[0]) + rows[1]).gelu(), 3)]
            if dtype == F16:
                programs += [(lambda: one() + wide.cast(F16), 2), (lambda: (one() + wide.cast(F16)).gelu(), 3)]
            for program, removed in programs:
                assert kernels_of(hip_backend, capfd, program)[-1] == kernel + edge + "_m"
                check(hip_backend, program, removed=removed)
            # groups: plain, with rows of their own, with GELU, of two and of four
            def group(n, member):
                outs = [member(i) for i in range(n)]     # (all of them first: a reader of one in between would end the group)
                return functools.reduce(lambda p, q: p * q, outs)

            groups = [(lambda: group(2, one), 1), (lambda: group(3, lambda i: one(i) + rows[i]), 5),
                      (lambda: group(4, lambda i: (one(i) + rows[i]).gelu()), 11)]
            for program, removed in groups:
                assert kernels_of(hip_backend, capfd, program).count(kernel + edge + "_m") == 1
                check(hip_backend, program, removed=removed)
