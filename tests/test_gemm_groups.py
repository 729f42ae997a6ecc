"""Recorded groups of products whose waves split K, with more tiles than there are compute units: a larger tile, the same bits."""
import functools

import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType
from honeycrisp_amd.tensor import Tensor
from recorded_kernels import kernels_of
from test_capture_fusion import check

pytestmark = pytest.mark.gpu

F32, F16 = DType.float32, DType.float16
SHORT = {F32: "f32", F16: "f16"}


@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)], ids=["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("dtype,tile", [(F16, "32x32"), (F32, "32x64")], ids=lambda v: getattr(v, "name", v))
def test_groups_take_a_larger_tile(hip_backend, capfd, dtype, tile, layout):
    ta, tb = layout
    modes = ("m" if ta else "k") + ("k" if tb else "n")
    rng = np.random.default_rng(7)
    t = lambda *shape: Tensor(data=rng.standard_normal(shape).astype(np.float32), dtype=dtype)
    with hip_backend.use():
        # (whole and partial tiles and blocks of K; a block or two of K per wave and dozens; 86 tiles of 16 x 32: three products have 258, two 172.
        # fp32 from K = 1280 on: more than twice as many tiles as compute units, 516 against 492.
        # Narrow products and, with B along K, those that 32 rows pad by a third: as they are in fp32.)
        for M, K, N, edge, members in [(32, 512, 1376, "", 3), (32, 512, 1376, "", 2), (56, 264, 2008, "_e", 4), (56, 1000, 1984, "_e", 2), (24, 136, 2056, "_e", 3),
                                       (64, 1280, 1376, "", 3), (56, 1288, 1312, "_e", 3), (40, 264, 2008, "_e", 4), (2000, 128, 32, "", 3), (1400, 136, 40, "_e", 3)]:
            print(dtype.name, layout, M, K, N, members, flush=True)
            x = t(K, M) if ta else t(M, K)
            ws = [t(N, K) if tb else t(K, N) for _ in range(members)]
            rows, res = [t(N) for _ in range(members)], t(M, N)

            def group(member):
                outs = [member(Tensor.matmul(x, ta, ws[i], tb, False), i) for i in range(members)]
                return functools.reduce(lambda p, q: p * q, outs)

            larger = -(-M // 16) * -(-N // 32) * members > (512 if dtype == F32 and K >= 1280 else 256)
            larger = larger and not (dtype == F32 and (N <= 32 or (tb and M == 40)))
            for program, merged in ((lambda: group(lambda h, i: h), 0), (lambda: group(lambda h, i: h + rows[i]), 1), (lambda: group(lambda h, i: (h + rows[i]).gelu()), 2),
                                    (lambda: group(lambda h, i: res + h), 1)):
                name = "hc_gemm_%s_ks_%s_%s%s_m" % (SHORT[dtype], tile if larger else "16x32", modes, edge)
                assert kernels_of(hip_backend, capfd, program).count(name) == 1
                check(hip_backend, program, removed=members * merged + members - 1)


# 344 and 172 tiles of 64 x 64, a K either side of the line and one that ends within a block; B along N
@pytest.mark.parametrize("K,members,tb,tile", [(448, 2, True, "64x64_kk"), (456, 2, True, "64x64_kk_e"), (440, 2, True, "32x64_kk_e"), (456, 4, True, "32x64_kk_e"),
                                               (448, 2, False, "32x64_kn")], ids=str)
def test_groups_along_k_take_tiles_of_64_by_64(hip_backend, capfd, K, members, tb, tile):
    M, N = 104, 2696
    rng = np.random.default_rng(8)
    t = lambda *shape: Tensor(data=rng.standard_normal(shape).astype(np.float32))
    with hip_backend.use():
        x, ws = t(M, K), [t(N, K) if tb else t(K, N) for _ in range(members)]
        rows, res = [t(N) for _ in range(members)], t(M, N)

        def group(member):
            outs = [member(Tensor.matmul(x, False, ws[i], tb, False), i) for i in range(members)]
            return functools.reduce(lambda p, q: p * q, outs)

        for program, merged in ((lambda: group(lambda h, i: h), 0), (lambda: group(lambda h, i: (h + rows[i]).gelu()), 2), (lambda: group(lambda h, i: res + h), 1)):
            assert kernels_of(hip_backend, capfd, program).count("hc_gemm_f32_ks_%s_m" % tile) == 1
            check(hip_backend, program, removed=members * merged + members - 1)
