"""Which kernel hc_matmul gives a product, either side of the lines of its rules, and the product's sums."""
import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType
from honeycrisp_amd.tensor import Tensor
from recorded_kernels import kernels_of

pytestmark = pytest.mark.gpu

NN, NT, TN, TT = (False, False), (False, True), (True, False), (True, True)


def kernel_of(hip_backend, capfd, batch, m, k, n, layout=NN):
    """Name of the one kernel that takes an fp16 product (batch 0: a single one), after its result was compared with 64-bit sums."""
    rng = np.random.default_rng(m + k + n)
    lead = (batch,) if batch else ()
    a = (rng.standard_normal(lead + (m, k)) / np.sqrt(k)).astype(np.float16)
    b = rng.standard_normal(lead + (k, n)).astype(np.float16)
    store = lambda x, transposed: Tensor(data=np.ascontiguousarray(np.swapaxes(x, -1, -2) if transposed else x))
    with hip_backend.use():
        x, y = store(a, layout[0]), store(b, layout[1])
        call = lambda: (Tensor.batchedMatmul if batch else Tensor.matmul)(x, layout[0], y, layout[1], False)
        kernels = kernels_of(hip_backend, capfd, call)
        got = call().numpy().astype(np.float64)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    # K roundings of fp32 partial sums of at most the sum of magnitudes, then one to fp16
    bound = (k + 8) * 2.0 ** -23 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)) + 2.0 ** -11 * np.abs(exact) + 2.0 ** -24
    assert (np.abs(got - exact) <= bound).all()
    assert len(kernels) == 1
    return kernels[0]


# The tiled kernels' single-slice variant takes it where an operand runs along K, unless both do and K ends within a 16-byte piece.
@pytest.mark.parametrize("k,layout,splits", [(64, NN, False), (65, NN, True), (64, TN, True), (60, NT, True), (56, NT, False), (72, NT, True)], ids=str)
def test_up_to_16_rows_with_a_k_of_one_slice(hip_backend, capfd, k, layout, splits):
    assert ("_ks_" in kernel_of(hip_backend, capfd, 0, 16, k, 96, layout)) == splits


# 48, 16, 32 and 3 rows of a tile start at odd elements; an even K
@pytest.mark.parametrize("k,n,layout,splits", [(341, 72, NT, True), (343, 72, NT, False), (4097, 72, NN, True), (513, 72, TT, False), (511, 72, TT, True),
                                               (4097, 3, TT, True), (4098, 72, NT, True)], ids=str)
def test_operands_along_k_whose_rows_start_at_odd_elements(hip_backend, capfd, k, n, layout, splits):
    assert ("_ks_" in kernel_of(hip_backend, capfd, 0, 40, k, n, layout)) == splits


# The 16x16x32 pipeline where its 128 x 128 tile fits both extents, and where a long K's tiles are on the device at once: 176 of 256 x 128
# and 257.
@pytest.mark.parametrize("batch,m,k,n,mi16", [(130, 128, 1032, 127, True), (130, 65, 1032, 65, True), (130, 128, 1032, 64, False), (130, 64, 1032, 127, False),
                                              (257, 130, 1025, 128, False), (176, 130, 1025, 128, True), (176, 130, 1025, 64, False),
                                              (256, 130, 1023, 128, False), (130, 130, 1025, 129, True), (260, 66, 256, 72, True), (260, 66, 255, 72, False)])
def test_pipeline_of_batches_of_few_columns(hip_backend, capfd, batch, m, k, n, mi16):
    assert ("_mi16_" in kernel_of(hip_backend, capfd, batch, m, k, n)) == mi16


# K of two to four 128-byte slices: 128 x 128 tiles, but not for slices of up to 8 tiles of 256 x 256 above K = 160
@pytest.mark.parametrize("batch,m,k,n,tile", [(64, 168, 249, 968, "256x256"), (64, 168, 161, 968, "256x256"), (64, 168, 160, 968, "128x128"),
                                              (36, 168, 249, 2100, "128x128")])
def test_tiles_of_batches_with_a_short_k(hip_backend, capfd, batch, m, k, n, tile):
    assert "_%s_" % tile in kernel_of(hip_backend, capfd, batch, m, k, n)
