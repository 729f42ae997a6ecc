"""Products of few tiles over a long K, computed in parts of K that are added up: the ends of tiles, parts and rows, every layout."""
from ctypes import c_void_p

import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType
from honeycrisp_amd.tensor import Tensor
from recorded_kernels import kernels_of

pytestmark = pytest.mark.gpu

# (m, k, n): one tile and the most parts; parts that end inside a 64 of K, with it, and one element after; whole and ragged tiles; rows that
# are no multiple of 16 bytes or of 4 elements; the fewest outputs; the most tiles there are (128 on a device of 256 compute units) and one more
SHAPES = [(64, 3072, 64), (64, 3136, 80), (9, 3073, 461), (5, 4097, 821), (65, 3137, 63), (16, 3200, 4096), (200, 4099, 130), (512, 3136, 1024),
          (127, 8191, 33), (300, 5000, 256), (40, 3330, 1001), (520, 3200, 1024)]

# one launch, by rows, K and columns of what is stored: more than half as many tiles as compute units; one output less than a tile; fp16 with few columns and
# many rows; fp32 with no more parts than an output has chains in that launch
WHOLE = {(520, 3200, 1024), (1024, 3200, 520), (65, 3137, 63), (63, 3137, 65)}
WHOLE = {DType.float16: WHOLE | {(4096, 3200, 16)},
         DType.float32: WHOLE | {(512, 3136, 1024), (1024, 3136, 512), (16, 3200, 4096), (4096, 3200, 16)}}
SHORT = {DType.float16: "f16", DType.float32: "f32"}


def error_bound(k, size, want, dtype):
    """k additions in fp32, each off by half a last place of a partial sum, and one rounding to the result's type."""
    return k * 2.0 ** -24 * size + (2.0 ** -11 * np.abs(want) + 2.0 ** -24 if dtype == DType.float16 else 0)


@pytest.mark.parametrize("dtype", [DType.float16, DType.float32], ids=lambda d: d.name)
@pytest.mark.parametrize("m,k,n", SHAPES, ids=str)
def test_against_float64(hip_backend, capfd, dtype, m, k, n):
    rng = np.random.default_rng(m * k + n)
    with hip_backend.use():
        for ta in (False, True):
            for tb in (False, True):
                for to in (False, True):
                    a = (rng.standard_normal((k, m) if ta else (m, k)) / np.sqrt(k)).astype(dtype.numpy)
                    b = rng.standard_normal((n, k) if tb else (k, n)).astype(dtype.numpy)
                    x, y = Tensor(data=a, dtype=dtype), Tensor(data=b, dtype=dtype)
                    a, b = (a.T if ta else a).astype(np.float64), (b.T if tb else b).astype(np.float64)
                    want, size = a @ b, np.abs(a) @ np.abs(b)
                    if to:
                        want, size = want.T, size.T
                    names = kernels_of(hip_backend, capfd, lambda: Tensor.matmul(x, ta, y, tb, to))
                    along = ("k" if tb else "m") + ("n" if ta else "k") if to else ("m" if ta else "k") + ("k" if tb else "n")
                    edge = "_e" if m % 64 or n % 64 or k % (128 // np.dtype(dtype.numpy).itemsize) else ""
                    in_parts = ["hc_gemm_%s_part_64x64_%s%s" % (SHORT[dtype], along, edge), "hc_gemm_part_sum_%s" % SHORT[dtype]]
                    rows, cols = (n, m) if to else (m, n)
                    whole = (rows, k, cols) in WHOLE[dtype] or (k < 4096 and (
                        along == "mn" and min(m, n) <= 16 if dtype == DType.float32 else along == "kn" and rows >= 640 and cols < 64))
                    assert (names == in_parts) == (not whole), (names, in_parts)
                    got = Tensor.matmul(x, ta, y, tb, to).numpy().astype(np.float64)
                    assert np.all(np.abs(got - want) <= error_bound(k, size, want, dtype)), (ta, tb, to, np.max(np.abs(got - want) / size))


# both sides of the rule's lines below K = 4096: fp32 with both operands along M and N and 16 or 17 columns; fp16 with A along K and B along N, 640 rows and 63
# columns, unless the rows start at odd halfs or the waves that split K are more than three quarters of the compute units
@pytest.mark.parametrize("dtype,m,k,n,ta,parts", [
    (DType.float32, 400, 4032, 16, True, False), (DType.float32, 400, 4096, 16, True, True), (DType.float32, 400, 4032, 17, True, True), (DType.float32, 400, 4032, 16, False, True),
    (DType.float32, 16, 4032, 400, True, False), (DType.float16, 640, 4032, 48, False, False), (DType.float16, 639, 4032, 48, False, True),
    (DType.float16, 640, 4096, 48, False, True), (DType.float16, 640, 4032, 64, False, True), (DType.float16, 640, 4031, 48, False, True),
    (DType.float16, 1552, 4032, 48, False, True), (DType.float16, 1536, 4032, 63, False, False), (DType.float16, 640, 4032, 48, True, True)], ids=str)
def test_short_products_of_few_columns(hip_backend, capfd, dtype, m, k, n, ta, parts):
    rng = np.random.default_rng(n)
    a, b = (rng.standard_normal((m, k)) / np.sqrt(k)).astype(dtype.numpy), rng.standard_normal((k, n)).astype(dtype.numpy)
    with hip_backend.use():
        x, y = Tensor(data=np.ascontiguousarray(a.T) if ta else a), Tensor(data=b)
        call = lambda: Tensor.matmul(x, ta, y, False, False)
        assert ("hc_gemm_part_sum_" + SHORT[dtype] in kernels_of(hip_backend, capfd, call)) == parts
        got = call().numpy().astype(np.float64)
    a, b = a.astype(np.float64), b.astype(np.float64)
    want = a @ b
    assert np.all(np.abs(got - want) <= error_bound(k, np.abs(a) @ np.abs(b), want, dtype))


@pytest.mark.parametrize("dtype", [DType.float16, DType.float32], ids=lambda d: d.name)
def test_operands_and_result_at_odd_elements(hip_backend, capfd, dtype):
    m, k, n, guard, es = 65, 3137, 80, 33, np.dtype(dtype.numpy).itemsize
    rng = np.random.default_rng(11)
    with hip_backend.use():
        for ta in (False, True):
            for tb in (False, True):
                a, b = (rng.standard_normal(shape).astype(dtype.numpy) for shape in ((k, m) if ta else (m, k), (n, k) if tb else (k, n)))
                around = lambda x: hip_backend.upload(np.concatenate([np.full(guard, np.nan, dtype.numpy), x.ravel(), np.full(guard, np.nan, dtype.numpy)]))
                x, y, out = around(a), around(b), around(np.zeros((m, n), dtype.numpy))
                at = lambda data: c_void_p(data.ptr + guard * es)
                call = lambda: hip_backend._check(hip_backend._lib.hc_matmul(hip_backend._ctx, dtype, 1, at(x), int(ta), at(y), int(tb), 0, m, k, n, at(out)))
                names = kernels_of(hip_backend, capfd, call)
                assert names[0] == "hc_gemm_%s_part_64x64_%s%s_e" % (SHORT[dtype], "m" if ta else "k", "k" if tb else "n"), names
                call()
                got = Tensor(dataHandle=out, shape=[m * n + 2 * guard], dtype=dtype).numpy().astype(np.float64)
                assert np.isnan(got[:guard]).all() and np.isnan(got[-guard:]).all()
                a, b = (a.T if ta else a).astype(np.float64), (b.T if tb else b).astype(np.float64)
                got, want = got[guard:-guard].reshape(m, n), a @ b
                assert np.all(np.abs(got - want) <= error_bound(k, np.abs(a) @ np.abs(b), want, dtype))


# a few rows, a few columns, both (the columns are too many tiles for parts, one launch), and both over operands that were copied to whole lines first
@pytest.mark.parametrize("dtype,m,k,n,parts,tb", [(DType.float16, 4104, 3200, 1024, "kn", False), (DType.float32, 4104, 4160, 1024, "kn", False),
                                                  (DType.float16, 1024, 3200, 4104, "kk", True), (DType.float16, 2061, 3072, 2056, "kn", False),
                                                  (DType.float16, 2061, 3201, 2053, "kk", True)], ids=str)
def test_fringes_in_parts(hip_backend, capfd, dtype, m, k, n, parts, tb):
    rng = np.random.default_rng(m + n)
    a, b = (rng.standard_normal((m, k)) / np.sqrt(k)).astype(dtype.numpy), rng.standard_normal((n, k) if tb else (k, n)).astype(dtype.numpy)
    with hip_backend.use():
        x, y = Tensor(data=a), Tensor(data=b)
        call = lambda: Tensor.matmul(x, False, y, tb, False)
        names = kernels_of(hip_backend, capfd, call)
        assert sum("_part_64x64_" + parts in name for name in names) == 1 and names.count("hc_gemm_part_sum_" + SHORT[dtype]) == 1, names
        assert ("hc_copy_lines_b2" in names) == (k % 2 == 1)
        got = call().numpy().astype(np.float64)
    a, b = a.astype(np.float64), (b.T if tb else b).astype(np.float64)
    want = a @ b
    assert np.all(np.abs(got - want) <= error_bound(k, np.abs(a) @ np.abs(b), want, dtype))


def same_bits(hip, fn):
    """fn() call by call, recorded (three replays) and batched."""
    bits = lambda t: t.numpy().view(np.uint8)
    want = [bits(t) for t in fn()]
    with hip.capture() as recording:
        outs = fn()
    for _ in range(3):
        recording.graph.launch()
        assert all(np.array_equal(bits(t), w) for t, w in zip(outs, want))
    recording.graph.destroy()
    with hip.batching():
        outs = fn()
    assert all(np.array_equal(bits(t), w) for t, w in zip(outs, want))


def test_a_recording_returns_the_bits_of_the_call(hip_backend):
    rng = np.random.default_rng(7)
    with hip_backend.use():
        x = Tensor(data=rng.standard_normal((48, 4100)).astype(np.float32), dtype=DType.float16)
        w = Tensor(data=(rng.standard_normal((4100, 300)) / 64).astype(np.float32), dtype=DType.float16)
        bias = Tensor(data=rng.standard_normal(300).astype(np.float32), dtype=DType.float16)
        same_bits(hip_backend, lambda: [(Tensor.matmul(x, False, w, False, False) + bias).gelu()])


# (whole and ragged tiles, a last part shorter than the others)
@pytest.mark.parametrize("dtype", [DType.float16, DType.float32], ids=lambda d: d.name)
@pytest.mark.parametrize("m,k,n", [(64, 3072, 768), (16, 4096, 1024), (13, 3208, 824)], ids=str)
def test_what_follows_is_merged_into_the_sum(hip_backend, capfd, dtype, m, k, n):
    rng = np.random.default_rng(m)
    tensor = lambda *shape, to=dtype: Tensor(data=rng.standard_normal(shape).astype(np.float32), dtype=to)
    with hip_backend.use():
        x, w, row, row2, rest = tensor(m, k), tensor(k, n), tensor(n), tensor(n), tensor(m, n)
        row32 = tensor(n, to=DType.float32)
        product = lambda: Tensor.matmul(x, False, w, False, False)
        for fn in (lambda: product() + row, lambda: (row + product()).gelu(), lambda: (product() + row) + rest, lambda: rest + product(),
                   lambda: ((product() + row) + rest) + row2, lambda: ((product() + row) + row2).gelu(), lambda: product().gelu(),
                   lambda: product() + row32.cast(dtype)):
            names = kernels_of(hip_backend, capfd, fn)
            assert len(names) == 2 and "_part_64x64_kn" in names[0] and names[1] == "hc_gemm_part_sum_%s_m" % names[0].split("_")[2], names
            same_bits(hip_backend, lambda: [fn()])
        # a result that the caller keeps is stored
        kept = []
        names = kernels_of(hip_backend, capfd, lambda: (kept.append(product()), kept[-1] + row))
        assert names[1] == "hc_gemm_part_sum_%s" % names[0].split("_")[2] and len(names) == 3
        del kept[:]


# (groups of two to four, and one more than a launch takes; at most as many parts of one tile, and few parts of many; fp16 above and at 128 tiles)
@pytest.mark.parametrize("dtype", [DType.float16, DType.float32], ids=lambda d: d.name)
@pytest.mark.parametrize("m,k,n,count", [(64, 3072, 768, 3), (16, 4096, 1024, 2), (13, 3208, 824, 5), (64, 4160, 64, 4), (300, 3072, 768, 3), (300, 3080, 840, 2), (64, 3072, 4096, 2),
                                       (512, 5064, 1024, 4)], ids=str)
def test_products_over_one_input_share_their_launches(hip_backend, capfd, dtype, m, k, n, count):
    rng = np.random.default_rng(m)
    tensor = lambda *shape: Tensor(data=rng.standard_normal(shape).astype(np.float32), dtype=dtype)
    with hip_backend.use():
        x, ws, rows = tensor(m, k), [tensor(k, n) for _ in range(count)], [tensor(n) for _ in range(count)]
        if "hc_gemm_part_sum_%s" % SHORT[dtype] not in kernels_of(
                hip_backend, capfd, lambda: Tensor.matmul(x, False, ws[0], False, False)):
            assert dtype == DType.float32 and m * n > 200000      # (longer chains than those of a workgroup's waves)
            return
        chain = dtype == DType.float16 and 2 * count * -(-m // 64) * -(-n // 64) > 256
        for fn in (lambda: [Tensor.matmul(x, False, w, False, False) for w in ws],
                   lambda: [Tensor.matmul(x, False, w, False, False) + row for w, row in zip(ws, rows)]):
            names = kernels_of(hip_backend, capfd, fn)
            assert len(names) == (1 if chain else 2 if count <= 4 else 4) and ("_chain_" in names[0]) == chain, names
            same_bits(hip_backend, fn)

        def used_between():
            first = Tensor.matmul(x, False, ws[0], False, False)
            return [first.exp(), Tensor.matmul(x, False, ws[1], False, False), first]

        assert len(kernels_of(hip_backend, capfd, used_between)) == 5
        same_bits(hip_backend, used_between)


@pytest.mark.parametrize("m,k,n", [(64, 3072, 768), (300, 3072, 768)], ids=str)
@pytest.mark.parametrize("which", [0, 1])
def test_an_operand_may_change_behind_its_product(hip_backend, m, k, n, which):
    """The parts are moved next to those of the other member, or next to their sum, only as far as what they read stays as it was."""
    rng = np.random.default_rng(m)
    tensor = lambda *shape: Tensor(data=rng.standard_normal(shape).astype(np.float32), dtype=DType.float16)
    with hip_backend.use():
        x, ws, row = tensor(m, k), [tensor(k, n) for _ in range(2)], tensor(n)
        fill = lambda w, v: hip_backend._check(hip_backend._lib.hc_fill(hip_backend._ctx, DType.float16, v, 0, w.data.ptr, k * n))

        def program():
            fill(ws[0], 0.25), fill(ws[1], 0.5)
            products = [Tensor.matmul(x, False, w, False, False) for w in ws]
            fill(ws[which], 2.0)
            return [y + row for y in products]

        same_bits(hip_backend, program)


@pytest.mark.parametrize("m,k,n", [(64, 3072, 768), (300, 3072, 768)], ids=str)
def test_sums_in_another_order_than_their_parts(hip_backend, capfd, m, k, n):
    """The second product's bias comes last, and what the third multiplies with is made between the two."""
    rng = np.random.default_rng(m)
    tensor = lambda *shape: Tensor(data=rng.standard_normal(shape).astype(np.float32), dtype=DType.float16)
    with hip_backend.use():
        x, ws, row = tensor(m, k), [tensor(k, n) for _ in range(3)], tensor(n)

        def program():
            a, b = (Tensor.matmul(x, False, w, False, False) for w in ws[:2])
            c = Tensor.matmul(x, False, ws[2] * ws[0], False, False)
            return [t + row for t in (a, c, b)]

        assert len(kernels_of(hip_backend, capfd, program)) == (2 if m == 300 else 3)
        same_bits(hip_backend, program)


def test_a_recording_shares_the_blocks_of_partial_sums(hip_backend):
    """Forty products whose sums take 768 KiB each in a recording, what follows them merged in all orders: at most nine blocks, and the bits of the calls."""
    m, k, n, count = 64, 3072, 256, 40
    rng = np.random.default_rng(3)
    tensor = lambda *shape: Tensor(data=rng.standard_normal(shape).astype(np.float32), dtype=DType.float16)
    with hip_backend.use():
        xs, w, row = [tensor(m, k) for _ in range(count)], tensor(k, n), tensor(n)

        def program():
            late = [Tensor.matmul(x, False, w, False, False) for x in xs[:20]]     # (their bias comes when the blocks have been used again)
            return [Tensor.matmul(x, False, w, False, False) + row for x in xs[20:]] + [y + row for y in late]

        same_bits(hip_backend, program)
        hip_backend.sync()
        assert hip_backend._lib.hc_trim(hip_backend._ctx) == 0
        with hip_backend.capture() as recording:
            outs = program()
        del outs
        recording.graph.destroy()
        held = hip_backend.memStats()[1]      # what the recording had: the sums, and 32 KiB for every product and every addition
        assert held <= 9 * (1 << 20) + 2 * count * (32 << 10), held


@pytest.mark.parametrize("dtype", [DType.float16, DType.float32], ids=lambda d: d.name)
def test_an_infinity_or_a_nan_stays_in_its_row_and_column(hip_backend, dtype):
    m, k, n = 70, 3100, 66
    a, b = np.ones((m, k), np.float32), np.ones((k, n), np.float32)
    a[3, 3099], a[69, 0], b[1024, 65] = np.inf, np.nan, -np.inf
    with hip_backend.use(), np.errstate(invalid="ignore"):
        got = Tensor.matmul(Tensor(data=a, dtype=dtype), False, Tensor(data=b, dtype=dtype), False, False).numpy()
        np.testing.assert_array_equal(got, (a.astype(np.float64) @ b.astype(np.float64)).astype(dtype.numpy))
