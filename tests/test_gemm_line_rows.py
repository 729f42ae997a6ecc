"""Large fp16 products along K whose rows start at odd halfs, copied to rows of whole cache lines first: the ends of K, ragged sides, fringes."""
import numpy as np
import pytest

from honeycrisp_amd.descriptors import DType
from honeycrisp_amd.tensor import Tensor
from recorded_kernels import kernels_of

pytestmark = pytest.mark.gpu


def operands(m, k, n):
    rng = np.random.default_rng(m + k + n)
    return (rng.standard_normal((m, k)) / np.sqrt(k)).astype(np.float16), rng.standard_normal((n, k)).astype(np.float16)


# K one past and one short of a whole line, and whole dwords; a side of one tile more; a result whose rows are aligned; a peeled column
@pytest.mark.parametrize("m,k,n,to", [(897, 8065, 901, False), (896, 8063, 904, False), (904, 8070, 1025, True), (1024, 3073, 2049, False)], ids=str)
def test_against_float64(hip_backend, capfd, m, k, n, to):
    a, b = operands(m, k, n)
    with hip_backend.use():
        x, y = Tensor(data=a), Tensor(data=b)
        call = lambda: Tensor.matmul(y, False, x, True, False) if to else Tensor.matmul(x, False, y, True, False)
        assert kernels_of(hip_backend, capfd, call)[0] == "hc_copy_lines_b2"
        got = call().numpy().astype(np.float64)
        with hip_backend.capture() as recording:
            out = call()
        for _ in range(2):
            recording.graph.launch()
            np.testing.assert_array_equal(out.numpy(), got.astype(np.float16))
    got = got.T if to else got
    a, b = a.astype(np.float64), b.T.astype(np.float64)
    exact = a @ b
    # k roundings of fp32 partial sums, one to the result's type
    assert np.all(np.abs(got - exact) <= k * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + 2.0 ** -11 * np.abs(exact) + 2.0 ** -24)


def test_what_follows_a_row_is_not_multiplied(hip_backend):
    """The copies end in zeros: an infinity in the first element of a row does not reach the row in front of it."""
    m, k, n = 900, 8001, 900
    a, b = np.ones((m, k), np.float16), np.ones((n, k), np.float16)
    a[5, 0], b[7, 0], a[9, k - 1] = np.inf, np.nan, -np.inf
    with hip_backend.use():
        got = Tensor.matmul(Tensor(data=a), False, Tensor(data=b), True, False).numpy()
    want = np.full((m, n), 8000.0, np.float16)     # (8001 rounds to 8000 in fp16)
    want[5], want[9], want[:, 7] = np.inf, -np.inf, np.nan
    np.testing.assert_array_equal(got, want)


def test_a_recording_shares_the_copies(hip_backend):
    """Six products whose operands are copied to rows of whole lines, 14 MiB each: one pair of copies in a recording, and the bits of the calls."""
    m, k, n, count = 900, 8001, 900, 6
    a, b = operands(m, k, n)
    with hip_backend.use():
        xs, y = [Tensor(data=np.roll(a, i, axis=0)) for i in range(count)], Tensor(data=b)
        program = lambda: [Tensor.matmul(x, False, y, True, False) for x in xs]
        want = [t.numpy() for t in program()]
        hip_backend.sync()
        assert hip_backend._lib.hc_trim(hip_backend._ctx) == 0
        with hip_backend.capture() as recording:
            outs = program()
        for _ in range(2):
            recording.graph.launch()
            assert all(np.array_equal(t.numpy(), v) for t, v in zip(outs, want))
        del outs
        recording.graph.destroy()
        held = hip_backend.memStats()[1]
        assert held <= 2 * (14 << 20) + count * (2 << 20), held
