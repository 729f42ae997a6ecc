"""honeycrisp_amd._native against a stand-in library that counts its blocks and notes what it was called with (no GPU)."""
import ctypes
import gc
import os
import subprocess
import sysconfig
import weakref

import numpy as np
import pytest

from honeycrisp_amd import backend as backend_module
from honeycrisp_amd.csrc import build
from honeycrisp_amd.descriptors import BroadcastStrides, DType

native = pytest.importorskip("honeycrisp_amd._native")

TYPED = r"""
#include <stdlib.h>
#include "hchip.h"
int live, calls, fail, locked; long long seen[16]; hc_strides shape;
int PyGILState_Check(void);
int hc_malloc(hc_ctx* c, size_t n, void** p) { if (!c) return HC_ERR_INVALID; if (fail == 2 && live) return HC_ERR_ALLOC; *p = malloc(1); live++; return 0; }
int hc_free(hc_ctx* c, void* p) { locked += PyGILState_Check(); free(p); live--; return 0; }
int hc_binary_op(hc_ctx* c, int op, int t, const void* a, const hc_strides* sa, const void* b, const hc_strides* sb, void* o) {
  seen[0] = op; seen[1] = t; seen[2] = (long long)a; seen[3] = (long long)b; shape = *sa; calls++; return fail ? HC_ERR_UNSUPPORTED : 0; }
int hc_matmul(hc_ctx* c, int t, int64_t n, const void* a, int ta, const void* b, int tb, int to, int64_t rows, int64_t inner, int64_t cols, void* o) {
  seen[0] = ta; seen[1] = tb; seen[2] = to; seen[3] = rows; seen[4] = inner; seen[5] = cols; calls++; return fail ? 4 : 0; }
int hc_fill(hc_ctx* c, int t, float f, int64_t i, void* o, size_t n) { seen[0] = t; seen[1] = (long long)(f * 4); seen[2] = i; seen[3] = n; calls++; return 0; }
"""
# (without the header: they do not read their arguments)
COUNTED = "extern int calls, fail;\n" + "".join("int %s() { calls++; return fail ? 4 : 0; }\n" % name for name in (
    "hc_binary_op_scalar hc_mul_add hc_add_mul hc_when hc_cast hc_pow hc_elemwise hc_reduce hc_cumulative hc_argsort hc_log_softmax "
    "hc_log_softmax_grad hc_normalize hc_gather hc_scatter hc_adamw hc_broadcast").split())


class Refused(Exception):
    pass


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    folder = tmp_path_factory.mktemp("native")
    path, include = str(folder / "libstand_in.so"), os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include")
    (folder / "typed.c").write_text(TYPED)
    (folder / "counted.c").write_text(COUNTED)
    subprocess.run(["gcc", "-shared", "-fPIC", "-I" + include, str(folder / "typed.c"), str(folder / "counted.c"), "-o", path], check=True)
    found = ctypes.CDLL(path)
    found.path = path
    return found


@pytest.fixture
def fake(lib):
    class Data(native.Data):
        pass

    class Fake:
        def _dev(self, data):
            self.uploaded = data
            return self.made(16)

        def _raise(self, status):
            raise Refused(status, value(lib, "live"))

        def made(self, n):
            return self._native.alloc(self, n)

    f = Fake()
    f._native = native.Context(lib.path, 4096, Data)
    f.Data = Data
    for name in ("live", "calls", "fail", "locked"):
        ctypes.c_int.in_dll(lib, name).value = 0
    return f


def value(lib, name):
    return ctypes.c_int.in_dll(lib, name).value


def seen(lib, n):
    return list((ctypes.c_longlong * 16).in_dll(lib, "seen"))[:n]


def test_a_result_is_sized_described_and_given_back(lib, fake):
    x, y = fake.made(24), fake.made(24)
    out = fake._native.binary(fake, np.int64(3), DType.float16, x, BroadcastStrides([2, 3], [3, 1]), y, BroadcastStrides([2, 3], [0, 1]))
    assert type(out) is fake.Data and out.backend is fake and out.byteCount == 12 and out.ptr
    assert seen(lib, 4) == [3, 2, x.ptr, y.ptr]
    shape = (ctypes.c_longlong * 17).in_dll(lib, "shape")
    assert (shape[0], shape[1], shape[2], shape[9], shape[10]) == (2, 2, 3, 3, 1) and not any(shape[3:9])
    assert value(lib, "live") == 3
    keep = weakref.ref(out)
    out.note, out.self = "own attributes", out
    del out
    gc.collect()
    assert keep() is None and value(lib, "live") == 2
    fake._native.fill(fake, DType.int64, 0.5, ctypes.c_int64(-7), 5)
    assert seen(lib, 4) == [0, 2, -7, 5] and value(lib, "live") == 2
    del x, y
    assert value(lib, "live") == 0


def test_a_refused_call_gives_its_results_back(lib, fake):
    x = fake.made(8)
    dense = BroadcastStrides([2], [1])
    ctypes.c_int.in_dll(lib, "fail").value = 1
    for call in (lambda: fake._native.binary(fake, 0, 3, x, dense, x, dense),
                 lambda: fake._native.adamw(fake, 3, x, x, x, x, 1, 1, 1, 1, 1, 1, 2)):
        with pytest.raises(Refused) as e:
            call()
        assert e.value.args[0] == 4 and e.value.args[1] > 1 and value(lib, "live") == 1     # (reported before the blocks go)
    ctypes.c_int.in_dll(lib, "fail").value = 2
    with pytest.raises(Refused):
        fake._native.adamw(fake, 3, x, x, x, x, 1, 1, 1, 1, 1, 1, 2)
    assert value(lib, "live") == 1
    del x
    assert value(lib, "locked") == 0    # (the library may wait for the device, and that for a host function in Python)


def test_what_is_no_argument_is_refused_before_the_library_sees_it(lib, fake):
    x = fake.made(8)
    dense, nine = BroadcastStrides([2], [1]), BroadcastStrides([1] * 9, [1] * 9)
    for error, call in ((ValueError, lambda: fake._native.broadcast(fake, 3, x, nine)),
                        (ValueError, lambda: fake._native.broadcast(fake, 7, x, dense)),
                        (TypeError, lambda: fake._native.broadcast(fake, 3, x)),
                        (TypeError, lambda: fake._native.cast(fake, x, 2.5, 3, 2)),
                        (TypeError, lambda: fake._native.normalize(fake, 3, x, 1, 2, 1, "eps")),
                        (AttributeError, lambda: fake._native.broadcast(fake, 3, x, None))):
        with pytest.raises(error):
            call()
    assert value(lib, "calls") == 0 and value(lib, "live") == 1


@pytest.mark.filterwarnings("error")
def test_flags_may_be_numbers_of_any_kind(lib, fake):
    x = fake.made(8)
    hip = backend_module.HIPBackend.__new__(backend_module.HIPBackend)
    hip._ctx, hip._native, hip._dev = None, fake._native, lambda data: data
    dims = backend_module.ReduceDims(2, 3, 1)
    hip.matmul(x, np.bool_(True), x, 0.0, np.bool_(False), 2, 3, 4, DType.float16)
    assert seen(lib, 6) == [1, 0, 0, 2, 3, 4]
    hip.batchedMatmul(1, x, 0, x, np.True_, 1, 2, 3, 4, DType.float16)
    assert seen(lib, 3) == [0, 1, 1]
    with pytest.raises(TypeError):
        hip.matmul(x, None, x, False, False, 2, 3, 4, DType.float16)
    hip.argsort(x, dims, np.bool_(True), np.bool_(True), DType.float16)
    hip.cumulativeSum(x, dims, np.bool_(True), 0.0, DType.float16)


def test_other_data_goes_through_the_backend(lib, fake):
    class Derived(fake.Data):
        pass

    for foreign in (b"bytes", Derived(fake, None, 4), fake.Data(object(), None, 4), np.zeros(4)):
        fake._native.elemwise(fake, 0, 3, foreign, None, 2)
        assert fake.uploaded is foreign
    fake._native.elemwise(fake, 0, 3, fake.made(8), fake.made(8), 2)
    assert value(lib, "calls") == 5 and value(lib, "live") == 0


def test_after_close_nothing_is_called_or_given_back(lib, fake):
    x = fake.made(8)
    fake._native.close()
    with pytest.raises(Refused) as e:
        fake.made(8)
    assert e.value.args[0] == 1
    del x
    assert value(lib, "live") == 1


def test_sizes_past_the_range_are_more_than_there_is(lib, fake):
    x = fake.made(8)
    out = fake._native.reduce(fake, 0, 3, 3, x, 1 << 40, 1, 1 << 40)
    assert out.byteCount == 2 ** 63 - 1
    assert fake._native.log_softmax(fake, 3, x, 1 << 40, 1 << 40, 0).byteCount == 0


def test_the_backend_says_what_is_missing(monkeypatch):
    monkeypatch.setattr(backend_module, "_native", None)
    with pytest.raises(ImportError, match="_native"):
        backend_module.HIPBackend()


def test_a_library_without_the_calls_leaves_no_context_behind(monkeypatch):
    class Library:
        shut = []

        def hc_init(self, device, out):
            out._obj.value = 4096
            return 0

        def hc_shutdown(self, ctx):
            self.shut.append(ctx.value)

    monkeypatch.setattr(backend_module._lib, "load", Library)
    monkeypatch.setattr(backend_module._lib, "LIB_PATH", "libc.so.6")
    with pytest.raises(ImportError, match="hc_malloc"):
        backend_module.HIPBackend()
    assert Library.shut == [4096]


def test_the_extension_is_built_last_and_for_one_python(monkeypatch):
    """What needs neither Python's headers nor gcc does not fail with it, and another Python does not take it for its own."""
    outputs = []
    monkeypatch.setattr(build, "_run", lambda command: outputs.append(command[command.index("-o") + 1]))
    monkeypatch.setattr(build, "build_kernel", lambda name, source, flags: name)
    build.build_all(verbose=False)
    assert os.path.basename(outputs[-1]) == "_native" + sysconfig.get_config_var("EXT_SUFFIX")
    assert os.path.basename(outputs[-2]) == "HCMatrixBench"
