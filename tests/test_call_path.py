"""The native call path (csrc/lh_py.cpp) against ctypes: the same values arrive for ordinary arguments, the same objects are refused."""
import copy
import ctypes as C
import gc
import shutil
import subprocess
import weakref

import numpy as np
import pytest

from lantern_amd import _lib
from lantern_amd import backend as B
from lantern_amd.tensor import Tensor, TensorR

P, I, F, L, Z = _lib.P, _lib.I, _lib.F, _lib.L, _lib.Z
SOURCE = """
#include <stdint.h>
#include <stddef.h>
#include <string.h>
unsigned char out[64];
static size_t at;
#define PUT(x) memcpy(out + at, &x, sizeof x); at += sizeof x
void f0(int op, void* x, void* y, int64_t n, float lo, float hi) { at = 0; PUT(op); PUT(x); PUT(y); PUT(n); PUT(lo); PUT(hi); }
void f1(void* a, size_t b) { at = 0; PUT(a); PUT(b); }
void* f2(size_t n) { return (void*)n; }
size_t f3(void) { return ~(size_t)0; }
"""


@pytest.mark.skipif(_lib._lhpy is None or shutil.which("gcc") is None, reason="needs the native module and a C compiler")
def test_arguments_arrive_as_through_ctypes(tmp_path):
    (tmp_path / "f.c").write_text(SOURCE)
    so = str(tmp_path / "f.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", so, str(tmp_path / "f.c")], check=True)
    lib = C.CDLL(so)
    out = (C.c_ubyte * 64).in_dll(lib, "out")
    ints = (C.c_int * 3)(1, 2, 3)
    forms = {"f0": ("vIPPLFF", None, [I, P, P, L, F, F]), "f2": ("PZ", P, [Z]), "f3": ("Z", Z, [])}
    calls = [("f0", a) for a in [(1, 2 ** 63 + 5, None, -7, 0.1, 3), (-1, ints, C.byref(ints), 2 ** 40, -1e300, 1e-300), (2 ** 32 + 3, -1, 0, 2 ** 70, float("nan"), True),
                                 (True, b"abc", C.c_void_p(77), 1, np.float64(0.3), np.float32(0.3)), (np.int64(3), 1, 1, 1, 0.0, 0.0), (1.0, 1, 1, 1, 0.0, 0.0),
                                 (1, 1.5, 1, 1, 0.0, 0.0), (1, "text", 1, 1, 0.0, 0.0), (1, 1, 1, 1, "x", 0.0), (1, 1, 1, 1, 10 ** 400, 0.0), (1, 2), (1,) * 9,
                                 (1, np.zeros(3), 1, 1, 0.0, 0.0), (1, [1], 1, 1, 0.0, 0.0)]] + [("f2", (0,)), ("f2", (12345,)), ("f2", (-1,)), ("f2", (None,)), ("f3", ())]

    def result(fn, args):
        C.memset(out, 0, 64)
        try:
            return fn(*args), bytes(out)
        except Exception as e:          # noqa: BLE001
            return type(e), str(e)
    for name, args in calls:
        letters, res, types = forms[name]
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = res, types
        native = _lib._lhpy.call(letters, C.cast(fn, P).value, fn)
        assert native is not fn and native.argtypes == types
        assert result(native, args) == result(fn, args), (name, args)
    fn = lib.f1
    assert _lib._lhpy.call("vPZZZZZZZZZ", 1, fn) is fn        # no such form: ctypes stays


@pytest.mark.parametrize("cls", [B.PyBuf, B.Buf])
def test_handles(cls):
    b = cls(np.int64(4096), 10, keep="owner")
    assert (type(b.ptr), b.ptr, b.n, b.keep) == (int, 4096, 10, "owner")
    o, p = b.offset(np.int64(3)), b.offset(2, 4)
    assert (o.ptr, o.n, o.keep, p.ptr, p.n) == (4108, 7, "owner", 4104, 4) and cls(1, 2).keep is None
    b.ptr = 8
    assert b.offset(1).ptr == 12
    for bad in ((), (1,), (1, 2, 3, 4), ("x", 2)):
        with pytest.raises((TypeError, ValueError)):
            cls(*bad)
    with pytest.raises(AttributeError):
        b.other = 1


@pytest.mark.parametrize("cls", [B.PyBuf, B.Buf])
def test_an_owner_that_holds_its_handle_is_collected(cls):
    class Owner:
        pass

    class Derived(cls):
        pass
    for kind in (cls, Derived):
        o = Owner()
        o.buf = kind(4096, 10, o).offset(1)
        assert isinstance(o.buf, (B.PyBuf, B.Buf)) and o.buf.keep is o
        o.direct = kind(4096, 10, o)
        gone = weakref.ref(o)
        del o
        gc.collect()
        assert gone() is None
    b = cls(4096, 10, keep=[1])
    c = copy.copy(b)
    assert (c.ptr, c.n, c.keep) == (4096, 10, [1]) and isinstance(b, cls) and isinstance(c, cls)
    for _ in range(1000):
        cls(1, 2, [b])
    gc.collect()


def test_tensors_still_take_attributes():
    t = Tensor(B.Buf(4096, 6), (2, 3))
    t.name = "weights"
    r = TensorR(t, t)
    r.tag = 1
    assert (t.name, r.tag, t.shape, t.scalarCount, t.rank) == ("weights", 1, (2, 3), 6, 2)
