"""The C ABI without a GPU: the library loads, exports every function that
include/faces_amd.h declares, and rejects invalid arguments before touching
the device."""
from __future__ import annotations

import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "faces_amd.h")
LIB = os.path.join(ROOT, "faces_amd", "lib", "libfaces_amd.so")

needs_lib = pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")


def declared():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(faces_[a-z0-9_]+)\s*\(", text)))


@pytest.fixture(scope="module")
def lib():
    import torch  # noqa: F401  (one HIP runtime for the process)
    return ctypes.CDLL(LIB)


def test_header_declares_the_plain_step():
    names = declared()
    for must in ["faces_plan_create", "faces_plan_destroy", "faces_share", "faces_strerror",
                 "faces_batch_create", "faces_batch_share", "faces_server_create",
                 "faces_server_submit", "faces_server_wait"]:
        assert must in names


@needs_lib
def test_every_declared_symbol_is_exported(lib):
    missing = [n for n in declared() if not hasattr(lib, n)]
    assert not missing, missing


@needs_lib
def test_strerror_and_version(lib):
    lib.faces_strerror.restype = ctypes.c_char_p
    lib.faces_version.restype = ctypes.c_char_p
    assert lib.faces_strerror(0) == b"ok" or lib.faces_strerror(0)
    for st in range(-7, 0):
        assert lib.faces_strerror(st)
    assert lib.faces_version()


@needs_lib
def test_plan_create_rejects_bad_arguments(lib):
    vp = ctypes.c_void_p()
    f = lib.faces_plan_create
    f.argtypes = [ctypes.POINTER(ctypes.c_void_p)] + [ctypes.c_int] * 9 + [ctypes.c_long]
    lib.faces_last_error.restype = ctypes.c_char_p
    cases = [(0, 1, 1, 1, 4, 4, 4, 1, 1, 0),     # n = 1
             (0, 1, 1, 1, 0, 4, 4, 5, 1, 0),     # mx = 0
             (4, 2, 1, 1, 4, 4, 4, 5, 1, 0),     # rank outside the grid
             (0, 1, 1, 1, 4, 4, 4, 5, 7, 0),     # unknown boundary
             (0, 0, 1, 1, 4, 4, 4, 5, 1, 0)]     # empty rank grid
    for c in cases:
        st = f(ctypes.byref(vp), *c, 0)
        assert st == -1, (c, st)
        assert lib.faces_last_error()
    assert f(None, 0, 1, 1, 1, 4, 4, 4, 5, 1, 0) == -1


@needs_lib
def test_field_doubles(lib):
    lib.faces_field_doubles.restype = ctypes.c_long
    lib.faces_field_doubles.argtypes = [ctypes.c_int] * 4 + [ctypes.c_long]
    assert lib.faces_field_doubles(5, 4, 4, 4, 0) == 8000
    assert lib.faces_field_doubles(7, 60, 60, 60, 0) == 74088000
    # padded planes: (mz - 1) strides plus one dense plane
    assert lib.faces_field_doubles(5, 4, 4, 4, 2048) == 3 * 2048 + 2000


@needs_lib
def test_batch_and_server_reject_bad_arguments(lib):
    vp = ctypes.c_void_p()
    ints = (ctypes.c_int * 1)
    lib.faces_batch_create.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_int] + \
        [ctypes.POINTER(ctypes.c_int)] * 4 + [ctypes.c_int]
    assert lib.faces_batch_create(ctypes.byref(vp), 0, ints(4), ints(2), ints(2), ints(2), 1) == -1
    assert lib.faces_batch_create(ctypes.byref(vp), 1, ints(1), ints(2), ints(2), ints(2), 1) == -1
    assert lib.faces_batch_create(ctypes.byref(vp), 1, ints(4), ints(2), ints(2), ints(2), 9) == -1
    lib.faces_server_create.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_double,
                                        ctypes.c_int, ctypes.c_int]
    assert lib.faces_server_create(ctypes.byref(vp), 0.0, 4, 1) == -1
    assert lib.faces_server_create(ctypes.byref(vp), 1e9, 0, 1) == -1
    assert lib.faces_server_create(ctypes.byref(vp), 1e9, 4, 0) == -1
    assert lib.faces_batch_share(None, 1, None) == -1
    assert lib.faces_share(None, None, 1, None) == -1


class _Tensor:
    """What the binding asks of a tensor before it takes its address."""

    def __init__(self, count):
        import torch
        self.dtype, self.is_cuda, self.count = torch.float64, True, count

    def is_contiguous(self):
        return True

    def numel(self):
        return self.count

    def data_ptr(self):
        return 1 << 20


@needs_lib
@pytest.mark.parametrize("kind", ["int", "int16", "int32", "int64"])
@pytest.mark.parametrize("shape", [(8, 10, 10, 10), (8, 400, 400, 400), (8, 2 ** 32 + 4, 4, 4)])
def test_submit_refuses_a_short_tensor_whatever_the_integers(kind, shape):
    """8x10x10x10 is beyond 16-bit, 8x400x400x400 beyond 32-bit integers, and 2^32 + 4 is the C int 4: the tensor one
    double short of the field is refused before its address is used, the whole one gets as far as the library, which
    refuses the null server."""
    import numpy as np

    import faces_amd as fa
    make = int if kind == "int" else getattr(np, kind)
    if shape[1] > 2 ** 31 and kind in ("int16", "int32"):
        pytest.skip("not a value of this type")
    args = [make(x) for x in shape]
    server = object.__new__(fa.Server)
    server._h = None
    need = shape[0] ** 3 * (shape[1] % 2 ** 32) * shape[2] * shape[3]
    with pytest.raises(fa.FacesError, match="elements, the field needs"):
        server.submit(_Tensor(need - 1), *args)
    with pytest.raises(fa.FacesError, match="null argument"):
        server.submit(_Tensor(need), *args)
