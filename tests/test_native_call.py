"""vkblas_amd._call.gemm_ex (csrc/pycall.c) hands a function the same values as
the ctypes prototype of vkblas_gemm_ex_async does, for the values at the ends of
each type and past them, and declines (None) what it does not convert itself."""
import ctypes

import pytest

import vkblas_amd as vk

L = vk.load()
PROTO = ctypes.CFUNCTYPE(ctypes.c_int, *L.vkblas_gemm_ex_async.argtypes)


def _receive():
    got = []

    def fn(*a):
        ep = a[-2]
        got.append([float(x) if isinstance(x, float) else x for x in a[:-2]] +
                   [[getattr(ep[0], f) for f, _ in vk.Epilogue._fields_] if ep else None, a[-1]])
        return -7
    return PROTO(fn), got


INTS = [0, 1, 2**31 - 1, 2**31, 2**32 - 1, 2**32 + 5, -1, -2**31, 2**63 - 1, -2**63, 2**64 - 1]


@pytest.mark.parametrize("value", INTS)
def test_same_values_as_ctypes(value):
    cb, got = _receive()
    addr = ctypes.cast(cb, ctypes.c_void_p).value
    for scal in (1.5, -0.0, 1e-60, 3, float("inf")):
        head = [value] * 7 + [scal, value, value, None, value, scal, value] + [value] * 5 + [value, None, value, value]
        ep = (value, value, value, None, value)
        assert vk._native(addr, *head, 1, *ep, value) == -7
        assert cb(*head, ctypes.byref(vk.Epilogue(*ep)), value) == -7
        assert got[-1] == got[-2]
        assert vk._native(addr, *head, 0, None, 0, 0, None, 0, None) == -7
        assert cb(*head, None, None) == -7
        assert got[-1] == got[-2]


def test_declines_what_ctypes_converts_itself():
    cb, got = _receive()
    addr = ctypes.cast(cb, ctypes.c_void_p).value
    head = [0, 0, 0, 1, 4, 4, 4, 1.0, 64, 4, 64, 4, 0.0, 64, 4, 1, 0, 0, 0, 0, None, None, 0]
    tail = [0, None, 0, 0, None, 0, None]
    for i, bad in ((4, True), (4, 4.0), (7, "1"), (8, ctypes.c_void_p(64)), (8, b"x"), (13, "x"), (7, 10**400)):
        a = list(head)
        a[i] = bad
        assert vk._native(addr, *a, *tail) is None
    assert got == []
    with pytest.raises(TypeError):
        vk._native(addr, *head)
    with pytest.raises(ValueError):
        vk._native(0, *head, *tail)
    # through the binding: the ctypes rules, as before
    with pytest.raises(ctypes.ArgumentError):
        vk.gemm_async(0, 0, 0, 1, 4.0, 4, 4, 1.0, 64, 4, 64, 4, 0.0, 64, 4)
    assert vk.gemm_async(0, 0, 0, 1, 0, 4, 4, 1.0, ctypes.c_void_p(64), 4, 64, 4, 0.0, 64, 4, check=False) == vk.ERR_PARAM
