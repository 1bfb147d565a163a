"""vkblas_amd._call.gemm_ex (csrc/pycall.c) hands a function the same values as
the ctypes prototype of vkblas_gemm_ex_async does, for the values at the ends of
each type and past them, and declines (None) what it does not convert itself; and
the binding and the library do without it."""
import ctypes
import os
import subprocess
import sys
import sysconfig

import pytest

import vkblas_amd as vk

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
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


def _child(code):
    env = dict(os.environ, PYTHONPATH=REPO)
    return subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=120)


def test_without_the_module():
    """An interpreter that cannot import the module makes every call through ctypes."""
    r = _child("import sys; sys.modules['vkblas_amd._call'] = None\n"
               "import vkblas_amd as vk\n"
               "a = (0, 0, 0, 1, 0, 4, 4, 1.0, 64, 4, 64, 4, 0.0, 64, 4)\n"
               "assert vk.gemm_async(*a, check=False) == vk.ERR_PARAM\n"
               "assert vk.gemm_ex_async(*a, check=False) == vk.ERR_PARAM\n"
               "print('ctypes ok')")
    assert r.returncode == 0 and "ctypes ok" in r.stdout, r.stderr[-2000:]


def test_module_is_tagged_for_its_interpreter():
    """Another interpreter never opens it: its file name carries this one's ABI tag."""
    import vkblas_amd._call as m
    assert os.path.basename(m.__file__) == "_call" + sysconfig.get_config_var("EXT_SUFFIX")


def test_library_builds_without_python_headers():
    r = subprocess.run(["make", "-n", "-B", "-C", os.path.join(REPO, "vkblas_amd"), "PYINC=/nonexistent", "all"],
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "libvkblas_hipblas.so" in r.stdout, r.stderr[-2000:]
    assert "pycall" not in r.stdout
