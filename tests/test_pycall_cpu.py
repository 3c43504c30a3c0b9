"""The native calls against ctypes: what either takes, refuses and answers, without a device (every call ends in a refusal of
its sizes or pointers)."""
import ctypes as C
import os
import subprocess
import sys
import sysconfig

import pytest


class Pointer:
    def __init__(self, value):
        self.value = value

    def data_ptr(self):
        if isinstance(self.value, Exception):
            raise self.value
        return self.value


class Number(int):
    pass


POINTERS = [0, 4096, None, Pointer(4096), Pointer(0), True, Number(4096), -16, 1 << 70, Pointer(1 << 70), C.c_void_p(4096),
            1.5, "x", Pointer(1.5), Pointer(RuntimeError("no storage")), Pointer(None), object()]
SIZES = [0, -1, 127, 1 << 40, (1 << 32) + 0, True, Number(0), 2.0, None, "8", C.c_int(0)]
STREAMS = [0, None, 16, True, 1.5, Pointer(0), object()]


def outcome(f, *args):
    try:
        return "ok", f(*args)
    except Exception as e:  # noqa: BLE001  both sides' exceptions are what is compared
        return type(e), getattr(e, "code", None), str(e)


def through_ctypes(pkg, monkeypatch, f, *args):
    class Nothing:
        gemm = gemm_ex = quantize_a = quantize_b = staticmethod(lambda *a: None)
    with monkeypatch.context() as m:
        m.setitem(f.__globals__, "_CALL", Nothing)
        return outcome(f, *args)


@pytest.mark.parametrize("position", range(13))
def test_gemm_ex_and_gemm(pkg, monkeypatch, position):
    ws_bytes = [0, 5, -1, 1 << 70, 2.0, None]
    options = [None, pkg.Options(), pkg.Options(kernel=9), C.c_int(3), object(), 0]
    values = [POINTERS] * 5 + [SIZES] * 3 + [options, POINTERS, ws_bytes, STREAMS]
    base = [4096, 4096, 4096, 4096, 4096, 16, 16, 100, None, None, 0, None]   # k is no multiple of 128
    if position == 12:
        assert outcome(pkg.gemm_ex, *base) == (pkg.Fp8GemmError, -2, outcome(pkg.gemm_ex, *base)[2])
        return
    for v in values[position]:
        args = list(base)
        args[position] = v
        assert outcome(pkg.gemm_ex, *args) == through_ctypes(pkg, monkeypatch, pkg.gemm_ex, *args), (position, v)
        if position not in (8, 9, 10):
            plain = args[:8] + [args[11]]
            assert outcome(pkg.gemm, *plain) == through_ctypes(pkg, monkeypatch, pkg.gemm, *plain), (position, v)


@pytest.mark.parametrize("name", ["quantize_a_1x128", "quantize_b_128x128"])
def test_quantisers(pkg, monkeypatch, name):
    f = getattr(pkg, name)
    base = [4096, 4096, 4096, 16, 100, 0, None]
    values = [POINTERS, POINTERS, POINTERS, SIZES, SIZES, [0, 1, 2, 3, -1, 1.0, None, True], STREAMS]
    for position, vs in enumerate(values):
        for v in vs:
            args = list(base)
            args[position] = v
            assert outcome(f, *args) == through_ctypes(pkg, monkeypatch, f, *args), (position, v)


def test_the_library_is_loaded_once(pkg):
    pkg.lib()
    outcome(pkg.gemm, 0, 0, 0, 0, 0, 1, 1, 128)
    paths = {line.split()[-1] for line in open("/proc/self/maps") if "libfp8gemm" in line}
    assert paths == {os.path.realpath(pkg.lib_path())}


@pytest.mark.parametrize("name,args", [("gemm", [4096] * 5 + [16, 16, 100]), ("gemm_ex", [4096] * 5 + [16, 16, 100]),
                                       ("quantize_a_1x128", [4096] * 3 + [16, 100]), ("quantize_b_128x128", [4096] * 3 + [16, 100])])
def test_without_the_module(pkg, monkeypatch, name, args):
    """not built, or for another interpreter: the library's answers all the same"""
    f = getattr(pkg, name)
    expected = outcome(f, *args)
    assert expected[:2] == (pkg.Fp8GemmError, -2), expected
    monkeypatch.setitem(f.__globals__, "_CALL", None)
    monkeypatch.delattr(pkg, "_pycall", raising=False)
    monkeypatch.setitem(sys.modules, pkg.__name__ + "._pycall", None)   # the import fails
    assert outcome(f, *args) == expected


HEADERS = pytest.mark.skipif(not os.path.exists(os.path.join(sysconfig.get_paths()["include"], "Python.h")), reason="no Python headers")


@HEADERS
def test_the_module_is_for_one_interpreter(pkg):
    outcome(pkg.gemm, 0, 0, 0, 0, 0, 1, 1, 128)
    assert pkg._pycall.__file__.endswith(sysconfig.get_config_var("EXT_SUFFIX"))


@HEADERS
def test_the_library_builds_without_pythons_headers(pkg):
    make = ["make", "-n", "-B", "-C", os.path.dirname(pkg.lib_path()), "all"]
    assert "pycall.cpp" in subprocess.run(make + [f"PYTHON={sys.executable}"], check=True, capture_output=True, text=True).stdout
    without = subprocess.run(make + ["PYTHON=/bin/false"], check=True, capture_output=True, text=True).stdout
    assert "pycall.cpp" not in without and "api.hip" in without
