"""Calls through native code: the same conversions as ctypes makes, for every entry point."""
import ctypes
import importlib.machinery
import importlib.util
import subprocess

import numpy as np
import pytest
import torch

from zipage_amd import _lib
from zipage_amd.build import calls_command


def test_every_entry_point_is_there():
    calls = _lib.load_calls()
    for name in [*_lib.EXPORTS, *(n for names in _lib.MODEL_EXPORTS.values() for n in names)]:
        if name not in ("zp_abi_version", "zp_last_error"):
            assert callable(calls.entry(name, 1))
    with pytest.raises(KeyError):
        calls.entry("zp_nothing", 1)


def test_numbers_and_pointers_arrive():
    # an entry point of another library in place of each: what it returns says what came
    calls, seen = _lib.load_calls(), []
    proto = ctypes.CFUNCTYPE(ctypes.c_int32, *[ctypes.c_void_p] * 4, *[ctypes.c_int32] * 2, *[ctypes.c_int64] * 3, ctypes.c_float,
                             ctypes.c_int32, ctypes.c_void_p)
    back = proto(lambda *a: (seen.append(a), -7)[1])
    add_rms = calls.entry("zp_add_rms_norm", ctypes.cast(back, ctypes.c_void_p).value)
    held = (ctypes.c_int64 * 3)(5, 6, 7)
    assert add_rms(0, None, held, 1 << 63, -1, True, 1 << 40, -(1 << 40), 3, 0.1, 2, 9) == -7
    assert seen == [(None, None, ctypes.addressof(held), 1 << 63, -1, 1, 1 << 40, -(1 << 40), 3, ctypes.c_float(0.1).value, 2, 9)]
    assert add_rms(1, 1, 1, 1, 1, 1, 1, 1, 1, 3, 1, 1) == -7 and seen[1][9] == 3.0      # a whole number is a number
    add_rms(0, 0, ctypes.byref(held), *[1] * 9)
    assert seen.pop()[2] == ctypes.addressof(held)
    for bad in ([0] * 11, [0] * 13, [0] * 4 + [0.5] + [0] * 7, ["x"] + [0] * 11, [0] * 9 + ["x", 0, 0], [1 << 64] + [0] * 11):
        with pytest.raises((TypeError, OverflowError)):
            add_rms(*bad)
    assert len(seen) == 2


def test_calls_agree_with_ctypes():
    for n in (1, 300, 4000):
        assert _lib.size("zp_moe_tile_rows", n, 32, 3, 0) == _lib.load_models("moe").zp_moe_tile_rows(n, 32, 3, 0)
    with pytest.raises(RuntimeError, match="silu_and_mul"):
        _lib.call("zp_silu_and_mul", None, None, 1, -8, 0, 0, 0, None)
    with pytest.raises(RuntimeError, match="run_attention"):
        _lib.call_models("zp_run_attention", *[None] * 7, _lib.AttentionForm(0.0, 2, 0.5, 1e-6, 0, None, 0), 1, 4, 4, 32, 0, 32, 0, 0, 1, 1,
                         256, 256, 0, 128, 1.0, 1.0, 0, None)


def test_addresses_of_tensors():
    assert _lib.dev_ptr(None) == 0
    with pytest.raises(RuntimeError, match="device tensors"):
        _lib.dev_ptr(torch.zeros(3))
    with pytest.raises(AttributeError):
        _lib.dev_ptr(3)


class _Numbers(ctypes.Structure):
    _fields_ = [("a", ctypes.c_int64), ("b", ctypes.c_int64)]


def test_what_stands_for_a_pointer():
    calls, seen = _lib.load_calls(), []
    back = ctypes.CFUNCTYPE(ctypes.c_int32, *[ctypes.c_void_p] * 3, ctypes.c_int32, ctypes.c_int32, ctypes.c_int64,
                            ctypes.c_void_p)(lambda *a: (seen.append(a[0]), 0)[1])
    gather = calls.entry("zp_gather_rows", ctypes.cast(back, ctypes.c_void_p).value)
    call = lambda o: (gather(o, 0, 0, 0, 0, 0, 0), seen.pop())[1]
    held, numbers = (ctypes.c_int64 * 3)(5, 6, 7), _Numbers(1, 2)
    at = ctypes.addressof(held)
    for o, want in ((None, None), (0, None), (at, at), (held, at), (ctypes.byref(held), at), (ctypes.byref(held, 8), at + 8),
                    (ctypes.c_void_p(at), at), (ctypes.c_void_p(), None), (ctypes.cast(held, ctypes.POINTER(ctypes.c_int64)), at),
                    (numbers, ctypes.addressof(numbers))):
        assert call(o) == want, o
    # what ctypes refuses for an address stays refused: a number that is not Python's, and what merely has a buffer
    for o in (np.int64(at), np.array([at]), bytearray(8), memoryview(b"12345678"), torch.zeros(2), 1.5, [at], ctypes.c_int64(at)):
        with pytest.raises(TypeError):
            gather(o, 0, 0, 0, 0, 0, 0)
    assert not seen


def test_what_stands_for_a_structure():
    calls, seen = _lib.load_calls(), []
    back = ctypes.CFUNCTYPE(ctypes.c_int32, ctypes.c_void_p, ctypes.c_int32, ctypes.c_void_p)(lambda *a: (seen.append(a[0]), 0)[1])
    scan = calls.entry("zp_linear_scan", ctypes.cast(back, ctypes.c_void_p).value)
    args = _lib.LinearArgs()
    for o in (args, ctypes.byref(args)):
        assert scan(o, 0, 0) == 0 and seen.pop() == ctypes.addressof(args)
    for o in (ctypes.addressof(args), _Numbers(), ctypes.byref(_Numbers()), _lib.AttentionForm(), ctypes.c_void_p(ctypes.addressof(args))):
        with pytest.raises(TypeError):
            scan(o, 0, 0)
    assert not seen


def test_built_for_another_python(tmp_path):
    path = str(tmp_path / "zipage_calls.so")
    subprocess.run([*calls_command(path), '-DZP_PYTHON="3.99."', "-O0"], check=True)
    loader = importlib.machinery.ExtensionFileLoader("zipage_calls", path)
    with pytest.raises(ImportError, match="Python 3.99.x"):
        importlib.util.module_from_spec(importlib.util.spec_from_loader("zipage_calls", loader))
