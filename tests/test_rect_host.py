"""Host checks of the rectangular entry points (no GPU)."""
import ctypes

import pytest

from testtimeideas_amd import _lib


class Shape(ctypes.Structure):
    _fields_ = [("keys", ctypes.c_int64)]


def _size(keys, seqlen=100, causal=0, window=0, entry=_lib.ENTRY_GG):
    lib = _lib.load()
    fn = lib.ttt_attn_workspace_size_shape
    fn.argtypes = [ctypes.POINTER(_lib._Problem), ctypes.POINTER(Shape), ctypes.c_int32, ctypes.c_int32]
    fn.restype = ctypes.c_int64
    pr = _lib._Problem(0, causal, 1, 1, seqlen, 64, 0.125, 0, window, 0, _lib._View(None, 0, 0, 0), 0)
    return fn(ctypes.byref(pr), None if keys is None else ctypes.byref(Shape(keys)), entry, 0)


def test_square_shapes_need_what_the_square_entry_needs():
    lib = _lib.load()
    pr = _lib._Problem(0, 1, 1, 1, 8192, 64, 0.125, 0, 0, 0, _lib._View(None, 0, 0, 0), 0)
    want = lib.ttt_attn_workspace_size(ctypes.byref(pr), _lib.ENTRY_GG, 0)
    assert want > 0
    for keys in (None, 0, 8192):
        assert _size(keys, seqlen=8192, causal=1) == want


def test_rectangular_problems_are_plain():
    assert _size(4096) >= 0 and _size(1) >= 0
    for kw in (dict(causal=1), dict(causal=1, window=16)):
        assert _size(101, **kw) == -1
        assert b"neither causal nor windowed" in _lib.load().ttt_last_error()


@pytest.mark.parametrize("keys", [-1, (1 << 24) + 1])
def test_key_counts_out_of_range(keys):
    assert _size(keys) == -1
