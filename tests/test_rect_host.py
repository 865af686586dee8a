"""Host checks of the entry points that take a shape (no GPU)."""
import ctypes

import pytest

from testtimeideas_amd import _lib


def _size(keys=0, cols=0, seqlen=100, causal=0, window=0, entry=_lib.ENTRY_GG, dtype=0, head_dim=64, square=False):
    pr = _lib._Problem(dtype, causal, 1, 1, seqlen, head_dim, 0.125, 0, window, 0, _lib._View(None, 0, 0, 0), 0)
    shape = None if square else ctypes.byref(_lib._Shape(keys, cols))
    return _lib.load().ttt_attn_workspace_size_shape(ctypes.byref(pr), shape, entry, 0)


def _refused(message, **kw):
    assert _size(**kw) == -1, kw
    assert message in _lib.load().ttt_last_error(), (kw, _lib.load().ttt_last_error())


def test_square_shapes_need_what_the_square_entry_needs():
    lib = _lib.load()
    pr = _lib._Problem(0, 1, 1, 1, 8192, 64, 0.125, 0, 0, 0, _lib._View(None, 0, 0, 0), 0)
    want = lib.ttt_attn_workspace_size(ctypes.byref(pr), _lib.ENTRY_GG, 0)
    assert want > 0
    assert _size(seqlen=8192, causal=1, square=True) == want
    for keys in (0, 8192):
        for cols in (0, 64):
            assert _size(keys, cols, seqlen=8192, causal=1) == want


def test_rectangular_problems_are_plain():
    assert _size(4096) >= 0 and _size(1) >= 0
    for kw in (dict(causal=1), dict(causal=1, window=16)):
        _refused(b"neither causal nor windowed", keys=101, **kw)


@pytest.mark.parametrize("keys", [-1, (1 << 24) + 1])
def test_key_counts_out_of_range(keys):
    _refused(b"keys", keys=keys)


@pytest.mark.parametrize("dtype,head_dim,cols", [(0, 64, 8), (1, 64, 56), (2, 64, 24), (0, 128, 80), (1, 128, 8),
                                                 (2, 128, 128)])
def test_columns_that_are_taken(dtype, head_dim, cols):
    assert _size(cols=cols, dtype=dtype, head_dim=head_dim) == _size(dtype=dtype, head_dim=head_dim)


@pytest.mark.parametrize("dtype,head_dim,cols,message", [
    (0, 64, -8, b"cols -8: must be a multiple of 8"), (0, 64, 4, b"cols 4: must be a multiple of 8"),
    (0, 64, 72, b"up to head_dim 64"), (1, 128, 136, b"up to head_dim 128"), (2, 64, 60, b"cols 60"),
    (2, 128, 80, b"16-bit types only")])
def test_columns_that_are_refused(dtype, head_dim, cols, message):
    _refused(message, cols=cols, dtype=dtype, head_dim=head_dim)


def test_splits_follow_the_shape():
    """A walk is as long as the other side's rows: a split forced past it is clipped to it."""
    pr = _lib._Problem(0, 0, 1, 1, 640, 128, 0.125, 1 << 30, 0, 0, _lib._View(None, 0, 0, 0), 0)
    for entry, tiles in ((_lib.ENTRY_BWD_DQ, 2), (_lib.ENTRY_GG_ROW, 2), (_lib.ENTRY_BWD_DKDV, 10),
                         (_lib.ENTRY_GG_COL, 10)):
        assert _lib.split_info(pr, entry, False, shape=_lib._Shape(128, 80))[0] == tiles
        assert _lib.split_info(pr, entry, False)[0] == 10


def test_version_tells_the_entry_points_with_a_shape():
    lib = _lib.load()
    for name in _lib._SHAPED:
        assert hasattr(lib, name + "_shape")
    assert lib.ttt_version() >= 500
