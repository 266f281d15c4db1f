"""The rules that pick a call's kernel and splits, evaluated on the host (no GPU): where a rule's line has been on the wrong
side of a measured pair before, and which kernel the shapes of the GPU tests reach."""
import ctypes

import pytest

import mechta_amd as mk

I = ctypes.c_int


def fn(symbol, restype=I):
    f = getattr(mk.lib(), symbol)
    f.restype = restype
    return f


def merge_width(ntok, n, start, span, nch):
    """The chunks a merge build takes: 4, 8, 16 (merge_few), 32 (in two groups), 144, 256 (decode_combine)."""
    return fn("_ZN3mkv11merge_widthEiiiii")(ntok, n, start, span, nch)


@pytest.mark.parametrize("ntok,n,start,nch,want", [
    (63, 9000, 8500, 32, 4), (63, 9000, 4500, 32, 144), (63, 9000, 0, 32, 144), (64, 9000, 0, 32, 32),
    (64, 9000, 8500, 32, 4), (512, 28000, 0, 8, 8), (512, 28000, 27500, 8, 4), (16, 20000, 19000, 128, 8),
    (16, 20000, 0, 128, 144)])
def test_merge_takes_the_window_chunks(ntok, n, start, nch, want):
    """By the chunks that hold a key of the window, not by the call's splits."""
    assert merge_width(ntok, n, start, n + ntok - 1, nch) == want
