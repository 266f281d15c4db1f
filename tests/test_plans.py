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


class PrefillPlan(ctypes.Structure):
    _fields_ = [("span", I), ("nch", I), ("ks", I)]


def prefill_plan(T, n, start=0):
    """prefill_f16's splits and key groups per work-group (1 or 2)."""
    return fn("_ZN3mkv12prefill_planEiiiPi", PrefillPlan)(T, n, start, None)


def prefill32_plan(T, n, start=0):
    return fn("_ZN3mkv14prefill32_planEiii", PrefillPlan)(T, n, start)


@pytest.mark.parametrize("T,n,start,least", [(63, 2000, 1500, 24), (64, 2000, 1500, 22), (48, 4000, 3500, 32),
                                             (80, 4000, 3500, 22), (16, 2000, 1500, 32)])
def test_f32_window_takes_more_splits(T, n, start, least):
    """A merge that reads two or three chunks does not pay for the others: on the splits of the same call without a window
    (mostly 16), these took 4-20% longer than on `least` splits or more."""
    assert prefill32_plan(T, n, start).nch >= least


@pytest.mark.parametrize("T,n,start", [(320, 9000, 8500), (384, 9000, 8500), (512, 6000, 5500), (184, 20000, 19500),
                                       (96, 45000, 44500)])
def test_f16_window_takes_one_group(T, n, start):
    """Two groups save half of a merge that reads little: 4-10% slower there with a window."""
    assert prefill_plan(T, n, start).ks == 1


# (tokens, positions, faster group count): pairs measured with the keys from HBM, 4% apart or more
GROUPS = [(512, 9000, 1), (512, 12000, 1), (512, 28000, 1), (384, 14000, 1), (320, 16000, 1), (256, 24000, 1), (160, 45000, 1),
          (128, 60000, 1), (96, 90000, 1), (64, 90000, 1), (64, 120000, 1), (512, 3000, 2), (384, 6000, 2), (256, 12000, 2),
          (200, 9000, 2), (200, 28000, 2), (128, 28000, 2), (72, 28000, 2), (64, 16000, 2)]


@pytest.mark.parametrize("T,n,ks", GROUPS)
def test_key_groups(T, n, ks):
    assert prefill_plan(T, n).ks == ks


class FlintPlan(ctypes.Structure):
    _fields_ = [(x, I) for x in ("klo", "span", "nch", "nrb", "blk", "fused")]


def flint_plan(fmt, pos0, T, win=0):
    """blk: 1-2 (fl_dec16), 4 (fl_attn), 32 (fl_pf)."""
    return fn("_ZN3mkv5flint4planEiiii", FlintPlan)(fmt, pos0, T, win)


@pytest.mark.parametrize("fmt,T,nch", [(0, 5, 64), (0, 12, 64), (0, 24, 64), (0, 48, 32), (1, 12, 64), (1, 24, 64), (1, 48, 32)])
def test_flint_long_spans_take_every_split(fmt, T, nch):
    """Splits of a dozen tiles or more finish sooner the more there are, also where the longest is as long."""
    p = flint_plan(fmt, 30000, T)
    assert (p.blk, p.nch) == (32, nch)


class Geom(ctypes.Structure):
    _fields_ = [("layers", I), ("ctx", I), ("fmt", I), ("plane_elems", ctypes.c_size_t)]


class SmallPlan(ctypes.Structure):
    _fields_ = [(x, I) for x in ("span", "nch", "c0", "s0", "nu", "nzb")]


class Launch(ctypes.Structure):
    _fields_ = [(x, ctypes.c_void_p) for x in ("s", "a", "b")]


@pytest.mark.parametrize("fmt,T", [(0, 0), (0, 257), (0, 512), (1, 16)])
def test_small_block_launcher_refuses(fmt, T):
    """hipErrorNotSupported (801) before any launch: the store's format, and blocks of more than 256 tokens."""
    launch = fn("_ZN3mkv20launch_small_prefillERKNS_4GeomEPKviPKfiiifRKNS_9SmallPlanEPfRKNS_6LaunchE")
    g, p, s = Geom(1, 4096, fmt, 4096 * 256), SmallPlan(0, 2, 0, 0, 2, 64), Launch(None, None, None)
    rc = launch(ctypes.byref(g), None, 0, None, T, 1, 0, ctypes.c_float(1.0), ctypes.byref(p), None, ctypes.byref(s))
    assert rc == 801
