"""Flint blocks at the edges of the plan that picks their kernel (fl_dec16, fl_attn, fl_pf) and splits: splits of one tile, a
last split of a few keys, merges of 1 to 64 splits (exactly full ones below), blocks and windows whose first or last rows
see no key of a split. Oracle and bars as test_gpu_flint.py: attn_pf within 1e-5."""
import pytest

from oracle import oracle as O
from tests.helpers import assert_attn_close
from tests.test_gpu_flint import D, F16, F32, H, TOL, dev, fill, mf, rng  # noqa: F401
from tests.test_plans import flint_plan

pytestmark = pytest.mark.gpu

# (sliding, pos0, T)
CASES = [(False, 27, 5), (False, 28, 5), (False, 250, 16), (False, 600, 5), (False, 1500, 17), (False, 2040, 8),
         (False, 33, 32), (False, 224, 33), (False, 2000, 64), (False, 2011, 100), (False, 600, 256),
         (False, 2046, 1), (False, 2047, 2), (False, 3071, 1), (False, 3072, 2), (False, 3400, 20), (False, 33, 128),
         (True, 520, 1), (True, 1024, 2), (True, 600, 5), (True, 1030, 31), (True, 511, 97), (True, 1000, 256)]


@pytest.mark.parametrize("fmt", [F32, F16])
@pytest.mark.parametrize("sliding,pos0,T", CASES)
def test_flint_block_splits(torch_gpu, mf, fmt, sliding, pos0, T):  # noqa: F811
    torch = torch_gpu
    print(f"flint block splits fmt={fmt} sliding={sliding} pos0={pos0} T={T}", flush=True)
    with mf.FlintStore(1, 4096, fmt, sliding=[sliding]) as st:
        kc, vc = O.fl_new_cache(st.rows(0), fmt), O.fl_new_cache(st.rows(0), fmt)
        fill(torch, st, kc, vc, 0, fmt, pos0 + T, seed=40 + pos0)
        q = rng(41).standard_normal((T, H, D), dtype="float32")
        sinks = rng(42).standard_normal(H, dtype="float32")
        out = st.attend(0, pos0, dev(torch, q), dev(torch, sinks)).cpu().numpy()
    ref = O.fl_attn_pf(fmt, kc, vc, q, pos0, 513 if sliding else 0, sinks)
    assert_attn_close(out, ref, atol=TOL, rtol=TOL, what="flint block vs attn_pf")


# (fmt, pos0, T, splits, tokens per block): exactly the chunks that fl_merge_few<8> and <16> hold, after fl_attn and fl_pf
FULL = [(F32, 1700, 64, 8, 4), (F16, 680, 64, 8, 4), (F32, 1000, 16, 16, 4), (F16, 1000, 16, 16, 4), (F32, 840, 128, 8, 32),
        (F16, 400, 96, 8, 32), (F32, 1880, 48, 16, 32), (F16, 2960, 96, 16, 32)]


@pytest.mark.parametrize("fmt,pos0,T,nch,blk", FULL)
def test_flint_merge_builds_full(torch_gpu, mf, fmt, pos0, T, nch, blk):  # noqa: F811
    torch = torch_gpu
    print(f"flint merge of {nch} splits fmt={fmt} pos0={pos0} T={T}", flush=True)
    p = flint_plan(fmt, pos0, T)
    assert (p.nch, p.blk) == (nch, blk)
    with mf.FlintStore(1, 4096, fmt, sliding=[False]) as st:
        kc, vc = O.fl_new_cache(st.rows(0), fmt), O.fl_new_cache(st.rows(0), fmt)
        fill(torch, st, kc, vc, 0, fmt, pos0 + T, seed=60 + T)
        q = rng(61).standard_normal((T, H, D), dtype="float32")
        sinks = rng(62).standard_normal(H, dtype="float32")
        out = st.attend(0, pos0, dev(torch, q), dev(torch, sinks)).cpu().numpy()
    assert_attn_close(out, O.fl_attn_pf(fmt, kc, vc, q, pos0, 0, sinks), atol=TOL, rtol=TOL, what=f"{nch} splits")


@pytest.mark.parametrize("fmt", [F32, F16])
@pytest.mark.parametrize("boost", [False, True])
def test_fl_pf_sliding_block(torch_gpu, mf, fmt, boost):  # noqa: F811
    """fl_pf on a sliding ring: rows of positions before the block's first window hold NaN (its tiles take them in, its V
    must not), or keys boosted 24x move the reference maximum inside the window (bar as test_gpu_rescale.py)."""
    torch = torch_gpu
    pos0, T = 3000, 256
    print(f"fl_pf sliding fmt={fmt} boost={boost}", flush=True)
    assert flint_plan(fmt, pos0, T, 513).blk == 32
    r = rng(71)
    k, v = (r.standard_normal((pos0 + T, 4, D), dtype="float32") for _ in range(2))
    if boost:
        for b in (pos0 - 400, pos0 - 100, pos0 + 30, pos0 + T - 1):
            k[b] *= 24.0
    with mf.FlintStore(1, 4096, fmt, sliding=[True]) as st:
        kc, vc = O.fl_new_cache(st.rows(0), fmt), O.fl_new_cache(st.rows(0), fmt)
        for p in range(0, pos0 + T, 512):
            m = min(512, pos0 + T - p)
            st.append(0, p, dev(torch, k[p:p + m]), dev(torch, v[p:p + m]))
            O.fl_kv_write(fmt, kc, vc, p, k[p:p + m], v[p:p + m])
        if not boost:  # every position that no token of the block sees: before the first window, down to the ring's oldest
            nan = torch.full((1, 4, D), float("nan"), device="cuda")
            nan = nan.half().view(torch.int16) if fmt == F16 else nan
            for p in range(pos0 + T - 1024, pos0 - 512):
                for which in (0, 1):
                    st.write_rows(0, which, p % 1024, p % 1024 + 1, nan)
        q = r.standard_normal((T, H, D), dtype="float32")
        sinks = r.standard_normal(H, dtype="float32")
        out = st.attend(0, pos0, dev(torch, q), dev(torch, sinks)).cpu().numpy()
    tol = dict(atol=1e-4, rtol=1e-5) if boost else dict(atol=TOL, rtol=TOL)
    assert_attn_close(out, O.fl_attn_pf(fmt, kc, vc, q, pos0, 513, sinks), what="fl_pf, sliding", **tol)
