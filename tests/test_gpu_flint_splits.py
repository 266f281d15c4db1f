"""Flint blocks at the edges of the plan that picks their kernel (fl_dec16, fl_attn, fl_pf) and splits: splits of one tile, a last split of a few
keys, 8, 9, 16 and more splits (each merge build), blocks and windows whose first or last rows see no key of a split.
Oracle and bars as test_gpu_flint.py: attn_pf within 1e-5."""
import pytest

from oracle import oracle as O
from tests.helpers import assert_attn_close
from tests.test_gpu_flint import D, F16, F32, H, TOL, dev, fill, mf, rng  # noqa: F401

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
