"""Decodes over the f32 store at the edges of their work split: one, two, three and four 32-key tiles per work-group, a
last work-group without a second tile, appended rows in one tile or across two, windows that start inside a tile. Oracle
and bar as test_gpu_kvpath.py: attn_fd within 1e-5; the fused append and decode bit for bit the plain decode's."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import assert_attn_close, q_inputs

pytestmark = pytest.mark.gpu

# (ctx, n0, ntok, start)
CASES = [(4096, 31, 4, 0), (4096, 32, 1, 0), (4096, 62, 4, 0), (4096, 64, 2, 0), (4096, 95, 4, 0), (4096, 127, 2, 33),
         (4096, 2045, 4, 0), (4096, 2046, 4, 0),
         (4096, 2049, 1, 0), (4096, 4093, 4, 0), (10240, 8188, 4, 0), (10240, 8193, 1, 0), (10240, 8290, 4, 63),
         (13312, 12285, 4, 0), (13312, 12289, 1, 0), (13312, 12320, 3, 20)]


@pytest.mark.parametrize("ctx,n0,ntok,start", CASES)
def test_decode32_splits(torch_gpu, ctx, n0, ntok, start):
    import mechta_amd as mk
    torch = torch_gpu
    print(f"f32 decode splits ctx={ctx} n0={n0} ntok={ntok} start={start}", flush=True)
    n = n0 + ntok - 1
    g = torch.Generator(device="cuda")
    g.manual_seed(n0 + ntok)
    k, v = (torch.randn((n, 2, 256), generator=g, device="cuda") for _ in range(2))
    kn, vn = (torch.randn((ntok, 2, 256), generator=g, device="cuda") for _ in range(2))
    tab = torch.randn((ntok, 64), generator=g, device="cuda")
    q = torch.from_numpy(q_inputs(700 + n0, ntok)).cuda()
    with mk.KvStore(1, ctx, mk.F32) as st:
        st.write_rows(0, mk.K, 0, n, k)
        st.write_rows(0, mk.V, 0, n, v)
        out = st.decode(0, q, n0, start=start).cpu().numpy()
        fused = st.append_decode(0, n0, kn, vn, tab, q, start=start).cpu().numpy()
        plain = st.decode(0, q, n0, start=start).cpu().numpy()
    ref = O.attn_fd(1, k.cpu().numpy(), v.cpu().numpy(), q.cpu().numpy(), n0, start=start)
    assert_attn_close(out, ref, atol=1e-5, rtol=1e-5, what="f32 vs attn_fd")
    assert np.array_equal(fused, plain), "fused append and decode differs from the plain decode"


def test_decode32_grid_of_any_size(torch_gpu):
    """A decode whose grid is no multiple of 8 (30,000 positions: 468 work-groups) costs no more than the next that is
    (30,208: 472). In XCD order it took 1.03 times as long, in launch order 0.99; the least of five measured ratios is held
    to 1.01."""
    import statistics

    import mechta_amd as mk
    torch = torch_gpu
    layers, ctx = 4, 32768
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    q = torch.randn((1, 16, 256), generator=g, device="cuda")
    out = torch.empty_like(q)
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)

    with mk.KvStore(layers, ctx, mk.F32) as st:
        for layer in range(layers):
            for which in (mk.K, mk.V):
                st.write_rows(layer, which, 0, ctx, torch.randn((ctx, 2, 256), generator=g, device="cuda"))

        def timed(n):
            torch.cuda.synchronize()
            torch.cuda._sleep(2000000)  # the calls below are queued by the time it ends
            a.record()
            for i in range(24):
                st.decode(i % layers, q, n, out=out)
            b.record()
            torch.cuda.synchronize()
            return a.elapsed_time(b)

        timed(30000), timed(30208)
        best = 9.0
        for trial in range(5):
            pairs = [(timed(30000), timed(30208)) for _ in range(5)]
            best = min(best, statistics.median(x for x, _ in pairs) / statistics.median(y for _, y in pairs))
            print(f"f32 decode, 468 against 472 work-groups: {best:.3f}", flush=True)
            if best <= 1.01:
                break
    assert best <= 1.01
