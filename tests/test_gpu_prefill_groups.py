"""f16 prefill blocks of 64 tokens or more on the three kernels' edges: the small-block kernel (short contexts, up to 256
tokens), and prefill_f16 with one or two key groups: waves of three tiles and more, an odd tile left over for one group,
ragged last blocks and tiles, key counts on both sides of the rules that pick. Bars as test_gpu_kvpath.py: attn_fa_mx at the
task tolerance, selected tokens (test_gpu_prefill_paths.py holds the small-block kernel to its own f32-class bar)."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import assert_attn_close, gate_inputs, prefill_reference, q_inputs

pytestmark = pytest.mark.gpu

# (n0, T, start): short contexts and up to 256 tokens: the small-block kernel; 257 and more: two groups, down to three tiles
# per wave; block edges at 16 and 32 tokens; windows; long contexts, where wide blocks take one group (256 tokens cross
# over near 22,000 positions, 512 near 9,000)
CASES = [(1, 64, 0), (2, 65, 0), (31, 79, 0), (160, 96, 0), (161, 97, 40), (700, 127, 0), (1000, 241, 500), (64, 256, 0),
         (1, 257, 0), (31, 300, 0), (33, 512, 0), (700, 273, 600), (5000, 511, 0), (6000, 128, 0), (9000, 200, 0),
         (9011, 500, 4000), (20000, 256, 0), (30000, 512, 0), (30001, 255, 0), (32000, 67, 31000)]


@pytest.mark.parametrize("n0,T,start", CASES)
def test_prefill_groups(torch_gpu, n0, T, start):
    import mechta_amd as mk
    torch = torch_gpu
    print(f"prefill groups n0={n0} T={T} start={start}", flush=True)
    n = n0 + T - 1
    ctx = max(4096, (n + 1023) // 1024 * 1024)
    g = torch.Generator(device="cuda")
    g.manual_seed(n0 + T)
    k, v = (torch.randn((n, 2, 256), generator=g, device="cuda").half() for _ in range(2))
    q, gate = q_inputs(9000 + T, T), gate_inputs(9100 + T, T)
    with mk.KvStore(1, ctx, mk.F16) as st:
        st.write_rows(0, mk.K, 0, n, k.view(torch.int16))
        st.write_rows(0, mk.V, 0, n, v.view(torch.int16))
        out = st.prefill(0, torch.from_numpy(q).cuda(), n0, start=start).cpu().numpy()
        gated = st.prefill(0, torch.from_numpy(q).cuda(), n0, start=start,
                           gate_src=torch.from_numpy(gate).cuda()).cpu().numpy()
    kc, vc = (x.cpu().numpy().view(np.uint16) for x in (k, v))
    sel = np.unique(np.r_[0:min(T, 3), T // 2, 15, 16, 31, 32, T - 2, T - 1]).astype(np.int32)
    sel = sel[(sel >= 0) & (sel < T)]
    ref, atol, rtol = prefill_reference(0, kc, vc, q, n0, start=start, sel=sel)
    assert_attn_close(out[sel], ref, atol=atol, rtol=rtol, what=f"prefill T {T}")
    sig = 1 / (1 + np.exp(-gate[..., 256:].astype(np.float64)))
    # the gate multiplies the normalized f32 output: a few roundings of 2^-24 each
    assert_attn_close(gated, out * sig, atol=1e-6, rtol=1e-6, what="gate")
