"""f16 prefill blocks of 64 tokens and more, each case on the kernel it names (asserted on the plan): the small-block kernel
(f32-class arithmetic: short contexts, up to 256 tokens) and prefill_f16 with two key groups and with one. What each has to
get right where it can go wrong: rows past the length, a reference maximum that moves inside a split, a window start, tiles
far into a large store, replays of a captured call."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import ATOL, RTOL, assert_attn_close, q_inputs
from tests.test_plans import fn, prefill_plan

pytestmark = pytest.mark.gpu


def kernel(T, n0, start=0):
    if fn("_ZN3mkv18small_prefill_paysEiii", ctypes.c_bool)(T, n0, start):
        return "small"
    return {1: "one group", 2: "two groups"}[prefill_plan(T, n0, start).ks]


def rows(torch, n, seed, boost=()):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    k, v = (torch.randn((n, 2, 256), generator=g, device="cuda").half() for _ in range(2))
    for p in boost:
        k[p] *= 24
    return k, v


def bits16(x):
    import torch
    return x.view(torch.int16)


def write(mk, st, layer, k, v):
    st.write_rows(layer, mk.K, 0, k.shape[0], bits16(k))
    st.write_rows(layer, mk.V, 0, v.shape[0], bits16(v))


def ctx_of(n):
    return max(4096, (n + 1023) // 1024 * 1024)


def bits(x):
    return x.cpu().numpy().view(np.uint16)


def tokens(T):
    s = np.unique(np.r_[0:3, T // 2, 15, 16, 31, 32, 63, T - 2, T - 1])
    return s[s < T].astype(np.int32)


@pytest.mark.parametrize("want,n0,T", [("small", 900, 96), ("two groups", 5000, 300), ("two groups", 31, 257),
                                       ("one group", 27990, 512), ("one group", 14001, 500)])
def test_nan_rows_past_the_length(torch_gpu, want, n0, T):
    import mechta_amd as mk
    torch = torch_gpu
    print(f"NaN rows, {want}: n0={n0} T={T}", flush=True)
    assert kernel(T, n0) == want
    n = n0 + T - 1
    assert n % 32, "a whole last tile holds no rows past the length"
    k, v = rows(torch, n, 31 + T)
    q = q_inputs(32 + T, T)
    with mk.KvStore(1, ctx_of(n + 64), mk.F16) as st:
        write(mk, st, 0, k, v)
        nan = torch.full((64, 2, 256), float("nan"), device="cuda").half().view(torch.int16)
        for which in (mk.K, mk.V):
            st.write_rows(0, which, n, n + 64, nan)
        st.set_len(n)
        out = st.prefill(0, torch.from_numpy(q).cuda(), n0).cpu().numpy()
    assert np.isfinite(out).all()
    sel = tokens(T)
    ref = O.attn_fa_mx(bits(k), bits(v), q, n0, sel=sel)
    assert_attn_close(out[sel], ref, atol=ATOL, rtol=RTOL, what=f"{want} next to NaN rows")


@pytest.mark.parametrize("want,n0,T,start", [("two groups", 6000, 300, 0), ("two groups", 9000, 200, 2000),
                                             ("one group", 14000, 512, 0), ("one group", 20000, 500, 7003),
                                             ("one group", 30000, 300, 29000)])
def test_max_jump_and_window(torch_gpu, want, n0, T, start):
    """Keys boosted 24x move the lazy reference maximum in the middle of a split (O and the sums are rescaled), in every
    split region, with and without a window start inside a tile."""
    import mechta_amd as mk
    torch = torch_gpu
    print(f"max jump, {want}: n0={n0} T={T} start={start}", flush=True)
    assert kernel(T, n0, start) == want
    n = n0 + T - 1
    boost = sorted({start + 700, (start + n0) // 2, n0 - 3, n0 + T // 2})
    k, v = rows(torch, n, 41 + T, boost)
    q = q_inputs(42 + T, T)
    with mk.KvStore(1, ctx_of(n), mk.F16) as st:
        write(mk, st, 0, k, v)
        out = st.prefill(0, torch.from_numpy(q).cuda(), n0, start=start).cpu().numpy()
    sel = np.unique(np.r_[tokens(T), T // 2 - 1, T // 2 + 1]).astype(np.int32)
    ref = O.attn_fa_mx(bits(k), bits(v), q, n0, start=start, sel=sel)
    assert_attn_close(out[sel], ref, atol=ATOL, rtol=RTOL, what=f"{want}, max jump")


@pytest.mark.parametrize("n0,T,start", [(1, 64, 0), (2, 65, 0), (31, 79, 0), (160, 96, 0), (161, 97, 40), (700, 127, 0),
                                        (3000, 64, 0), (1000, 241, 500), (64, 256, 0), (500, 256, 0)])
def test_small_block_kernel_is_f32_class(torch_gpu, n0, T, start):
    """Blocks of 64 tokens and more on the small-block kernel keep the arithmetic of the blocks under 64: attn_fd4 (with a
    window attn_fd) within 1e-5, where f16 Q and P are 30 times further away."""
    import mechta_amd as mk
    torch = torch_gpu
    print(f"f32-class block n0={n0} T={T} start={start}", flush=True)
    assert kernel(T, n0, start) == "small"
    n = n0 + T - 1
    k, v = rows(torch, n, 51 + T)
    q = q_inputs(52 + T, T)
    with mk.KvStore(1, 4096, mk.F16) as st:
        write(mk, st, 0, k, v)
        out = st.prefill(0, torch.from_numpy(q).cuda(), n0, start=start).cpu().numpy()
    ref = O.attn_fd(0, bits(k), bits(v), q, n0, start=start) if start else O.attn_fd4(0, bits(k), bits(v), q, n0)
    assert_attn_close(out, ref, atol=1e-5, rtol=1e-5, what=f"small-block kernel, {T} tokens")


@pytest.mark.parametrize("want,T", [("one group", 320), ("small", 64)])
def test_block_at_the_end_of_a_large_store(torch_gpu, want, T):
    """The last layer of a 5 GB store: tile addresses past 2^32 from its base, their low words on both sides of 2^31."""
    import mechta_amd as mk
    torch = torch_gpu
    layers, ctx = 10, 262144
    n0 = ctx - T + 1
    start = n0 - 2048
    print(f"end of a large store, {want}: T={T}", flush=True)
    assert kernel(T, n0, start) == want
    n = n0 + T - 1
    k, v = rows(torch, n, 61 + T)
    q = q_inputs(62 + T, T)
    with mk.KvStore(layers, ctx, mk.F16) as st:
        write(mk, st, layers - 1, k, v)
        out = st.prefill(layers - 1, torch.from_numpy(q).cuda(), n0, start=start).cpu().numpy()
    sel = tokens(T)
    ref = O.attn_fa_mx(bits(k), bits(v), q, n0, start=start, sel=sel)
    assert_attn_close(out[sel], ref, atol=ATOL, rtol=RTOL, what=f"{want} at the end of the store")


@pytest.mark.parametrize("want,n0,T", [("two groups", 5000, 300), ("one group", 14000, 512)])
def test_captured_block_replays(torch_gpu, want, n0, T):
    import mechta_amd as mk
    torch = torch_gpu
    print(f"captured block, {want}: n0={n0} T={T}", flush=True)
    assert kernel(T, n0) == want
    n = n0 + T - 1
    k, v = rows(torch, n, 71 + T)
    q = torch.from_numpy(q_inputs(72 + T, T)).cuda()
    with mk.KvStore(1, ctx_of(n), mk.F16) as st:
        write(mk, st, 0, k, v)
        torch.cuda.synchronize()
        out = torch.empty((T, 16, 256), device="cuda")
        base = torch.cuda.current_stream()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):  # before any eager attention call of the store
            st.set_stream(torch.cuda.current_stream())
            st.prefill(0, q, n0, out=out)
        st.set_stream(base)
        eager = st.prefill(0, q, n0).clone()
        torch.cuda.synchronize()
        for r in range(3):
            out.fill_(float("nan"))
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, eager), f"replay {r} differs from the eager call"
            assert torch.isfinite(st.prefill(0, q[:200], n0 - 700)).all()  # eager work of the store in between
            torch.cuda.synchronize()
