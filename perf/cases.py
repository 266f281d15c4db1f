"""Timed cases of the KV-cache path: what an engine asks of this library, through its public entry points.

Kinds of work, and the ranges the listed cases stand for:

- `step`: a decode step of 1 to 4 tokens (4: the verify of 3 MTP drafts), append + attention (mkv_append_decode), over
  every layer of the store, then the next step after the rejected drafts were rolled back (mkv_set_len). The second
  step reads rows the first one wrote. Contexts from a few hundred to 262,140 positions, both store formats, with and
  without the sigmoid output gate, the gated output in f32 or f16 (mkv_append_decode_g16), and the window start of the
  MTP layer.
- `block`: a prompt block of 5 to 512 tokens on one layer: the q/k producer (mkv_qk_norm_rope), the append, the causal
  attention with the gate. Full 512-token chunks, a user's turn of a few hundred tokens, the ragged tail of a prompt.
- `flint_step` / `flint_block`: the same for the Flint model's layers (a sliding layer and a full layer): RoPE of q and
  k, ring append, attention with sinks.
- `rows`: a layer's K and V rows out of the store and into another store in the reference's position-major layout
  (the words of a root file).

The token steps call the C ABI through `lib()` on the store's handle with device pointers taken beforehand, as bench.py
does and as an engine that binds the library does (a serving loop holds its buffers); the blocks use the Python classes.
Inputs are seeded N(0,1) values (K and q leave an RMSNorm in the engine), the caches filled row by row through
write_rows. All shapes are the model's: 16 query and 2 KV heads of 256 (Flint: 32 and 4 of 128).
"""
import ctypes
import math

import numpy as np
import torch

import mechta_amd as mk
from mechta_amd import flint as mf

SCALE = 1.0 / 16  # 1 / sqrt(256)
EPS = 1e-6        # the engine's RMSNorm epsilon
FLINT_BASE = 10000.0
KEEP = 2          # positions a verify of 4 tokens moves on by (2 drafts rejected)


def listed():
    return [
        # the first answer of a short chat: one token, one layer, a short context, gated; latency of the two launches
        dict(name="step_1tok_700", kind="step", fmt=0, layers=1, ntok=1, n=701, start=0, out="gate"),
        # plain generation at 4K, the 10 attention layers of the model, gated
        dict(name="step_1tok_4k", kind="step", fmt=0, layers=10, ntok=1, n=4097, start=0, out="gate"),
        # speculative decoding at 64K: the 4-token verify of the 10 layers, 2 drafts rejected
        dict(name="verify_64k", kind="step", fmt=0, layers=10, ntok=4, n=65537, start=0, out="plain"),
        # the same near the largest context, f16 gated output (the form the f16 output projection takes)
        dict(name="verify_256k", kind="step", fmt=0, layers=2, ntok=4, n=262001, start=0, out="g16"),
        # the f32 store's verify at 16K
        dict(name="verify_f32_16k", kind="step", fmt=1, layers=10, ntok=4, n=16385, start=0, out="plain"),
        # a full 512-token chunk of a long prompt
        dict(name="chunk_28k", kind="block", fmt=0, T=512, n0=28000),
        # a user's turn on top of a conversation
        dict(name="turn_200_9k", kind="block", fmt=0, T=200, n0=9001),
        # the last, ragged block of a prompt (blocks under 64 tokens run f32-class)
        dict(name="tail_37_20k", kind="block", fmt=0, T=37, n0=20003),
        # a full chunk on the f32 store
        dict(name="chunk_f32_16k", kind="block", fmt=1, T=512, n0=16000),
        # Flint generation at 20K: one token through a sliding and a full layer (f32 K/V, that model's default)
        dict(name="flint_step_20k", kind="flint_step", fmt=1, n=20001),
        # Flint prompt chunk through a sliding and a full layer
        dict(name="flint_chunk_20k", kind="flint_block", fmt=1, T=512, n0=20000),
        # the words of a layer's K and V for a root file of 8,192 positions, out and back in
        dict(name="rows_8k", kind="rows", fmt=0, p=8192),
    ]


def _logint(rng, lo, hi):
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "block", "block", "block", "flint_step", "flint_block", "rows"])
    fmt = rng.choice([0, 0, 1])
    if kind == "step":
        # at most the bytes of verify_64k (10 f16 layers of 65,540 positions)
        n = _logint(rng, 200, 262000 if fmt == 0 else 131000)
        layers = max(1, min(rng.choice([1, 2, 10]), 655400 // (n * (1 + fmt))))
        start = rng.choice([0, 0, 0, rng.randrange(0, n // 2)])
        return dict(kind=kind, fmt=fmt, layers=layers, ntok=rng.choice([1, 1, 2, 3, 4, 4]), n=n, start=start,
                    out=rng.choice(["plain", "gate", "g16"]))
    if kind == "block":
        return dict(kind=kind, fmt=fmt, T=_logint(rng, 5, 512), n0=_logint(rng, 64, 28000 if fmt == 0 else 16000))
    if kind == "flint_step":
        return dict(kind=kind, fmt=fmt, n=_logint(rng, 200, 32000))
    if kind == "flint_block":
        return dict(kind=kind, fmt=fmt, T=_logint(rng, 5, 512), n0=_logint(rng, 64, 20000))
    return dict(kind=kind, fmt=fmt, p=_logint(rng, 100, 16384))


# ---- inputs: from the seed alone, on the GPU ----

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _theta(p0, p1, count, base):
    """theta_i of positions [p0, p1): theta_0 = pos, theta_{i+1} = theta_i * base^(-1/count), each step in f32."""
    scale = np.float32(float(base) ** (-1.0 / count))
    th = np.empty((p1 - p0, count), np.float32)
    th[:, 0] = np.arange(p0, p1, dtype=np.float32)
    for i in range(1, count):
        th[:, i] = th[:, i - 1] * scale
    return torch.from_numpy(th).to("cuda")


def _rope_rows(p0, p1, count, base):
    th = _theta(p0, p1, count, base).double()
    return torch.cat([th.cos(), th.sin()], 1).float().contiguous()


def _ctx(n):
    return max(4096, (n + 1023) // 1024 * 1024)


def _kv_rows(g, fmt, p):
    """K and V rows of p positions in the store's element type (f16 as bit patterns), [p][heads][dim] flattened."""
    k, v = _randn(g, p, 512), _randn(g, p, 512)
    return (k.half(), v.half()) if fmt == 0 else (k, v)


def _bits(x):
    return x.view(torch.int16) if x.dtype == torch.float16 else x


def _step_inputs(case, seed):
    """Per layer: the cache's rows [0, n - 1), then for both steps k_normed, v, q and the gate source."""
    g = _gen(seed)
    nt, per = case["ntok"], []
    for _ in range(case["layers"]):
        rows = _kv_rows(g, case["fmt"], case["n"] - 1)
        steps = []
        for _ in range(2):
            steps.append((_randn(g, nt, 2, 256), _randn(g, nt, 512), _randn(g, nt, 16, 256), _randn(g, nt, 16, 512)))
        per.append((rows, steps))
    return per


def _block_inputs(case, seed):
    g = _gen(seed)
    T = case["T"]
    rows = _kv_rows(g, case["fmt"], case["n0"])
    return dict(rows=rows, qf=_randn(g, T, 16, 512), kb=_randn(g, T, 2, 256), v=_randn(g, T, 512),
                qw=1 + 0.1 * _randn(g, 256), kw=1 + 0.1 * _randn(g, 256))


def _flint_inputs(case, seed):
    g = _gen(seed)
    T = case.get("T", 1)
    n0 = case["n0"] if "T" in case else case["n"] - 1
    layers = []
    for sliding in (True, False):
        rows = _kv_rows(g, case["fmt"], min(n0, mf.RING_SWA) if sliding else n0)
        layers.append(dict(sliding=sliding, rows=rows, q=_randn(g, T, 32, 128), k=_randn(g, T, 4, 128),
                           v=_randn(g, T, 4, 128), sinks=_randn(g, 32)))
    return T, n0, layers


def _put_rows(st, layer, rows):
    p = rows[0].shape[0]
    for which, x in ((mk.K, rows[0]), (mk.V, rows[1])):
        st.write_rows(layer, which, 0, p, _bits(x).contiguous())


# ---- what the program holds before the call ----

def prepare(case, seed):
    return {"step": _prepare_step, "block": _prepare_block, "flint_step": _prepare_flint,
            "flint_block": _prepare_flint, "rows": _prepare_rows}[case["kind"]](case, seed)


def _vp(t):
    return ctypes.c_void_p(t.data_ptr())


def _prepare_step(case, seed):
    n, nt, layers, out = case["n"], case["ntok"], case["layers"], case["out"]
    st = mk.KvStore(layers, _ctx(n + KEEP + nt), case["fmt"])
    keep, calls = [], []
    for s in range(2):
        pos = n - 1 + s * _advance(case)
        tab = _rope_rows(pos, pos + nt, 32, 1e7)
        keep.append(tab)
        calls.append((pos + 1, _vp(tab), []))
    outs = []
    for layer, (rows, steps) in enumerate(_step_inputs(case, seed)):
        _put_rows(st, layer, rows)
        for s, (kn, v, q, gs) in enumerate(steps):
            o = torch.empty((nt, 16, 256), dtype=torch.float16 if out == "g16" else torch.float32, device="cuda")
            keep += [kn, v, q, gs]
            outs.append(o)
            calls[s][2].append((layer, _vp(kn), _vp(v), _vp(q), _vp(o), None if out == "plain" else _vp(gs)))
    st.sync()
    torch.cuda.synchronize()
    return dict(kind="step", st=st, nt=nt, start=case["start"], calls=calls, outs=outs, keep=keep,
                fn=mk.lib().mkv_append_decode_g16 if out == "g16" else mk.lib().mkv_append_decode)


def _advance(case):
    return KEEP if case["ntok"] == 4 else 1


def _prepare_block(case, seed):
    x = _block_inputs(case, seed)
    T, n0 = case["T"], case["n0"]
    st = mk.KvStore(1, _ctx(n0 + T), case["fmt"])
    _put_rows(st, 0, x.pop("rows"))
    x["tab"] = st.rope_table_dev(n0, T)
    x.update(q=torch.empty((T, 16, 256), device="cuda"), kn=torch.empty((T, 2, 256), device="cuda"),
             out=torch.empty((T, 16, 256), device="cuda"))
    torch.cuda.synchronize()
    return dict(kind="block", st=st, n0=n0, **x)


def _prepare_flint(case, seed):
    T, n0, layers = _flint_inputs(case, seed)
    st = mf.FlintStore(2, _ctx(n0 + T), case["fmt"], [x["sliding"] for x in layers])
    tab = _rope_rows(n0, n0 + T, 64, FLINT_BASE)
    for i, x in enumerate(layers):
        _put_rows(st, i, x.pop("rows"))  # a ring's row r: the last position below n0 that is r modulo the ring
        x.update(qr=torch.empty_like(x["q"]), kr=torch.empty_like(x["k"]), out=torch.empty_like(x["q"]))
    torch.cuda.synchronize()
    state = dict(kind=case["kind"], st=st, T=T, n0=n0, tab=tab, layers=layers)
    if case["kind"] == "flint_step":
        state["calls"] = [tuple(_vp(x[k]) for k in ("q", "k", "v", "sinks", "qr", "kr", "out")) for x in layers]
        state["ptab"] = _vp(tab)
    return state


def _prepare_rows(case, seed):
    p, fmt = case["p"], case["fmt"]
    src, dst = mk.KvStore(1, _ctx(p), fmt), mk.KvStore(1, _ctx(p), fmt)
    _put_rows(src, 0, _kv_rows(_gen(seed), fmt, p))
    dt = torch.int16 if fmt == 0 else torch.float32
    buf = [torch.empty((p, 2, 256), dtype=dt, device="cuda") for _ in range(4)]
    torch.cuda.synchronize()
    return dict(kind="rows", src=src, dst=dst, p=p, buf=buf)


# ---- one pass ----

def run(state):
    return {"step": _run_step, "block": _run_block, "flint_step": _run_flint_step, "flint_block": _run_flint_block,
            "rows": _run_rows}[state["kind"]](state)


def _ok(rc):
    if rc != 0:
        raise mk.MkvError(rc, mk.lib().mkv_last_error().decode())


def _run_step(s):
    st, fn, nt, start = s["st"], s["fn"], s["nt"], s["start"]
    h = st.handle
    for i, (n, tab, layers) in enumerate(s["calls"]):
        if i:  # the rejected drafts' positions are given back; the next step's append overwrites them
            st.set_len(n - 1)
        for layer, kn, v, q, o, gs in layers:
            _ok(fn(h, layer, n, nt, kn, v, tab, q, start, SCALE, o, gs))
    return s["outs"]


def _run_block(s):
    st, n0 = s["st"], s["n0"]
    st.qk_norm_rope(n0, s["qf"], s["kb"], s["qw"], s["kw"], EPS, q_out=s["q"], kn_out=s["kn"])
    st.append(0, n0, s["kn"], s["v"], s["tab"])
    st.prefill(0, s["q"], n0 + 1, out=s["out"], gate_src=s["qf"])
    return [s["q"], s["kn"], s["out"]]


def _run_flint_step(s):
    lib, h, n0, tab = mf.lib(), s["st"].handle, s["n0"], s["ptab"]
    for layer, (q, k, v, sinks, qr, kr, out) in enumerate(s["calls"]):
        _ok(lib.mfl_rope(h, 1, 32, q, tab, qr))
        _ok(lib.mfl_rope(h, 1, 4, k, tab, kr))
        _ok(lib.mfl_append(h, layer, n0, 1, kr, v))
        _ok(lib.mfl_attend(h, layer, n0, 1, qr, sinks, out))
    return [x["out"] for x in s["layers"]]


def _run_flint_block(s):
    st, n0, tab = s["st"], s["n0"], s["tab"]
    for layer, x in enumerate(s["layers"]):
        st.rope(x["q"], tab, out=x["qr"])
        st.rope(x["k"], tab, out=x["kr"])
        st.append(layer, n0, x["kr"], x["v"])
        st.attend(layer, n0, x["qr"], x["sinks"], out=x["out"])
    return [x["out"] for x in s["layers"]]


def _run_rows(s):
    src, dst, p, b = s["src"], s["dst"], s["p"], s["buf"]
    for i, which in enumerate((mk.K, mk.V)):
        src.read_rows(0, which, 0, p, out=b[i])
        dst.write_rows(0, which, 0, p, b[i])
        dst.read_rows(0, which, 0, p, out=b[2 + i])
    return b


# ---- what a pass cannot do without ----

def work(case):
    kind, bpe = case["kind"], 2 + 2 * case["fmt"]
    if kind == "step":
        n, nt = case["n"], case["ntok"]
        by = fl = 0
        for s in range(2):
            first = n + s * _advance(case)
            keys = first + nt - 1 - case["start"]
            by += 2 * 512 * bpe * keys + 4 * nt * (512 + 512 + 64 + 4096 + (0 if case["out"] == "plain" else 4096))
            by += nt * 4096 * (2 if case["out"] == "g16" else 4)
            fl += 4 * 256 * 16 * sum(first + t - case["start"] for t in range(nt))
        return dict(bytes=by * case["layers"], flops=fl * case["layers"])
    if kind == "block":
        T, n0 = case["T"], case["n0"]
        by = 2 * 512 * bpe * (n0 + 2 * T)  # the cache read once, the new rows written and read
        by += 4 * T * (8192 + 512 + 512 + 64) + 4 * T * (4096 + 512 + 4096)
        return dict(bytes=by, flops=4 * 256 * 16 * sum(n0 + 1 + t for t in range(T)))
    if kind in ("flint_step", "flint_block"):
        T = case.get("T", 1)
        n0 = case["n0"] if "T" in case else case["n"] - 1
        by = fl = 0
        for win in (513, n0 + T):
            by += 2 * 512 * bpe * (min(n0, win - 1) + 2 * T) + 4 * T * (4096 * 2 + 512 * 2 + 128)
            fl += 4 * 128 * 32 * sum(min(n0 + t + 1, win) for t in range(T))
        return dict(bytes=by, flops=fl)
    # rows: per K and V, read out (2 x), written in (2 x), read out again (2 x)
    return dict(bytes=2 * 6 * case["p"] * 512 * bpe, flops=0)


# About four times the largest relative error against float64 that the listed cases and thirty drawn ones showed
# (exact() below). f16 arithmetic (Q and P rounded to f16, 2^-11 each, averaged over the keys) 3.0e-4, with the f16
# output 3.7e-4; f32-class arithmetic (f32 sums, the split operands' 2^-22) up to 8.6e-7, with the f16 output 2.2e-4.
def tolerance(case):
    if case["kind"] == "rows":
        return "exact"
    if case.get("out") == "g16":
        return dict(rel=1.5e-3 if _f16_class(case) else 9e-4)
    return dict(rel=1.2e-3 if _f16_class(case) else 3.5e-6)


def _f16_class(case):
    """The f16 store's arithmetic with Q and P in f16: verifies without a window, blocks of 64 tokens or more."""
    if case["fmt"] == 1 or case["kind"].startswith("flint"):
        return False
    return case["T"] > 63 if case["kind"] == "block" else case["ntok"] > 1 and case["start"] == 0


# ---- the same in float64, by plain torch ----

def _rope64(x, p0, base, rot):
    """x [T][heads][dim] float64: the first `rot` dims rotated in pairs (i, i + rot / 2) by the positions' angles (the
    f32 angles of the reference's table)."""
    T, h = x.shape[0], rot // 2
    th = _theta(p0, p0 + T, h, base).double()
    c, s = th.cos()[:, None], th.sin()[:, None]
    a, b = x[..., :h], x[..., h:rot]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., rot:]], -1)


def _stored(x, fmt):
    return x.half().double() if fmt == 0 else x.double()


def _attend64(q, k, v, first, start, scale, group, sinks=None, win=0):
    """q [T][heads][d]; k, v [keys][kv heads][d], key j at position j; token t sees [max(start, window), first + t)."""
    T, H, d = q.shape
    out = torch.empty_like(q)
    pos = torch.arange(k.shape[0], device=q.device)
    end = first + torch.arange(T, device=q.device)
    lo = torch.clamp(end - win, min=start) if win else torch.full_like(end, start)
    hide = (pos[None] >= end[:, None]) | (pos[None] < lo[:, None])
    for h in range(H):
        s = torch.matmul(q[:, h], k[:, h // group].t().contiguous()) * scale
        s.masked_fill_(hide, -math.inf)
        m = s.amax(1, keepdim=True)
        if sinks is not None:
            m = torch.maximum(m, sinks[h].double())
        w = (s - m).exp_()
        den = w.sum(1, keepdim=True)
        if sinks is not None:
            den = den + (sinks[h].double() - m).exp()
        out[:, h] = torch.matmul(w, v[:, h // group].contiguous()) / den
    return out


def exact(case, seed):
    kind, fmt = case["kind"], case["fmt"]
    if kind == "rows":
        k, v = _kv_rows(_gen(seed), fmt, case["p"])
        k, v = (_bits(x).view(-1, 2, 256) for x in (k, v))
        return [k, v, k, v]
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "block":
        return _exact_block(case, seed)
    T, n0, layers = _flint_inputs(case, seed)
    outs = []
    for x in layers:
        q = _rope64(x["q"].double(), n0, FLINT_BASE, 128)
        nk = _stored(_rope64(x["k"].double(), n0, FLINT_BASE, 128), fmt)
        nv = _stored(x["v"], fmt)
        k, v = (r.double().view(-1, 4, 128) for r in x["rows"])
        if x["sliding"] and n0 > mf.RING_SWA:  # ring rows to the positions they hold; older ones are out of every window
            order = torch.arange(n0 - mf.RING_SWA, n0, device="cuda") % mf.RING_SWA
            k, v = k[order], v[order]
        base = n0 - k.shape[0]
        k, v = torch.cat([k, nk]), torch.cat([v, nv])
        outs.append(_attend64(q, k, v, n0 + 1 - base, 0, 1 / math.sqrt(128), 8, x["sinks"],
                              mf.WINDOW if x["sliding"] else 0))
    return outs


def _exact_step(case, seed):
    n, nt, fmt = case["n"], case["ntok"], case["fmt"]
    outs = []
    for rows, steps in _step_inputs(case, seed):
        k, v = (r.double().view(-1, 2, 256) for r in rows)
        for s, (kn, nv, q, gs) in enumerate(steps):
            pos = n - 1 + s * _advance(case)
            k = torch.cat([k[:pos], _stored(_rope64(kn.double(), pos, 1e7, 64), fmt)])
            v = torch.cat([v[:pos], _stored(nv.view(nt, 2, 256), fmt)])
            o = _attend64(q.double(), k, v, pos + 1, case["start"], SCALE, 8)
            if case["out"] != "plain":
                o = o * torch.sigmoid(gs[..., 256:].double())
            outs.append(o)
    return outs


def _exact_block(case, seed):
    x = _block_inputs(case, seed)
    T, n0, fmt = case["T"], case["n0"], case["fmt"]

    def norm(a, w):
        a = a.double()
        return a / torch.sqrt((a * a).mean(-1, keepdim=True) + EPS) * w.double()

    q = _rope64(norm(x["qf"][..., :256], x["qw"]), n0, 1e7, 64)
    kn = norm(x["kb"], x["kw"])
    k = torch.cat([x["rows"][0].double().view(-1, 2, 256), _stored(_rope64(kn, n0, 1e7, 64), fmt)])
    v = torch.cat([x["rows"][1].double().view(-1, 2, 256), _stored(x["v"].view(T, 2, 256), fmt)])
    o = _attend64(q, k, v, n0 + 1, 0, SCALE, 8) * torch.sigmoid(x["qf"][..., 256:].double())
    return [q, kn, o]
