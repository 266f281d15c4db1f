"""Row conversion (read_rows / write_rows) over ragged ranges: the 16-position kernel takes 16-byte aligned rows, the
element kernel the others. Both are compared with the rows themselves, bit for bit, and positions outside the range must
stay as they were."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# edges of the 4- and 8-position V groups, the 16-position work-group and the 32-position K block
RANGES = [(0, 1), (0, 8), (3, 5), (7, 9), (5, 37), (15, 17), (16, 48), (31, 97), (13, 1000)]


def _store(torch, model, fmt):
    if model == "kv":
        import mechta_amd as mk
        return mk.KvStore(1, 4096, fmt), (2, 256)
    from mechta_amd import flint as mf
    return mf.FlintStore(1, 1024, fmt, [False]), (4, 128)


def _buf(torch, n, shape, dt, aligned):
    """A device tensor [n][heads][dim] whose address is 16-byte aligned, or one element past such an address."""
    k = n * 512
    base = torch.zeros(k + 8, dtype=dt, device="cuda")
    off = 0 if aligned else 1
    t = base[off:off + k]
    assert (t.data_ptr() % 16 == 0) == aligned
    return t.view(n, *shape)


@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("model", ["kv", "flint"])
def test_rows_ragged(torch_gpu, model, fmt, aligned):
    torch = torch_gpu
    dt = torch.int16 if fmt == 0 else torch.float32
    r = np.random.default_rng(17 + fmt)
    st, shape = _store(torch, model, fmt)
    with st:
        for which in (0, 1):
            want = np.zeros((1024, *shape), np.int16 if fmt == 0 else np.float32)
            fill = r.integers(-30000, 30000, want.shape).astype(want.dtype)
            st.write_rows(0, which, 0, 1024, torch.from_numpy(fill).cuda())
            want[:] = fill
            for p0, p1 in RANGES:
                print(f"rows {model} fmt={fmt} which={which} aligned={aligned} [{p0}, {p1})", flush=True)
                new = r.integers(-30000, 30000, (p1 - p0, *shape)).astype(want.dtype)
                b = _buf(torch, p1 - p0, shape, dt, aligned)
                b.copy_(torch.from_numpy(new))
                st.write_rows(0, which, p0, p1, b)
                want[p0:p1] = new
                got = st.read_rows(0, which, 0, 1024).cpu().numpy()
                assert np.array_equal(got, want)
                o = _buf(torch, p1 - p0, shape, dt, aligned)
                st.read_rows(0, which, p0, p1, out=o)
                assert np.array_equal(o.cpu().numpy(), want[p0:p1])
