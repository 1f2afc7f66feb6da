"""The gather in memory order against the sorted order, bit for bit (FP32, and
FP64 without modes):
every mode count, with and without the next push, particles outside the grid,
ids past Np_stay, the last block part empty, boxes that do not fit (a run that
goes over the end of a grid row) and a shuffled memory order, which keeps the
sorted one."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

NX, NR, N = 67, 24, 2**21 + 333


@pytest.mark.parametrize("pre", [False, True])
@pytest.mark.parametrize("sfx,M,drift", [
    ("f32", 0, 0.5), ("f32", 1, 0.5), ("f32", 2, 0.5), ("f32", 3, 0.5), ("f32", 4, 0.5),
    ("f32", 1, 0.0), ("f32", 2, None), ("f32", 1, None), ("f64", 0, 0.5), ("f64", 0, None),
    ("f64", 1, 0.5)])
def test_gather_orders(sfx, M, drift, pre):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from chimeracl_amd import _lib
    real = torch.float64 if sfx == "f64" else torch.float32
    gen = torch.Generator(device="cuda").manual_seed(M)

    def ru(*s):
        return torch.rand(*s, generator=gen, device="cuda", dtype=real)

    def p(t):
        return t.data_ptr() if t is not None else None

    cell = torch.arange(N, device="cuda") * ((NX - 3) * (NR - 2)) // N
    x, r = 1 + cell % (NX - 3) + ru(N), cell // (NX - 3) + ru(N)
    if drift is None:
        o = torch.randperm(N, generator=gen, device="cuda")
        x, r = x[o], r[o]
    else:
        x += drift * (2 * ru(N) - 1)
        r = (r + drift * (2 * ru(N) - 1)).abs()
        x[::101] += 1e3  # outside
    th = 6.3 * ru(N)
    x, y, z = x.contiguous(), r * torch.cos(th), r * torch.sin(th)
    g = _lib.Grid(Nx=NX, Nr=NR, M=M, xmin=0.0, dx_inv=1.0, rmin=-0.5, dr_inv=1.0)
    nb = (NX - 1) * (NR - 1) + 1
    i32 = dict(dtype=torch.int32, device="cuda")
    keys, srt, off = torch.empty(N, **i32), torch.empty(N, **i32), torch.empty(nb + 1, **i32)
    nst, flag = torch.zeros(1, **i32), torch.zeros(1, **i32)
    ws = torch.empty(_lib.lib.chm_sort_workspace_bytes(N, nb), dtype=torch.uint8, device="cuda")
    _lib.call(f"chm_index_sort_{sfx}", p(x), p(y), p(z), N, g, p(keys), p(off), p(srt), p(nst), p(ws),
              ws.numel(), 0)
    skey = _lib.lib.chm_sort_sorted_keys(p(ws), N, g)
    E, B, keep = (_lib.Planes * 3)(), (_lib.Planes * 3)(), []
    for f in (E, B):
        for c in range(3):
            keep.append(ru(NR, NX) - 0.5)
            f[c].m0 = p(keep[-1])
            for m in range(M):
                keep.append(ru(NR, NX, 2) - 0.5)
                f[c].mc[m] = p(keep[-1])
    pid = torch.randperm(N, generator=gen, device="cuda").int()
    out = []
    for k in (None, keys.clone()):
        u = [torch.full((N,), v, device="cuda", dtype=real) for v in (0.1, -0.2, 0.3, 0.9)]
        h = [torch.zeros(N, device="cuda", dtype=real) for _ in range(3)] if pre else [None] * 3
        # the next keys over the present ones, as the step has them
        nk = (torch.zeros(N, **i32) if k is None else k) if pre else None
        _lib.call(f"chm_gather_push_keys_{sfx}", p(x), p(y), p(z), *map(p, u), N, p(srt), p(off),
                  p(nst), p(pid), skey, p(k), p(flag), 0.01, 0.02, *map(p, h), p(nk), g, E, B, 0)
        out.append(u + (h + [nk] if pre else []))
    assert flag.item() == (drift is not None and M < (4 if sfx == "f32" else 1))
    for a, b in zip(*out):
        assert torch.equal(a, b)
