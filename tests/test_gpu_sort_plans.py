"""chm_sort_from_keys where its plan changes: one digit pass, the bucket sort
with small and large tiles, LSD passes for few keys on many cells, skewed
buckets, tiles that end on and beside bucket borders; against numpy's stable
argsort and searchsorted (exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# (Nx, Nr, n, keys): 9 .. 22-bit keys
CASES = [
    (5, 3, 1, "random"), (5, 3, 5000, "random"), (33, 33, 70000, "random"),       # one pass
    (46, 46, 40000, "random"), (65, 33, 4096, "last"),                            # 11 bits
    (65, 65, 200000, "near"), (65, 65, 16 * 4096, "few"), (256, 64, 250976, "near"),  # 8-bit digits
    (256, 64, 300, "random"), (4096, 512, 3000, "near"),                          # LSD: few keys
    (1024, 201, 700001, "near"), (512, 257, 1 << 20, "skew"),                     # 11-bit digits
    (2048, 256, (1 << 23) - 1, "near"), (2048, 256, (1 << 23) + 5, "near"),       # below and above the
    (2048, 256, 1 << 23, "skew"), (60, 40, (1 << 23) + 77, "random"),             # larger tiles
    (4096, 1024, (1 << 23) + 1, "near"), (64, 64, (1 << 23) + 3, "outside"),
]


def _keys(rng, nbins, n, how):
    top = nbins - 1
    if how == "random":
        return rng.integers(0, nbins, n)
    if how == "last":
        return np.full(n, top)
    if how == "few":
        return rng.choice(rng.integers(0, nbins, 3), n)
    if how == "outside":
        return np.where(rng.random(n) < 0.9, top, rng.integers(0, nbins, n))
    if how == "skew":  # half of the keys in one cell
        return np.where(rng.random(n) < 0.5, nbins // 3, rng.integers(0, nbins, n))
    k = np.sort(rng.integers(0, nbins, n)) + rng.integers(-40, 41, n)
    return np.clip(k, 0, top)


@pytest.mark.parametrize("Nx,Nr,n,how", CASES)
def test_sort_plans(Nx, Nr, n, how):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from chimeracl_amd import _lib
    nbins = (Nx - 1) * (Nr - 1) + 1
    key = _keys(np.random.default_rng(n + Nx), nbins, n, how).astype(np.uint32)
    dev = dict(dtype=torch.int32, device="cuda")
    k = torch.from_numpy(key.view(np.int32)).cuda()
    off, srt, stay = torch.empty(nbins + 1, **dev), torch.empty(n, **dev), torch.empty(1, **dev)
    nws = _lib.lib.chm_sort_workspace_bytes(n, nbins)
    ws = torch.full((nws,), 0xA5, dtype=torch.uint8, device="cuda")
    g = _lib.Grid(Nx=Nx, Nr=Nr, M=0)
    ref = np.argsort(key, kind="stable")
    for _ in range(2):  # a used workspace too
        _lib.call("chm_sort_from_keys", n, g, k.data_ptr(), off.data_ptr(), srt.data_ptr(),
                  stay.data_ptr(), ws.data_ptr(), nws, None)
        torch.cuda.synchronize()
        assert np.array_equal(srt.cpu().numpy().view(np.uint32), ref)
        want = np.searchsorted(key[ref], np.arange(nbins + 1), side="left")
        assert np.array_equal(off.cpu().numpy().view(np.uint32), want)
        assert int(stay.item()) == want[nbins - 1]
        at = _lib.lib.chm_sort_sorted_keys(ws.data_ptr(), n, g) - ws.data_ptr()
        assert np.array_equal(ws[at:at + 4 * n].cpu().numpy().view(np.uint32), key[ref])
