"""chm_sort_from_keys with buckets of many tiles, which the bucket sort counts
in chunks of 32 tiles: buckets that begin and end on and beside chunk borders,
neighbours that share a chunk, one bucket with (almost) every key, with 8- and
11-bit digits, small and large tiles; against numpy's stable argsort (exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

T = 4096  # keys of a tile below 2^23 keys, 2 T from there on where the buckets are large

# (Nx, Nr, cells of a bucket, {bucket: keys}, keys everywhere)
CASES = [
    (512, 257, 2048, {0: 32 * T}, 60000), (512, 257, 2048, {0: 32 * T - 1}, 60000),
    (512, 257, 2048, {3: 64 * T}, 70000), (512, 257, 2048, {3: 31 * T, 4: 33 * T}, 70000),
    (512, 257, 2048, {2: 95 * T + 5, 3: 1, 5: 63 * T}, 131072), (512, 257, 2048, {63: 130 * T}, 3),
    (512, 257, 2048, {10: 300 * T + 17, 11: 40 * T, 12: 20 * T, 13: 64 * T}, 200000),
    (65, 65, 256, {0: 200 * T, 16: 33 * T + 1}, 40000),
    (2048, 256, 2048, {100: 1 << 23}, 600000), (64, 64, 256, {7: 40 * 2 * T, 8: 1 << 23}, 300000),
]


@pytest.mark.parametrize("Nx,Nr,cells,heavy,spread", CASES)
def test_sort_of_large_buckets(Nx, Nr, cells, heavy, spread):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from chimeracl_amd import _lib
    nbins = (Nx - 1) * (Nr - 1) + 1
    rng = np.random.default_rng(len(heavy) + Nx)
    parts = [rng.integers(0, nbins, spread)]
    for b, k in heavy.items():
        parts.append(rng.integers(b * cells, min((b + 1) * cells, nbins), k))
    key = rng.permutation(np.concatenate(parts)).astype(np.uint32)
    n = key.size
    dev = dict(dtype=torch.int32, device="cuda")
    k = torch.from_numpy(key.view(np.int32)).cuda()
    off, srt, stay = torch.empty(nbins + 1, **dev), torch.empty(n, **dev), torch.empty(1, **dev)
    nws = _lib.lib.chm_sort_workspace_bytes(n, nbins)
    ws = torch.full((nws,), 0xA5, dtype=torch.uint8, device="cuda")
    g = _lib.Grid(Nx=Nx, Nr=Nr, M=0)
    ref = np.argsort(key, kind="stable")
    want = np.searchsorted(key[ref], np.arange(nbins + 1), side="left")
    for _ in range(2):  # a used workspace too
        _lib.call("chm_sort_from_keys", n, g, k.data_ptr(), off.data_ptr(), srt.data_ptr(),
                  stay.data_ptr(), ws.data_ptr(), nws, None)
        assert np.array_equal(srt.cpu().numpy().view(np.uint32), ref)
        assert np.array_equal(off.cpu().numpy().view(np.uint32), want)
        assert int(stay.item()) == want[nbins - 1]
        at = _lib.lib.chm_sort_sorted_keys(ws.data_ptr(), n, g) - ws.data_ptr()
        assert np.array_equal(ws[at:at + 4 * n].cpu().numpy().view(np.uint32), key[ref])
