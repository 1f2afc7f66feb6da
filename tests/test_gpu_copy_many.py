"""chm_copy_many at the edges of its pieces: no bytes, fewer than 16, ends
beside multiples of 16 and of 64 KB, unaligned source or destination, zeros,
more arrays than a launch takes; and the double push against two pushes (bit
for bit)."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("so,do", [(0, 0), (1, 0), (0, 3), (8, 8), (None, 0), (None, 5)])
def test_copy_many(so, do):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from chimeracl_amd import _lib
    sizes = [0, 1, 15, 16, 17, 255, 4096, 65535, 65536, 65537, 3 * 65536 + 31]
    src = [torch.randint(0, 256, (n + 16,), dtype=torch.uint8, device="cuda") for n in sizes]
    dst = [torch.full((n + 32,), 7, dtype=torch.uint8, device="cuda") for n in sizes]
    n = len(sizes)
    s = (ctypes.c_void_p * n)(*(None if so is None else t.data_ptr() + so for t in src))
    d = (ctypes.c_void_p * n)(*(t.data_ptr() + do for t in dst))
    nb = (ctypes.c_int64 * n)(*sizes)  # kept: only addresses are passed on
    _lib.call("chm_copy_many", n, ctypes.addressof(s), ctypes.addressof(d), ctypes.addressof(nb), 0)
    for k, a, b in zip(sizes, src, dst):
        want = torch.full_like(b, 7)
        want[do:do + k] = 0 if so is None else a[so:so + k]
        assert torch.equal(b, want), k
    assert _lib.lib.chm_copy_many(_lib.CHM_COPY_MAXARR + 1, s, d, None, 0) == -1


@pytest.mark.parametrize("sfx,dt", [("f64", torch.float64), ("f32", torch.float32)])
@pytest.mark.parametrize("n", [1, 255, 1000])
def test_push_x_twice(sfx, dt, n):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from chimeracl_amd import _lib
    a = [torch.randn(n, dtype=dt, device="cuda") for _ in range(7)]
    x1, x2 = ([torch.empty_like(t) for t in a[:3]] for _ in range(2))
    p = lambda ts: [t.data_ptr() for t in ts]
    _lib.call(f"chm_push_x_twice_{sfx}", *p(a), 0.3, n, *p(x1), *p(x2), 0)
    x = [t.clone() for t in a[:3]]
    for want in (x1, x2):
        _lib.call(f"chm_push_x_{sfx}", *p(x), *p(a[3:]), 0.3, n, 0)
        for u, v in zip(x, want):
            assert torch.equal(u, v)
