"""The DHT products of all modes in one launch: more products than a launch
takes (six fields, M = 4), one mode, column and row tiles with remainders, and
the 128 x 128 split-BF16 tiles, against the oracle on the solver's own
tables, the inverse being ill-conditioned (FP64, 1e-12 relative L2)
and the FP64 form (mixed, 1e-5: three times the thirty-odd FP32 roundings of
6e-8 along a transform)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _solver(Nx, Nr, M, precision):
    import chimeracl_amd as CA
    from chimeracl_amd.methods.generic_methods_hip import Communicator
    from tests import simpair as S
    g = S.tiny_grid(Nx=Nx, Nr=Nr, M=M, damp=2)
    return g, CA.Solver(dict(g), Communicator(precision=precision))


@pytest.mark.parametrize("Nx,Nr,M", [(16, 6, 4), (32, 66, 4), (64, 65, 0), (128, 130, 3)])
def test_products_fp64(Nx, Nr, M):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from oracle import oracle as O
    from tests import simpair as S
    g, s = _solver(Nx, Nr, M, "f64")
    o = O.OracleSolver(dict(g))
    for m in range(M + 1):  # the products are compared, on one set of tables
        for k, n in (("DHT", "DHT_m"), ("DHT_inv", "DHT_inv_m")):
            o.dht[k][m] = s.DataDev[f"{n}{m}"].cpu().numpy()
    rng = np.random.default_rng(Nr)
    for f in "EB":
        for c in "xyz":
            for m in range(M + 1):
                n = f"{f}{c}_fb_m{m}"
                v = rng.normal(0, 1, o.f[n].shape) + 1j * rng.normal(0, 1, o.f[n].shape)
                o.f[n][...] = v
                s.DataDev[n].copy_(torch.from_numpy(v))
    for sim in (s, o):
        sim.fb_transform(vects=["E", "B"], dir=1)
        sim.fb_transform(vects=["E", "B"], dir=0)
    for f in "EB":
        for c in "xyz":
            for m in range(M + 1):
                n = f"{f}{c}_fb_m{m}"
                assert S.rel_l2(S.field_host(s, n), o.f[n]) < 1e-12, n


@pytest.mark.parametrize("Nx,Nr,M", [(16, 6, 4), (2048, 258, 1), (2048, 130, 4), (64, 129, 0)])
def test_products_mixed(Nx, Nr, M):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    _, a = _solver(Nx, Nr, M, "mixed")
    _, b = _solver(Nx, Nr, M, "f64")
    gen = torch.Generator(device="cuda").manual_seed(Nr)
    names = [f"{f}{c}_m{m}" for f in "EB" for c in "xyz" for m in range(M + 1)]
    for n in names:
        t = a.DataDev[n]
        t.copy_(torch.randn(t.shape, generator=gen, device="cuda", dtype=t.dtype))
        b.DataDev[n].copy_(t)
    for sim in (a, b):
        sim.fb_transform(vects=["E", "B"], dir=0)
    for n in names:
        x, y = (s.DataDev[n.replace("_m", "_fb_m")] for s in (a, b))
        assert float((x - y).norm() / y.norm()) < 1e-5, n
