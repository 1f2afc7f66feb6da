"""The push and keys of the particles outside the grid, which the J sums' tail
blocks and the pre-pushing gather's own launch make: fewer and more of them
than those have lanes, all of them and none, against push_coords (bit for
bit)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _species(g, precision, n, out):
    import chimeracl_amd as CA
    from chimeracl_amd import config as C
    from chimeracl_amd.methods.generic_methods_hip import Communicator
    comm = Communicator(precision=precision)
    s = CA.Solver(dict(g), comm)
    cfg, _ = C.species_config("C1", s.Args, ppc=(2, 2, 4), dens=0.002)
    rng = np.random.default_rng(n)
    th, r = 2 * np.pi * rng.random(n), s.Args["dr"] * (0.5 + rng.random(n) * (s.Args["Nr"] - 4))
    a = {"x": g["Xmin"] + s.Args["dx"] * (1.5 + rng.random(n) * (s.Args["Nx"] - 4)),
         "y": r * np.cos(th), "z": r * np.sin(th), "w": rng.random(n)}
    a["y"][rng.random(n) < out] += 1e3
    a.update({k: rng.normal(0, 0.3, n) for k in ("px", "py", "pz")})
    a["g_inv"] = 1 / np.sqrt(1 + a["px"] ** 2 + a["py"] ** 2 + a["pz"] ** 2)
    e = CA.Particles(dict(cfg), comm)
    e.add_particles(source=C.ParticleSource(a))
    gen = torch.Generator(device="cuda").manual_seed(5)
    for c in "xyz":
        for f in "EB":
            for m in range(g["M"] + 1):
                t = s.DataDev[f"{f}{c}_m{m}"]
                t.copy_(torch.randn(t.shape, generator=gen, dtype=t.dtype, device="cuda"))
    return s, e


@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("n,out", [(1, 1.0), (65, 0.5), (131073, 1.0), (600000, 0.9), (70000, 0.0)])
def test_push_of_particles_outside(precision, n, out):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from tests import simpair as S
    g = S.tiny_grid(Nx=64, Nr=24, M=2, damp=2)
    (s, e), (t, f) = (_species(g, precision, n, out) for _ in range(2))
    # J deposit with the half push
    e.sort_parts(s)
    s.depose_currents([e], push_half=True)
    f.sort_parts(t)
    t.depose_currents([f])
    f.push_coords(mode="half", grid=t)
    for k in ("x", "y", "z", "indx_in_cell"):
        assert torch.equal(e.DataDev[k], f.DataDev[k]), k
    # gather with the next half push
    e.sort_parts(s)
    s.gather_and_push([e], prepush=True)
    f.sort_parts(t)
    t.gather_and_push([f])
    f.push_coords(mode="half", grid=t)
    for k, q in (("xh", "x"), ("yh", "y"), ("zh", "z"), ("px", "px"), ("py", "py"), ("pz", "pz"),
                 ("g_inv", "g_inv"), ("indx_in_cell", "indx_in_cell")):
        assert torch.equal(e.DataDev[k], f.DataDev[q]), k
