"""Row transforms and damping at every row length, with row counts that leave
the last block part empty: both directions against the oracle, damping with
and without the PSATD advance, and the transposed damping by <L x, y> =
<x, L^T y>.  Bounds (relative L2): FP64 1e-12; FP32 1e-5 - per field some
thirty roundings of 6e-8 along a transform and its product, three times that
for the split product's truncated terms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

LENGTHS = [16, 32, 64, 128, 256, 512, 1024, 2048, 4096]


@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("Nx", LENGTHS)
def test_rows(precision, Nx):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import chimeracl_amd as CA
    from chimeracl_amd import _lib
    from chimeracl_amd.methods.generic_methods_hip import Communicator
    from oracle import oracle as O
    from tests import simpair as S
    M = 1
    g = S.tiny_grid(Nx=Nx, Nr=12 if Nx > 16 else 134, M=M, damp=max(2, Nx // 16))
    solver = CA.Solver(dict(g), Communicator(precision=precision))
    s = O.OracleSolver(dict(g))
    tol = 1e-12 if precision == "f64" else 1e-5
    rng = np.random.default_rng(Nx)

    def fill(name, cplx):
        v = rng.normal(0, 1, s.f[name].shape) + (1j * rng.normal(0, 1, s.f[name].shape) if cplx else 0)
        s.f[name][...] = v
        solver.DataDev[name].copy_(torch.from_numpy(np.ascontiguousarray(v)))

    def same(name, rows=slice(None)):
        assert S.rel_l2(S.field_host(solver, name)[rows], s.f[name][rows]) < tol, name

    fb = [f"{f}{c}_fb_m{m}" for f in "EG" for c in "xyz" for m in range(M + 1)]
    for m in range(M + 1):
        for n in ("rho", "Jx", "Jy", "Jz"):
            fill(f"{n}_m{m}", m > 0)
    for sim in (solver, s):
        sim.fb_transform(scals=["rho"], vects=["J"], dir=0)
    for n in ("rho", "Jx", "Jy", "Jz"):
        for m in range(M + 1):
            same(f"{n}_fb_m{m}")
    for n in fb + [f"{f}{c}_fb_m{m}" for f in ("dN0", "dN1") for c in "xyz" for m in range(M + 1)]:
        fill(n, True)
    solver.damp_edges(("E", "G"))
    s.damp_fields()
    for n in fb:
        same(n)
    solver.damp_edges(("E", "G"), advance_with=("J", "dN0", "dN1"))
    s.push_fields()
    s.damp_fields()
    for n in fb:
        same(n)
    solver.fb_transform(vects=["E"], dir=1)
    s.fb_transform(vects=["E"], dir=1)
    for n in S.real_names(M, flds=("E",), scal=()):
        same(n, slice(1, None))
    if precision != "f64":
        return
    from chimeracl_amd.adjoint import _fb_arr

    def planes(f):
        return [[solver.DataDev[f"{f}{c}_fb_m{m}"] for m in range(M + 1)] for c in "xyz"]

    def dot(v, w):
        return sum(float((torch.view_as_real(a) * torch.view_as_real(b)).sum())
                   for p, q in zip(v, w) for a, b in zip(p, q))

    x = {f: [[t.clone() for t in c] for c in planes(f)] for f in ("E", "G", "J", "dN0", "dN1")}
    solver.damp_edges(("E", "G"), advance_with=("J", "dN0", "dN1"))
    y = {f: [[torch.randn_like(t) for t in c] for c in x[f]] for f in ("E", "G")}
    lhs = sum(dot(planes(f), y[f]) for f in "EG")
    size = sum(dot(planes(f), planes(f)) for f in "EG") * sum(dot(y[f], y[f]) for f in "EG")
    for f in ("J", "dN0", "dN1"):
        y[f] = [[torch.zeros_like(t) for t in c] for c in x[f]]
    _lib.call("chm_damp_fields_adj_f64", solver._sp, _fb_arr(y["E"]), _fb_arr(y["G"]), None,
              _fb_arr(y["J"]), _fb_arr(y["dN0"]), _fb_arr(y["dN1"]), 0)
    assert abs(lhs - sum(dot(x[f], y[f]) for f in x)) < 1e-12 * size ** 0.5


@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("Nx", LENGTHS)
def test_twiddle_orders(precision, Nx):
    """Both forms of the twiddle table give the same bits."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import chimeracl_amd as CA
    from chimeracl_amd.methods.generic_methods_hip import Communicator
    from tests import simpair as S
    M = 1
    g = S.tiny_grid(Nx=Nx, Nr=12, M=M, damp=max(2, Nx // 16))
    solver = CA.Solver(dict(g), Communicator(precision=precision))
    D, out = solver.DataDev, []
    for plain in (False, True):
        if plain:
            solver._sp.twiddle_form = 0
        gen = torch.Generator(device="cuda").manual_seed(Nx)
        for n in sorted(k for k in D if k.startswith(("E", "G", "J", "rho", "dN")) and "_m" in k):
            D[n].copy_(torch.randn(D[n].shape, generator=gen, device="cuda", dtype=D[n].dtype))
        solver.fb_transform(scals=["rho"], vects=["J"], dir=0)
        solver.damp_edges(("E", "G"), advance_with=("J", "dN0", "dN1"))
        solver.fb_transform(vects=["E"], dir=1)
        out.append({n: D[n].clone() for n in D if n.startswith(("E", "G", "J", "rho")) and "_m" in n})
    for n in out[0]:
        assert torch.equal(out[0][n], out[1][n]), n
