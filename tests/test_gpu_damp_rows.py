"""The damping with and without the update at every row length, few rows and
many, FP32 and FP64, against the two launches it stands for (advance_fields,
then the round trip made from the transforms' row lengths in float64)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("Nx,Nr,M", [(16, 4, 0), (32, 70, 1), (64, 24, 1), (128, 131, 2), (256, 66, 1),
                                     (512, 34, 3), (1024, 9, 1), (2048, 5, 1), (4096, 4, 1)])
@pytest.mark.parametrize("advance", [False, True])
def test_damping_rows(precision, Nx, Nr, M, advance):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import chimeracl_amd as CA
    from chimeracl_amd import config as C
    from chimeracl_amd.methods.generic_methods_hip import Communicator
    s = CA.Solver(C.grid_config("C1", Nx=Nx, Nr=Nr, M=M, DampCells=max(2, Nx // 16)),
                  Communicator(precision=precision))
    D = s.DataDev
    gen = torch.Generator(device="cuda").manual_seed(Nx)
    names = {f: [f"{f}{c}_fb_m{m}" for c in "xyz" for m in range(M + 1)]
             for f in ("E", "G", "J", "dN0", "dN1")}
    for f in names:
        for k in names[f]:
            D[k].copy_(torch.randn(D[k].shape, generator=gen, dtype=torch.complex128, device="cuda"))
    start = {k: D[k].clone() for f in ("E", "G") for k in names[f]}
    if advance:  # the update alone, by its own launch
        s.advance_fields(vecs=["E", "G", "J", "dN0", "dN1"])
    want = {k: D[k].to(torch.complex128, copy=True) for f in ("E", "G") for k in names[f]}
    for k, v in start.items():
        D[k].copy_(v)
    f = np.ones(Nx)
    nd, prof = s.Args["DampProfile"].size, s.Args["DampProfile"]
    f[:nd] *= prof
    for x in range(Nx - nd + 1, Nx):
        f[x] *= prof[Nx - x]
    f = torch.from_numpy(f).cuda()
    kx = torch.from_numpy(s.Args["kx"]).cuda()
    ph = torch.exp(1j * kx * s.Args["Xmin"])
    for k, v in want.items():
        u = torch.fft.ifft(v * ph, dim=1)
        g = torch.complex(u.real, torch.zeros_like(u.real)) if k.endswith("_m0") else u
        want[k] = v - torch.fft.fft(u - f * g, dim=1) * ph.conj()
    s.damp_edges(("E", "G"), advance_with=("J", "dN0", "dN1") if advance else None)
    # rounding of two transforms of length Nx (log2 Nx stages each) and of four
    # products with phases and profile: (2 log2 Nx + 8) eps of the row's rms, on
    # values that the update may scale by its coefficients first (<= 4 more)
    eps = np.finfo(np.float64 if precision == "f64" else np.float32).eps
    tol = (2 * np.log2(Nx) + 12) * eps
    for k, v in want.items():
        d = (D[k].to(torch.complex128) - v).abs()
        assert float(d.norm() / v.norm()) < tol, (k, float(d.norm() / v.norm()), tol)
