"""The deposits with the planes' zeroing and post-processing in the node pass,
and the out-of-domain push in the sums' launch, against the separate calls
(zero_planes, deposit, postproc), bit for bit: one and two species, an
immobile one kept staged, few and many particles outside the grid."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("Nx,Nr,M,out", [(16, 4, 0, 0.0), (64, 24, 1, 0.1), (128, 33, 2, 0.9),
                                         (32, 17, 3, 0.0)])
def test_depose_stages(precision, Nx, Nr, M, out):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from chimeracl_amd import _lib
    from chimeracl_amd.methods.generic_methods_hip import ptr
    from tests import simpair as S
    g = S.tiny_grid(Nx=Nx, Nr=Nr, M=M, damp=2)
    a, _ = S.make_pair(g, None, precision=precision, with_oracle=False)
    b, _ = S.make_pair(g, None, precision=precision, with_oracle=False)
    rng = np.random.default_rng(Nx)
    n = a["eons"].Args["Np"]
    far = torch.from_numpy(rng.random(n) < out).cuda()
    mom = {k: torch.from_numpy(rng.normal(0, 0.3, n)) for k in ("px", "py", "pz")}
    for sim in (a, b):
        d = sim["eons"].DataDev
        d["y"][far] += 1e3
        for k, v in mom.items():
            d[k].copy_(v)
        for nm in [f + c for f in "J" for c in "xyz"] + ["rho"]:  # stale planes
            for m in range(M + 1):
                sim["solver"].DataDev[f"{nm}_m{m}"].fill_(3.0)
    for _ in range(2):
        s, e, i = a["solver"], a["eons"], a["ions"]
        s.depose_currents([e, i], push_half=True)
        s.depose_charge([e, i])
        s, e, i = b["solver"], b["eons"], b["ions"]
        e.sort_parts(s)
        i.sort_parts(s)
        d, w = e.DataDev, s._dep_ws()
        J = s._planes_arr(["Jx", "Jy", "Jz"])
        s.zero_planes(["Jx", "Jy", "Jz"])
        e._ensure_sort_buffers(s)
        s.call("chm_deposit_vector_push", ptr(d["sort_indx"]), ptr(d["cell_offset"]), *(
            ptr(d[k]) for k in ("x", "y", "z", "x", "y", "z", "px", "py", "pz", "g_inv", "w")), -1,
            e.Args["dt_2"], n, ptr(d["indx_in_cell"]), s._grid(), J, ptr(w), w.numel())
        s.postproc_depose_vector("J")
        e._keys_for, e.flag_sorted = s, False
        e.sort_parts(s)
        s.zero_planes(["rho"])
        for p, q in ((e, -1), (i, 1)):
            d = p.DataDev
            s.call("chm_deposit_scalar", ptr(d["sort_indx"]), ptr(d["cell_offset"]), ptr(d["x"]),
                   ptr(d["y"]), ptr(d["z"]), ptr(d["w"]), q, s._grid(), s._planes_arr(["rho"]), ptr(w),
                   w.numel())
        s.postproc_depose_scalar("rho")
        for nm in ("Jx", "Jy", "Jz", "rho"):
            for m in range(M + 1):
                x, y = (sim["solver"].DataDev[f"{nm}_m{m}"] for sim in (a, b))
                assert torch.equal(x, y), (nm, m)
        for k in ("x", "y", "z", "sort_indx", "cell_offset", "indx_in_cell"):
            assert torch.equal(a["eons"].DataDev[k], b["eons"].DataDev[k]), k
