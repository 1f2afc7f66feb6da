"""chm_depose_vector_* with the push of a species without particles: what
surrounds the deposit (zeroing, post-processing) is still done, bit for bit as
by chm_zero_planes_* and chm_postproc_deposit_*, and nothing else."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("M", [0, 2])
@pytest.mark.parametrize("first", [0, 1])
@pytest.mark.parametrize("last", [False, True])
def test_depose_empty_species(precision, M, first, last):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from chimeracl_amd.methods.generic_methods_hip import ptr
    from tests import simpair as S
    sim, _ = S.make_pair(S.tiny_grid(Nx=64, Nr=17, M=M, damp=2), None, precision=precision,
                         with_oracle=False)
    s, d = sim["solver"], sim["eons"].DataDev
    sim["eons"].sort_parts(s)
    D = s.DataDev
    names = [f"J{c}_m{m}" for c in "xyz" for m in range(M + 1)]
    gen = torch.Generator(device="cuda").manual_seed(M)
    start = {k: torch.randn(D[k].shape, generator=gen, dtype=D[k].dtype, device="cuda") for k in names}
    J, w = s._planes_arr(["Jx", "Jy", "Jz"]), s._dep_ws()

    def put():
        for k in names:
            D[k].copy_(start[k])

    put()
    if first:
        s.zero_planes(["Jx", "Jy", "Jz"])
    if last:
        s.postproc_depose_vector("J")
    want = {k: D[k].clone() for k in names}
    put()
    before = {k: d[k].clone() for k in ("x", "y", "z", "indx_in_cell")}
    xyz = [ptr(d[k]) for k in "xyz"]
    s.call("chm_depose_vector", ptr(d["sort_indx"]), ptr(d["cell_offset"]), *xyz, *xyz,
           *(ptr(d[k]) for k in ("px", "py", "pz", "g_inv", "w")), -1, 0.01, 0,
           ptr(d["indx_in_cell"]), s._grid(), J, first, ptr(D["dV_inv"]) if last else None, ptr(w),
           w.numel())
    for k in names:
        assert torch.equal(D[k], want[k]), k
    for k, v in before.items():
        assert torch.equal(d[k], v), k
