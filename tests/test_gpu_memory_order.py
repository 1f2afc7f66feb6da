"""The memory-order gather inside steps and runs of a species large enough for
it (2^21 particles): realigned, pre-pushed and replayed steps leave the same
state, bit for bit, as with the sorted order alone, so the keys it takes are
never those of another moment."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

NAMES = ("x", "y", "z", "px", "py", "pz", "g_inv", "pid")


@pytest.mark.parametrize("precision,M", [("mixed", 1), ("mixed", 2), ("f64", 0)])
@pytest.mark.parametrize("graph,align", [(False, 0), (False, 2), (True, 2), (True, 0)])
def test_steps_with_memory_order(precision, M, graph, align):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import chimeracl_amd as CA
    from tests import simpair as S
    g = S.tiny_grid(Nx=256, Nr=64, M=M, damp=4)
    out, taken = [], []
    for mem in (True, False):
        sim, _ = S.make_pair(g, S.tiny_laser(g), ppc=(2, 2, 36), precision=precision, with_oracle=False)
        s, e = sim["solver"], sim["eons"]
        assert e.Args["Np"] >= 1 << 21
        if not mem:
            e.memory_keys_ptr = lambda grid: None
        loop = CA.PIC_loop(solvers=[s], species=[e, sim["ions"]], graph=graph, align_every=align)
        taken.append(0)

        def seen():
            taken[-1] += int(e._gather_flag.item())

        loop.step()
        seen()
        loop.run(4)
        seen()
        loop.step()
        seen()
        e.sort_parts(s)  # calls of a user's own program, between the steps
        e.reorder_parts()
        s.gather_and_push([e], prepush=True)
        e.use_prepushed(s)
        e.sort_parts(s)
        s.depose_currents([e], push_half=True, half_in=True)
        e.sort_parts(s)
        s.gather_and_push([e])
        seen()
        s.gather_and_push([e])  # the keys of the same sort again
        seen()
        loop.run(2)
        seen()
        out.append({k: e.DataDev[k].clone() for k in NAMES if k in e.DataDev})
        out[-1].update({f"{f}{c}_m{m}": s.DataDev[f"{f}{c}_m{m}"].clone() for f in "EBJ" for c in "xyz"
                        for m in range(M + 1)})
        del loop, sim, s, e
    assert taken[0] >= 4 and taken[1] == 0, taken
    assert out[0].keys() == out[1].keys()
    for k in out[0]:
        assert torch.equal(out[0][k], out[1][k]), k
