"""The Grid methods take their arguments by the reference's names too (no
launch: the library call is recorded)."""
import pytest


@pytest.mark.parametrize("args,kw,want", [(("E",), {}, 3), ((), {"vec_fld": "B"}, 3),
                                          (("E", "B"), {}, 6)])
def test_preproc_project_vec_arguments(args, kw, want):
    from chimeracl_amd.methods.grid_methods_hip import GridMethodsHIP

    class G(GridMethodsHIP):
        def __init__(self):
            self.Args = {"vec_comps": ("x", "y", "z"), "Nx": 16, "Nr": 8, "M": 1}
            self.calls = []

        def _planes_arr(self, names):
            return list(names)

        def call(self, name, *a):
            self.calls.append((name, a))

    g = G()
    g.preproc_project_vec(*args, **kw)
    (name, a), = g.calls
    assert name == "chm_warp_axis" and len(a[0]) == a[1] == want
    with pytest.raises(TypeError):
        g.preproc_project_vec()
