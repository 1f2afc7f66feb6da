"""Copies of many arrays in one launch: DiffPIC._copy_many leaves what differs
in shape, type or strides to Tensor.copy_ (the kernel copies bytes by the
destination's size) and splits longer lists; chm_copy_many refuses more arrays
than a launch takes.  Nothing is launched."""
import ctypes

import pytest
import torch


@pytest.fixture
def sim(monkeypatch):
    from chimeracl_amd import _lib, adjoint

    class Comm:
        def stream(self):
            return 0

    s = adjoint.DiffPIC.__new__(adjoint.DiffPIC)
    s.comm, s.launched = Comm(), []
    monkeypatch.setattr(_lib, "call", lambda name, n, *a: s.launched.append((name, n)))
    return s


@pytest.mark.parametrize("dst,src", [
    (torch.zeros(8), torch.zeros(7)), (torch.zeros(8), torch.zeros(9)),
    (torch.zeros(2, 4), torch.zeros(4, 2))])
def test_shapes_that_do_not_match_are_refused(sim, dst, src):
    with pytest.raises(RuntimeError):
        sim._copy_many([torch.zeros(3), dst], [torch.zeros(3), src])
    with pytest.raises(ValueError):
        sim._copy_many([torch.zeros(3), dst], [torch.zeros(3)])
    assert sim.launched == []


@pytest.mark.parametrize("dst,src", [
    (torch.zeros(8), torch.rand(8, dtype=torch.float64)), (torch.zeros(4, 4).t(), torch.rand(4, 4)),
    (torch.zeros(8), torch.rand(16)[::2]), (torch.zeros(16)[::2], torch.rand(8)),
    (torch.zeros(8), torch.rand(1))])
def test_other_types_and_strides_go_through_copy(sim, dst, src):
    sim._copy_many([torch.zeros(3), dst], [torch.zeros(3), src])
    assert torch.equal(dst, src.to(dst.dtype).expand_as(dst))
    assert sim.launched == [("chm_copy_many", 1)]
    sim._copy_many([dst])
    if not dst.is_contiguous():
        assert not dst.any()


def test_clones_of_strided_tensors(sim):
    src = [torch.rand(3), torch.rand(4, 5).t(), torch.rand(16)[::2], torch.rand(1).expand(6)]
    out = sim._clones(src)
    assert sim.launched == [("chm_copy_many", 1)]
    for o, s in zip(out[1:], src[1:]):
        assert torch.equal(o, s) and o.dtype == s.dtype


@pytest.mark.parametrize("n", [0, 1, 64, 65, 130])
def test_lists_are_split(sim, n):
    from chimeracl_amd import _lib
    m = _lib.CHM_COPY_MAXARR
    want = [("chm_copy_many", min(m, n - i)) for i in range(0, n, m)]
    sim._copy_many([torch.zeros(4) for _ in range(n)], [torch.ones(4) for _ in range(n)])
    assert sim.launched == want
    sim._copy_many([torch.zeros(4) for _ in range(n)])
    assert sim.launched == want * 2


@pytest.mark.parametrize("n,want", [(64, 0), (65, -1), (-1, -1)])
def test_arrays_of_a_launch(n, want):
    """(no bytes: an accepted call launches nothing)"""
    from chimeracl_amd import _lib
    src, dst, nb = (ctypes.c_void_p * 65)(), (ctypes.c_void_p * 65)(), (ctypes.c_int64 * 65)()
    a = ctypes.addressof
    assert _lib.lib.chm_copy_many(n, a(src), a(dst), a(nb), None) == want
