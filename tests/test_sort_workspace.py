"""chm_sort_workspace_bytes never falls when the number of particles grows,
also where the sort's plan changes: a workspace for the largest species is
enough for every smaller one.  Host-only query."""
import pytest


@pytest.mark.parametrize("Nx,Nr", [(4096, 512), (2048, 256), (1024, 256), (512, 128), (512, 257),
                                   (60, 40), (64, 64), (65, 65), (33, 33), (4096, 1025), (8192, 1024)])
def test_sort_workspace_grows_with_particles(Nx, Nr):
    from chimeracl_amd import _lib
    nbins = (Nx - 1) * (Nr - 1) + 1
    marks = [1 << 23, 1 << 26]
    for cells in (256, 2048):  # cells of a bucket
        nbk = -(-nbins // cells)
        marks += [2048 * nbk, 16384 * nbk]
    ns = sorted({max(0, m + d) for m in marks for d in (-70001, -4097, -2, -1, 0, 1, 4097, 70001)}
                | {0, 1, 100, 4096, 100003})
    need = [_lib.lib.chm_sort_workspace_bytes(n, nbins) for n in ns]
    for a, b, n in zip(need, need[1:], ns[1:]):
        assert b >= a, (n, a, b)
