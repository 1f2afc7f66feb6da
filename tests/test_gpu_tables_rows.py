"""Tables of more than 16384 rows, whose first panels do not fit a workgroup's
registers: DHT DHT_inv = 1.  |error| <= growth cond eps in the 2-norm; the
condition number grows as 3.3 sqrt(n) (128 .. 2048 rows: 34 .. 150), so below
1e3 here, and the growth of the elimination is taken as 200, as for the smaller
sizes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_tables_above_16384_rows():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import chimeracl_amd as CA
    from chimeracl_amd import config as C
    from chimeracl_amd.methods.generic_methods_hip import Communicator
    Nk = 16384 + 3 * 8 + 5
    s = CA.Solver(C.grid_config("C1", Nx=16, Nr=Nk + 1, M=0, DampCells=2),
                  Communicator(precision="f64"))
    one = s.DataDev["DHT_m0"] @ s.DataDev["DHT_inv_m0"]
    one -= torch.eye(Nk, dtype=torch.float64, device="cuda")
    assert float(one.norm()) / Nk ** 0.5 < 200 * 1e3 * np.finfo(float).eps + 1e-13
