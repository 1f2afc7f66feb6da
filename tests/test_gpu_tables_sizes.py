"""The spectral tables at the sizes where the blocked inverse changes: one
panel, whole panels, remainders, several update tiles, and the wide form of
more than 1024 rows; against numpy's inverse and products in float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("Nr,M", [(4, 0), (17, 2), (33, 1), (34, 4), (64, 1), (65, 0), (130, 2),
                                  (301, 3), (1025, 0), (1026, 0), (1100, 0)])
def test_tables_sizes(Nr, M):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import chimeracl_amd as CA
    from chimeracl_amd import config as C
    from chimeracl_amd.methods.generic_methods_hip import Communicator
    from scipy.special import jn_zeros, jv
    s = CA.Solver(C.grid_config("C1", Nx=16, Nr=Nr, M=M, DampCells=2), Communicator(precision="f64"))
    D = s.DataDev
    r = s.Args["Rgrid"][1:, None]
    R = r[-1] + 0.5 * s.Args["dr"]
    for m in range(M + 1):
        k0, kp, km = (jn_zeros(abs(q), Nr - 1) / R for q in (m, m + 1, m - 1))
        inv = jv(m, r * k0)
        fwd = np.linalg.inv(inv)
        # |error| <= cond * eps * growth, in the 2-norm: cond(J) < 1e4 here
        cond = np.linalg.cond(inv)
        tol = 200 * cond * np.finfo(float).eps + 1e-13
        want = {"DHT_inv_m": inv, "DHT_m": fwd, "dDHT_plus_m": fwd @ (0.5 * kp * jv(m, r * kp)),
                "dDHT_minus_m": fwd @ (0.5 * km * jv(m, r * km))}
        for key, ref in want.items():
            got = D[key + str(m)].cpu().numpy()
            err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
            assert err < tol, (key, m, err, tol)
        one = D[f"DHT_m{m}"].cpu().numpy() @ D[f"DHT_inv_m{m}"].cpu().numpy()
        assert np.linalg.norm(one - np.eye(Nr - 1)) / np.sqrt(Nr - 1) < tol, m


def test_tables_above_4096_rows():
    """The widest panels: DHT DHT_inv = 1 (same bound, cond < 1e4)."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import chimeracl_amd as CA
    from chimeracl_amd import config as C
    from chimeracl_amd.methods.generic_methods_hip import Communicator
    Nr = 4099
    s = CA.Solver(C.grid_config("C1", Nx=16, Nr=Nr, M=0, DampCells=2), Communicator(precision="f64"))
    one = s.DataDev["DHT_m0"] @ s.DataDev["DHT_inv_m0"]
    one -= torch.eye(Nr - 1, dtype=torch.float64, device="cuda")
    assert float(one.norm()) / (Nr - 1) ** 0.5 < 200 * 1e4 * np.finfo(float).eps + 1e-13
