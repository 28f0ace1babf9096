"""GPU: exchange on 120 x 120, the grid whose derivative has two forms and
whose plane does not fit in LDS: the choice between the forms is timed while
the context is created, before the exchange term's arrays exist.

Bar: one right-hand side within 1e-11 relative (as the other parity tests)."""
import numpy as np
import pytest

import edus
from conftest import hbn_params

oracle_py = pytest.importorskip("oracle_py")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("field", [[0.0, 0.0, 0.0], [4e-3, -3e-3, 0.0]])
def test_created_and_parity(field):
    o = oracle_py.Oracle(hbn_params(coulomb=True, grid=[120, 120, 1]))
    rng = np.random.default_rng(17)
    a = rng.standard_normal((o.Nk, 2, 2)) + 1j * rng.standard_normal((o.Nk, 2, 2))
    rho = o.rho + 0.01 * (a + a.conj().transpose(0, 2, 1))
    ref = o.rhs_E(field, rho)
    print("case", field, flush=True)
    eng = edus.Engine(2, o.N0, o.N1, o.get("H0k"), (o.get("rk0"), o.get("rk1"), o.get("rk2")), A=o.lattice(),
                      filledbands=1, U=o.get("U"), coulomb=True, W=o.get("Wscr"), hartree=o.get("hartree"),
                      rho0k=o.rho)
    t = eng.get_tuning()
    for form in (t.grad_fused, 1 - t.grad_fused):
        t.grad_fused = form
        eng.set_tuning(t)
        assert np.abs(eng.rhs(field, rho) - ref).max() <= 1e-11 * max(1.0, np.abs(ref).max())
        assert np.abs(eng.clone().rhs(field, rho) - ref).max() <= 1e-11 * max(1.0, np.abs(ref).max())
