"""GPU: both axes' derivatives in one launch on plane sets above 8 MB whose line
splits have factors above 12, where an axis has no two-step kernel: one
right-hand side against the oracle, within 1e-11 relative (as the other parity
tests), and members of a batch bit for bit where they end alone."""
import os

import numpy as np
import pytest

import edus
from edus import models

oracle_py = pytest.importorskip("oracle_py")

pytestmark = pytest.mark.gpu


def _engine(o, p, layout):
    return edus.Engine(o.nb, o.N0, o.N1, o.get("H0k"), (o.get("rk0"), o.get("rk1"), o.get("rk2")), A=o.lattice(),
                       filledbands=p["filledbands"], U=o.get("U"), layout=layout)


def _rho(o, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((o.Nk, o.nb, o.nb)) + 1j * rng.standard_normal((o.Nk, o.nb, o.nb))
    return 0.5 * (a + a.conj().transpose(0, 2, 1))


@pytest.mark.parametrize("name,grid,layout", [("ipa6_hex96", (130, 154), edus.LAYOUT_FULL),
                                              ("ipa6_hex96", (150, 128), edus.LAYOUT_FULL),
                                              ("ipa14_hex120", (112, 112), edus.LAYOUT_HERMITIAN)])
def test_right_hand_side_and_batch(model_dir, name, grid, layout):
    print("case", name, grid, layout, flush=True)
    p = models.workload(name, os.path.join(model_dir, f"axes_{name}_{grid[0]}x{grid[1]}"), grid=[*grid, 1])
    o = oracle_py.Oracle(p)
    engines = [_engine(o, p, layout) for _ in range(2)]
    engines[0].timing_enable(True)
    rho = _rho(o, 11)
    E = [4e-3, -3e-3, 0.0]
    ref, got = o.rhs_E(E, rho), engines[0].rhs(E, rho)
    iu = np.triu_indices(o.nb)
    d = np.abs(got - ref) if layout == edus.LAYOUT_FULL else np.abs(got - ref)[:, iu[0], iu[1]]
    assert d.max() <= 1e-11 * max(1.0, np.abs(ref).max())
    assert engines[0].timing_get("grad_axes")[1] == 1
    engines[0].timing_enable(False)
    rng = np.random.default_rng(5)
    fields = rng.uniform(-4e-3, 4e-3, (3, 3, 2, 3)) * np.array([1.0, 1.0, 0.0])
    for i, e in enumerate(engines):
        e.set_state(o.rho + 0.05 * _rho(o, 20 + i))
    batch = edus.Batch(engines)
    batch.rk4_steps(0.05, fields)
    for i, e in enumerate(engines):
        e.rk4_steps(0.05, np.ascontiguousarray(fields[:, :, i]))
        alone = e.get_state()
        batch.store(i)
        assert np.array_equal(e.get_state(), alone)
