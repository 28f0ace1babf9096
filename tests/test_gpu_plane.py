"""GPU: the spectral passes of plane_fft.hip against the oracle: both axes'
derivatives in one launch (most grids), and one work-group per plane in LDS
(exchange, the Peierls phase, and derivatives of large fields on grids whose
line splits have large factors).  The lengths cover one-step lines (at most
16), both orders of a short and a long axis, every radix of the kernels, and
for exchange and phase planes up to the limit of LDS.

Bar: one right-hand side within 1e-11 relative (as the other parity tests)."""
import os

import numpy as np
import pytest

import edus
from edus import models

oracle_py = pytest.importorskip("oracle_py")

pytestmark = pytest.mark.gpu

FULL, HERM = edus.LAYOUT_FULL, edus.LAYOUT_HERMITIAN


def _model(name, model_dir, grid, peierls=False):
    p = models.workload(name, os.path.join(model_dir, f"plane_{name}_{grid[0]}x{grid[1]}"), grid=[*grid, 1])
    p["peierls"] = peierls
    return p


def _engine(o, p, layout=FULL):
    args = dict(H0k=o.get("H0k"), xik=(o.get("rk0"), o.get("rk1"), o.get("rk2")), A=o.lattice(),
                filledbands=p["filledbands"], U=o.get("U"), layout=layout, peierls=p["peierls"])
    if p["coulomb"]:
        args.update(coulomb=True, W=o.get("Wscr"), hartree=o.get("hartree"), rho0k=o.rho)
    return edus.Engine(o.nb, o.N0, o.N1, **args)


def _rho(o, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((o.Nk, o.nb, o.nb)) + 1j * rng.standard_normal((o.Nk, o.nb, o.nb))
    return 0.5 * (a + a.conj().transpose(0, 2, 1))


def _fields(o):
    """Along both lattice vectors, and perpendicular to either."""
    A, z = o.lattice(), np.array([0.0, 0.0, 1.0])
    e0, e1 = np.cross(A[:, 1], z), np.cross(A[:, 0], z)
    return [[4e-3, -3e-3, 0.0], list(3e-3 * e0 / np.linalg.norm(e0)), list(3e-3 * e1 / np.linalg.norm(e1))]


GRIDS = [(22, 16), (13, 45), (45, 2), (2, 39), (169, 26), (42, 182), (165, 12), (45, 208), (98, 99), (99, 100)]


@pytest.mark.parametrize("grid", GRIDS)
def test_derivative(model_dir, grid):
    p = _model("ipa2_square30", model_dir, grid)
    print("case", grid, flush=True)
    o = oracle_py.Oracle(p)
    eng = _engine(o, p)
    rho = _rho(o, 4)
    for E in _fields(o):
        ref = o.rhs_E(E, rho)
        assert np.abs(eng.rhs(E, rho) - ref).max() <= 1e-11 * max(1.0, np.abs(ref).max())


def test_derivative_in_lds(model_dir):
    """14 bands on 66 x 45: above the field size up to which factors of 11 take
    the one-launch form of both axes."""
    p = _model("ipa14_hex120", model_dir, (66, 45))
    o = oracle_py.Oracle(p)
    eng = _engine(o, p)
    rho = _rho(o, 9)
    for E in _fields(o):
        ref = o.rhs_E(E, rho)
        assert np.abs(eng.rhs(E, rho) - ref).max() <= 1e-11 * max(1.0, np.abs(ref).max())


# 196 planes: one launch of work-groups of one wave (radices of at most 8), two,
# three and four, with whole and ragged groups of columns and rows
@pytest.mark.parametrize("grid", [(56, 35), (49, 30), (20, 120), (18, 100), (36, 60), (63, 45)])
def test_derivative_work_groups(model_dir, grid):
    p = _model("ipa14_hex120", model_dir, grid)
    print("case", grid, flush=True)
    o = oracle_py.Oracle(p)
    eng = _engine(o, p)
    rho = _rho(o, 10)
    for E in _fields(o):
        ref = o.rhs_E(E, rho)
        assert np.abs(eng.rhs(E, rho) - ref).max() <= 1e-11 * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("grid,layout", [((16, 16), FULL), ((3, 21), HERM), ((13, 33), HERM), ((30, 14), FULL),
                                         ((45, 22), FULL)])
def test_exchange(model_dir, grid, layout):
    p = _model("hsex8_hex90", model_dir, grid)
    print("case", grid, layout, flush=True)
    o = oracle_py.Oracle(p)
    eng = _engine(o, p, layout)
    rho = o.rho + 0.05 * _rho(o, 5)
    iu = np.triu_indices(o.nb)
    for E in _fields(o) + [[0.0, 0.0, 0.0]]:
        ref, got = o.rhs_E(E, rho), eng.rhs(E, rho)
        d = np.abs(got - ref) if layout == FULL else np.abs(got - ref)[:, iu[0], iu[1]]
        assert d.max() <= 1e-11 * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("grid", [(45, 63), (7, 26), (91, 10)])
def test_phase(model_dir, grid):
    p = _model("ipa2_square30", model_dir, grid, peierls=True)
    print("case", grid, flush=True)
    o = oracle_py.Oracle(p)
    eng = _engine(o, p)
    rho = _rho(o, 6)
    E, A = [4e-3, -3e-3, 0.0], [0.21, -0.37, 0.0]
    ref = o.rhs_EA(E, A, rho)
    assert np.abs(eng.rhs_peierls(E, A, rho) - ref).max() <= 1e-11 * max(1.0, np.abs(ref).max())


def test_batch_with_one_axis_members(model_dir):
    """Members whose fields lie along one lattice vector end in a batch, whose
    kernels see both axes, bit for bit where they end alone."""
    p = _model("ipa2_square30", model_dir, (45, 21))
    o = oracle_py.Oracle(p)
    engines = [_engine(o, p) for _ in range(3)]
    E = np.zeros((4, 3, 3, 3))
    rng = np.random.default_rng(7)
    for i, e in enumerate(_fields(o)):
        E[:, :, i, :] = rng.uniform(0.5, 1.0, (4, 3, 1)) * np.array(e)
    for e in engines:
        e.set_state(o.rho + 0.05 * _rho(o, 8))
    batch = edus.Batch(engines)
    batch.rk4_steps(0.05, E)
    for i, e in enumerate(engines):
        e.rk4_steps(0.05, E[:, :, i])
        alone = e.get_state()
        batch.store(i)
        assert np.array_equal(e.get_state(), alone)


def test_batch_of_two_pass_members(model_dir):
    """As above where the axes are separate passes (240 x 180, above the field size
    up to which such splits take one launch): groups of rows that hold the last
    rows of one member and the first of the next."""
    p = _model("ipa6_hex96", model_dir, (240, 180))
    o = oracle_py.Oracle(p)
    engines = [_engine(o, p) for _ in range(3)]
    E = np.zeros((4, 3, 3, 3))
    rng = np.random.default_rng(7)
    for i, e in enumerate(_fields(o)):
        E[:, :, i, :] = rng.uniform(0.5, 1.0, (4, 3, 1)) * np.array(e)
    for e in engines:
        e.set_state(o.rho + 0.05 * _rho(o, 8))
    batch = edus.Batch(engines)
    batch.rk4_steps(0.05, E)
    for i, e in enumerate(engines):
        e.rk4_steps(0.05, E[:, :, i])
        alone = e.get_state()
        batch.store(i)
        assert np.array_equal(e.get_state(), alone)
