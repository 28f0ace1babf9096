"""GPU: populations and current of a given state against plain numpy sums, at
the ends of the kernel's ranges: one band and sixteen, fewer k-points than a
tile, a ragged last tile, more tiles than work-groups, both layouts, mixed
precision (whose rotation to the Bloch gauge is FP32), and no eigenvectors.

Tolerances: the sums are of Nk terms of order one with FP64 rounding, 1e-12;
the FP32 rotation rounds its operands to 6e-8 of values of order one, nb times
over, 2e-6."""
import numpy as np
import pytest

import edus

pytestmark = pytest.mark.gpu


def _herm(rng, nk, nb):
    a = rng.standard_normal((nk, nb, nb)) + 1j * rng.standard_normal((nk, nb, nb))
    return 0.5 * (a + a.conj().transpose(0, 2, 1)) / max(1, nb)


@pytest.mark.parametrize("nb,grid,layout,precision,with_u", [
    (1, (2, 3), edus.LAYOUT_FULL, edus.PREC_FP64, True), (16, (3, 3), edus.LAYOUT_FULL, edus.PREC_FP64, True),
    (15, (5, 5), edus.LAYOUT_HERMITIAN, edus.PREC_FP64, True), (2, (66, 65), edus.LAYOUT_FULL, edus.PREC_FP64, True),
    (3, (70, 60), edus.LAYOUT_HERMITIAN, edus.PREC_FP64, True), (14, (9, 11), edus.LAYOUT_FULL, edus.PREC_MIXED, True),
    (5, (7, 6), edus.LAYOUT_FULL, edus.PREC_FP64, False)])
def test_observables(nb, grid, layout, precision, with_u):
    print("case", nb, grid, layout, precision, with_u, flush=True)
    rng = np.random.default_rng(nb)
    nk, nf = grid[0] * grid[1], max(1, nb // 2)
    U = np.linalg.qr(rng.standard_normal((nk, nb, nb)) + 1j * rng.standard_normal((nk, nb, nb)))[0]
    vel = [_herm(rng, nk, nb), None, _herm(rng, nk, nb)]
    eng = edus.Engine(nb, *grid, _herm(rng, nk, nb), U=U if with_u else None, vel=vel, filledbands=nf,
                      layout=layout, precision=precision)
    rho = _herm(rng, nk, nb)
    eng.set_state(rho)
    pb, pw, v = eng.observables()
    h = np.einsum("kan,kab,kbn->kn", U.conj(), rho, U, optimize=True).real.mean(0)
    want = np.where(np.arange(nb) < nf, 1.0 - h, h) if with_u else np.zeros(nb)
    assert np.abs(pb - want).max() <= (2e-6 if precision == edus.PREC_MIXED else 1e-12)
    assert np.abs(pw - np.einsum("kii->ki", rho).real.mean(0)).max() <= 1e-12
    for d in range(3):
        tr = np.einsum("kij,kji->k", vel[d], rho).mean() if vel[d] is not None else 0.0
        assert abs(complex(v[2 * d], v[2 * d + 1]) - tr) <= 1e-12
