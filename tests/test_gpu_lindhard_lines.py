"""GPU: the Lindhard response on both sides of the lines between its two
kernels, and with one, two and three units per wave of each matrix-core
instantiation, at a dozen points q against plain numpy sums over all k.

Tolerance 1e-11 of max|X| (as the other tests of this response)."""
import numpy as np
import pytest

import edus

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,nf,grid", [
    (3, 1, (64, 64)), (3, 1, (72, 72)), (6, 1, (39, 26)), (6, 1, (48, 48)), (6, 5, (52, 52)), (7, 1, (45, 45)),
    (7, 3, (52, 52)), (7, 6, (48, 48)), (7, 6, (52, 52)), (8, 1, (20, 20)), (8, 2, (42, 42)), (8, 2, (45, 45)),
    (8, 3, (48, 48)), (8, 4, (48, 48)), (8, 5, (33, 33)), (8, 7, (32, 32)), (8, 7, (45, 26)), (8, 7, (40, 40)),
    (9, 4, (20, 20)), (11, 8, (28, 28)), (11, 10, (39, 39)),
    (12, 8, (36, 21)), (12, 8, (44, 44)), (12, 9, (18, 48)), (12, 11, (33, 33)), (13, 12, (20, 20)), (14, 13, (20, 20))])
def test_at_points(nb, nf, grid):
    print("case", nb, nf, grid, flush=True)
    rng = np.random.default_rng(100 * nb + nf)
    n0, n1 = grid
    nk = n0 * n1
    U = np.linalg.qr(rng.standard_normal((nk, nb, nb)) + 1j * rng.standard_normal((nk, nb, nb)))[0]
    eps = np.sort(rng.uniform(0, 1, (nk, nb)), axis=1)
    eps[:, nf:] += 0.5
    X = edus.lindhard(U, eps, n0, n1, nf)
    A = np.einsum("kav,kbv->kvab", U[:, :, :nf], U[:, :, :nf].conj()).reshape(nk, nf, nb * nb)
    B = np.einsum("kac,kbc->kcab", U[:, :, nf:].conj(), U[:, :, nf:]).reshape(nk, nb - nf, nb * nb)
    k = np.arange(nk)
    scale = np.abs(X).max()
    for q in [0, n1 - 1, nk - 1, *rng.integers(0, nk, 9)]:
        kq = (k // n1 + q // n1) % n0 * n1 + (k % n1 + q % n1) % n1
        r = 1.0 / (eps[kq][:, nf:, None] - eps[:, None, :nf])
        ref = -((r @ A) * B[kq]).sum((0, 1)).reshape(nb, nb) / nk
        assert np.abs(X[q] - ref).max() <= 1e-11 * scale
