"""GPU: the two kernels of the Lindhard response against plain numpy sums, at
the ends of the matrix-core form's ranges: window longer than a grid row, one
row, few rows (no split of the k range), ragged last window, every number of
band quadruples, the most bands, and shapes left to the vector form.

Tolerance 1e-11 of max|X| (as the other tests of this response)."""
import numpy as np
import pytest

import edus

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,nf,grid", [
    (3, 1, (1, 7)), (3, 2, (5, 2)), (4, 1, (2, 33)), (5, 4, (13, 3)), (5, 1, (9, 10)), (6, 3, (12, 18)),
    (7, 2, (1, 21)), (8, 4, (16, 17)), (8, 7, (4, 18)), (8, 1, (6, 9)), (11, 3, (5, 6)), (12, 6, (7, 5)),
    (13, 9, (3, 8)), (16, 8, (5, 4)), (16, 1, (3, 5)), (16, 15, (2, 9)), (2, 1, (6, 6)), (10, 5, (4, 6))])
def test_response(nb, nf, grid):
    print("case", nb, nf, grid, flush=True)
    rng = np.random.default_rng(100 * nb + nf)
    n0, n1 = grid
    nk = n0 * n1
    U = np.linalg.qr(rng.standard_normal((nk, nb, nb)) + 1j * rng.standard_normal((nk, nb, nb)))[0]
    eps = np.sort(rng.uniform(0, 1, (nk, nb)), axis=1)
    eps[:, nf:] += 0.5
    X = edus.lindhard(U, eps, n0, n1, nf)
    A = np.einsum("kav,kbv->kvab", U[:, :, :nf], U[:, :, :nf].conj())
    B = np.einsum("kac,kbc->kcab", U[:, :, nf:].conj(), U[:, :, nf:])
    k = np.arange(nk)
    ref = np.empty_like(X)
    for q in range(nk):
        kq = (k // n1 + q // n1) % n0 * n1 + (k % n1 + q % n1) % n1
        r = 1.0 / (eps[:, :nf, None] - eps[kq][:, None, nf:])
        ref[q] = np.einsum("kvc,kvab,kcab->ab", r, A, B[kq], optimize=True) / nk
    assert np.abs(X - ref).max() <= 1e-11 * np.abs(ref).max()
    assert np.array_equal(edus.lindhard(U, eps, n0, n1, nf), X)  # no order of summation depends on timing
