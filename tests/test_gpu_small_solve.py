"""Systems shorter than two blocks of 16 columns through the 16-lane solve,
with bands up to and beyond the matrix, against the matrix itself.

Tolerance: LU with partial pivoting is backward stable, ||A x - b|| <=
c n (kl + ku + 1) u growth ||A|| ||x|| (infinity norms), with growth = max|U| /
max|A| of LAPACK's factors, which eliminate in the same order; c = 8 covers the
complex products and the reciprocal of the diagonal (one rounding more than a
division).
"""
import numpy as np
import pytest
import scipy.linalg.lapack as lap

from oracle import coral_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def solver_mod():
    from coral_amd import solver
    return solver


@pytest.mark.parametrize("n", [1, 2, 5, 15, 16, 17, 31, 32, 33])
@pytest.mark.parametrize("kl,ku", [(0, 0), (0, 1), (1, 0), (1, 2), (5, 4), (15, 16), (16, 27)])
def test_short_systems(solver_mod, n, kl, ku):
    rng = np.random.default_rng(100 * n + kl)
    ns = 6   # a full wavefront of four systems and a part of one
    A = np.zeros((ns, n, n), np.complex128)
    for i in range(n):
        j = slice(max(0, i - kl), min(n, i + ku + 1))
        w = j.stop - j.start
        A[:, i, j] = rng.normal(size=(ns, w)) + 1j * rng.normal(size=(ns, w))
    A[:, np.arange(n), np.arange(n)] += 2.0
    ab = np.stack([O.dense_to_lapack_band(a, kl, ku) for a in A])
    b = rng.normal(size=(ns, n)) + 1j * rng.normal(size=(ns, n))
    x, info = solver_mod.banded_solve(ab, kl, ku, b)
    assert not info.any()
    for s in range(ns):
        lu, _, _ = lap.zgbtrf(ab[s].T.copy(), kl, ku)
        growth = max(1.0, np.abs(lu[: kl + ku + 1]).max() / np.abs(A[s]).max())
        norm = np.abs(A[s]).sum(axis=1).max() * np.abs(x[s]).max()
        bound = 8 * n * (kl + ku + 1) * np.finfo(float).eps / 2 * growth * norm
        assert np.abs(A[s] @ x[s] - b[s]).max() <= bound
