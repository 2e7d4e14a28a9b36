"""Ridge solves at the edges of the factorization's blocks (64-column steps,
128-wide update tiles, 256-wide panels and inverse blocks) and of the batch of
ridge parameters, against LAPACK posv: backward error <= 1e-14 and a forward
difference within 100 cond eps, as for the sizes of the other ridge tests."""

import numpy as np
import pytest

from oracle.numerics import solver_ridge_posv
from pypolymlp_amd import mlp_dev

pytestmark = pytest.mark.gpu


def system(F, seed):
    rng = np.random.default_rng(seed)
    X = rng.normal(size=(2 * F + 5, F)) * np.logspace(0, -2, F)[None, :]
    X[:, 1:] += 0.3 * X[:, :-1]
    return X.T @ X, X.T @ rng.normal(size=X.shape[0])


@pytest.mark.parametrize("F,n_alpha", [(1, 1), (2, 3), (63, 1), (64, 2), (65, 1), (127, 2), (129, 1),
                                       (191, 1), (256, 2), (257, 1), (320, 1), (321, 8), (449, 9),
                                       (513, 2), (641, 1), (769, 10)])
def test_ridge_block_edges(F, n_alpha):
    A, b = system(F, F)
    alphas = np.logspace(-5, -1, n_alpha) * np.trace(A) / F
    C = mlp_dev.solver_ridge(A, b, alphas)
    Cr = solver_ridge_posv(A, b, alphas)
    eps = np.finfo(np.float64).eps
    for k, a in enumerate(alphas):
        Aa = A + a * np.eye(F)
        c = C[:, k]
        assert np.linalg.norm(Aa @ c - b) <= 1e-14 * np.linalg.norm(Aa, 2) * np.linalg.norm(c)
        fwd = np.linalg.norm(c - Cr[:, k]) / np.linalg.norm(Cr[:, k])
        assert fwd <= max(100 * np.linalg.cond(Aa) * eps, 1e-13)


@pytest.mark.parametrize("F,bad", [(40, 0), (200, 130), (300, 299), (700, 400)])
def test_not_positive_definite_in_a_batch(F, bad):
    """Only the ridge parameters that leave the matrix indefinite fail."""
    A, b = system(F, 7)
    A[bad] = A[:, bad] = 0.0
    A[bad, bad] = -1.0
    alphas = np.array([0.5, 2.0, 1e-3, 3.0])
    C = mlp_dev.solver_ridge(A, b, alphas)
    assert np.all(C[:, [0, 2]] == 1e30)
    Cr = solver_ridge_posv(A, b, alphas[[1, 3]])
    assert np.linalg.norm(C[:, [1, 3]] - Cr) <= 1e-10 * np.linalg.norm(Cr)
