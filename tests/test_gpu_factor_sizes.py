"""The dataflow Cholesky at the sizes where its accumulation changes: one tile, two and three block columns (no
ordinary tiles), the early tiles' columns, and block columns on both sides of the 64 terms that one scan of the
published tiles covers, each with an order that is not a multiple of the tile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def spd(n, seed):
    """A symmetric matrix with eigenvalues in [1, 6]."""
    g = np.random.default_rng(seed).standard_normal((n, n))
    return g @ g.T / n + np.eye(n)


# block columns: 1, 2, 3, 7, 64, 65, 66 and 67
@pytest.mark.parametrize("n", [64, 65, 190, 385, 4096, 4097, 4161, 4225])
def test_cholesky_against_lapack(rsd, n):
    A = spd(n, n)
    L, info = rsd.cholesky(A)
    ref = np.linalg.cholesky(A)
    assert info == 0
    # forward error of a Cholesky factor: n eps cond(A), cond <= 6
    assert np.max(np.abs(L - ref)) <= 6.0 * n * np.finfo(float).eps * np.max(np.abs(ref))
