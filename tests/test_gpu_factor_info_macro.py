"""INFO and the inverse of large matrices, whose factorisation goes by macro tasks: a non-positive pivot in the first
tile, in the columns that start early, in a macro task's rows and in the last block row of an odd number of them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 8743  # 137 block columns


@pytest.fixture(scope="module")
def spd():
    """A symmetric matrix with eigenvalues in about [1, 5]: 3 plus a random one of spectral radius about 2."""
    g = np.random.default_rng(9).standard_normal((N, N))
    return (g + g.T) / np.sqrt(2.0 * N) + 3.0 * np.eye(N)


# the leading minors before a negative diagonal entry are positive definite, and the one with it is not
@pytest.mark.parametrize("bad", [[0], [63], [447], [448], [4500], [8639, 4500], [8703], [8704], [8742]])
def test_first_bad_pivot(rsd, spd, bad):
    A = spd.copy()
    A[bad, bad] = -1.0
    assert rsd.cholesky(A)[1] == min(bad) + 1


def test_inverse(rsd, spd):
    X, info = rsd.matrev(spd)
    assert info == 0
    v = np.random.default_rng(2).standard_normal((N, 4))
    # an inverse by Cholesky: |A (X v) - v| <= a few n eps cond(A) |v|, cond <= 6
    assert np.linalg.norm(spd @ (X @ v) - v) <= 4 * 6.0 * N * np.finfo(float).eps * np.linalg.norm(v)
    bad = spd.copy()
    bad[5000, 5000] = -1.0
    assert rsd.matrev(bad)[1] == 5001
