"""INFO of the Cholesky factorisation: the first non-positive pivot, wherever it lies in the 16-column panels and 64-row
tiles, as LAPACK's DPOTRF gives it."""
import numpy as np
import pytest
import scipy.linalg as sl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [[0], [1], [15], [16], [31], [32], [48], [62], [63], [64], [79], [127], [128], [199],
                                 [50, 20], [150, 70], [63, 64]])
def test_first_bad_pivot(rsd, bad):
    n = 200
    rng = np.random.default_rng(5)
    B = rng.standard_normal((n, n))
    A = B @ B.T / n + np.eye(n)
    for k in bad:
        A[k, k] = -1.0
    want = sl.lapack.dpotrf(A, lower=0)[1]
    assert want == min(bad) + 1
    assert rsd.matrev(A)[1] == want
    assert rsd.cholesky(A)[1] == want
