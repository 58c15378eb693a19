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


# 135 block columns (single tiles only), 136 (the fewest with macro tasks), and an odd number, whose last block row
# goes by single tiles
@pytest.mark.parametrize("n", [8640, 8704, 8743])
def test_cholesky_of_large_matrices(rsd, n):
    A = spd(n, n)
    L, info = rsd.cholesky(A)
    assert info == 0
    # backward error of a Cholesky factor: n eps ||A||, checked on a product with vectors
    x = np.random.default_rng(1).standard_normal((n, 4))
    r = L @ (L.T @ x) - A @ x
    assert np.linalg.norm(r) <= 6.0 * n * np.finfo(float).eps * np.linalg.norm(x)
    assert np.all(np.triu(L, 1) == 0.0)


# 138 and 141 block columns of the 11N system: macro tasks and inv(L_S) in one launch
@pytest.mark.parametrize("n", [800, 817])
def test_schur_step_with_macro_tasks(rsd, n):
    from rsd_amd.configs import random_suspension
    conf, radii, edge = random_suspension(n, 0.2, seed=n)
    out = []
    for route in (rsd.Suspension.RESIST_SCHUR, rsd.Suspension.RESIST_EXPLICIT):
        s = rsd.Suspension(conf, radii, rsd.default_config(edge))
        s.set_resistance_route(route)
        _, info = s.step(5e-4, 0.0)
        assert info == 0
        out.append(s.last()[:2])
        s.close()
    # both routes are held to 1e-10 of the reference
    for a, b in zip(*out):
        assert np.max(np.abs(a - b)) <= 1e-10 * np.max(np.abs(a))
