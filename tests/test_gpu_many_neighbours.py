"""A large sphere among small ones: more than 64 lubrication neighbours in one block row, where the neighbour products
hold two neighbours' indices on a lane."""
import numpy as np
import pytest

from conftest import relerr
from test_gpu_gnn_sizes import reference

pytestmark = pytest.mark.gpu


def crowd(n, seed=3):
    """A sphere of radius 3 and n of radius 1 around it, all within 2 (3 + 1) of its centre (a pair is lubricated up to
    there), apart by 0.02 at least, in a box that keeps the images away."""
    rng = np.random.default_rng(seed)
    L = 30.0
    centre = np.full(3, L / 2)
    pos = [centre]
    while len(pos) <= n:
        v = rng.standard_normal(3)
        p = centre + v / np.linalg.norm(v) * rng.uniform(4.02, 7.9)
        if np.min(np.linalg.norm(np.array(pos[1:] or [centre + 100.0]) - p, axis=1)) > 2.02:
            pos.append(p)
    radii = np.ones(n + 1)
    radii[0] = 3.0
    return np.array(pos), radii, L


# one neighbour fewer and more than a wave's lanes, and all that a row holds
@pytest.mark.parametrize("n", [63, 64, 65, 80, 96])
@pytest.mark.parametrize("precond", [1, 2, 3, 4])
def test_iterative_step_against_the_direct_route(rsd, n, precond):
    conf, radii, L = crowd(n)
    out = []
    for route in (rsd.Suspension.RESIST_SCHUR, rsd.Suspension.RESIST_ITERATIVE):
        s = rsd.Suspension(conf, radii, rsd.default_config(L, gravity=0.5))
        s.set_resistance_route(route)
        s.set_iterative(precond, max_iter=4000)
        s.set_gnn(rsd.Gnn.load(rsd.GNN_PARAMS_PATH))
        yeta, info = s.step(5e-4, 0.0)
        assert info == 0
        if route == rsd.Suspension.RESIST_ITERATIVE:
            assert not s.iterative_stats()[2]  # no redo by the direct route
        u, sh, _ = s.last()
        out.append((u, sh, yeta))
        s.close()
    # both routes are held to 1e-10 of the reference
    for a, b in zip(out[0], out[1]):
        assert np.max(np.abs(a - b)) <= 1e-10 * np.max(np.abs(a))


@pytest.mark.parametrize("n", [65, 96])
def test_loss_and_gradient(rsd, n):
    conf, radii, L = crowd(n)
    sus = rsd.Suspension(conf, radii, rsd.default_config(L))
    sus.prepare_iterative(0.0)
    M, R, nnb, col, dist, cap = sus.iterative_system()
    assert nnb[0] == n and len(set(col[0, :n])) == n
    gnn = rsd.Gnn(seed=3)
    p = gnn.params()
    p[-133:] = (0.05 * np.random.default_rng(4).standard_normal(133)).astype(np.float32)
    gnn.set_params(p)
    loss, grad, Z = sus.gnn_loss(gnn, nz=3, seed=11)
    want, gwant = reference(p, M, R, nnb, col, dist, radii, Z)
    # 7 stages of sums of up to 132 terms in FP32: 7 * 132 * 2^-24 = 5.5e-5 forward; forward and backward twice that,
    # and units whose pre-activation is that close to zero may switch: 1e-3 of a group's norm
    assert abs(loss - want) <= 5.5e-5 * want
    off = [0, 192, 192 + 16768, 192 + 2 * 16768, 192 + 3 * 16768, len(p)]
    for a, b in zip(off[:-1], off[1:]):
        assert relerr(gwant[a:b], grad[a:b]) < 1e-3, (a, b)
    gnn.close()
    sus.close()
