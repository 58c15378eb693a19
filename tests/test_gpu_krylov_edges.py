"""The iterative route at the sizes and iteration counts where its kernels' shapes change: fewer particles than a
workgroup holds, orders that are no multiple of the 16-byte vectors, of 256 rows or of the columns a workgroup takes,
and one to the largest number of inner iterations."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 11N: 22, 33, 55 (odd: scalar tails), 253 and 264 (about one 256-row group), 1441 (odd, several groups)
@pytest.mark.parametrize("n", [2, 3, 5, 23, 24, 131])
@pytest.mark.parametrize("precond,inner", [(1, 20), (2, 1), (2, 31), (3, 20), (4, 7)])
def test_iterative_step_against_the_direct_route(rsd, n, precond, inner):
    from rsd_amd.configs import random_suspension
    conf, radii, edge = random_suspension(n, 0.25, seed=40 + n)
    out = []
    for route in (rsd.Suspension.RESIST_SCHUR, rsd.Suspension.RESIST_ITERATIVE):
        s = rsd.Suspension(conf, radii, rsd.default_config(edge, gravity=0.5))
        s.set_resistance_route(route)
        s.set_iterative(precond, inner_iters=inner, max_iter=4000)
        s.set_gnn(rsd.Gnn.load(rsd.GNN_PARAMS_PATH))
        yeta, info = s.step(5e-4, 0.0)
        if info and route == rsd.Suspension.RESIST_SCHUR:
            pytest.skip(f"the mobility of these {n} spheres in their small box is indefinite (LAPACK's INFO {info})")
        assert info == 0
        if route == rsd.Suspension.RESIST_ITERATIVE:
            assert not s.iterative_stats()[2]  # no redo by the direct route
        u, sh, _ = s.last()
        out.append((u, sh, yeta))
        s.close()
    # both routes are held to 1e-10 of the reference
    for a, b in zip(out[0], out[1]):
        assert np.max(np.abs(a - b)) <= 1e-10 * np.max(np.abs(a))
