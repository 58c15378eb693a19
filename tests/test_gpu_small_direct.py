"""The direct routes at the small and odd sizes that the iterative route is compared with: INFO is LAPACK's for the same
mobility, which is positive definite."""
import numpy as np
import pytest
import scipy.linalg as sl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 5, 23, 24, 131])
def test_info_is_lapacks(rsd, oracle, n):
    from rsd_amd.configs import random_suspension
    conf, radii, edge = random_suspension(n, 0.25, seed=40 + n)
    lat = oracle.lattice(0.0, [edge] * 3, 1.0)
    oracle.calc_lattice_inverse(lat, 1e-4, radii)
    app, apq, aqq, overlaps = oracle.per_grpery_inv_fri(conf, radii, lat, 1e-4)
    want = sl.lapack.dpotrf(np.block([[app, apq], [apq.T, aqq]]))[1]
    assert want == 0 and overlaps == 0
    for route in (rsd.Suspension.RESIST_SCHUR, rsd.Suspension.RESIST_EXPLICIT):
        s = rsd.Suspension(conf, radii, rsd.default_config(edge, gravity=0.5))
        s.set_resistance_route(route)
        assert s.step(5e-4, 0.0)[1] == want
        s.close()
