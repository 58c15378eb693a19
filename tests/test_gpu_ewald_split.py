"""The split image sums of the grand mobility's assembly, at the pair counts where the split changes.

A pair's blocks depend on the pair and the lattice only, so the assembly of the first n particles of a suspension,
with the same lattice record, is a sub-matrix of the whole one's.  The whole is pinned to the oracle at its own size
by the parity tests; here every n takes another route through the sums.
"""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def assemble(L, n, pos, rad, lat):
    ld = 11 * n
    p = torch.tensor(pos[:n], device="cuda").contiguous()
    a = torch.tensor(rad[:n], device="cuda").contiguous()
    G = torch.full((ld, ld), float("nan"), dtype=torch.float64, device="cuda")
    nov = torch.zeros(1, dtype=torch.int32, device="cuda")
    rc = L.rsd_per_grpery_inv_fri_noalloc(n, C.c_void_p(p.data_ptr()), C.c_void_p(a.data_ptr()), C.byref(lat), 2,
                                          C.c_double(1.0 / np.pi), C.c_void_p(G.data_ptr()), ld,
                                          C.c_void_p(nov.data_ptr()), None)
    assert rc == 0
    torch.cuda.synchronize()
    return G.cpu().numpy().T, int(nov.item())


def rows(n, m):
    """Rows of the first m particles in an n-particle grand vector."""
    i3, i5 = np.arange(3 * m), np.arange(5 * m)
    return np.concatenate([i3, 3 * n + i3, 6 * n + i5])


# pairs: 1; 990 and 1035 (16 lanes a pair, then 4); 4095 and 4186 (4, then 1); 32640 and 32896 (1, then none);
# 65341 and 65703 (one round of waves, then one and a split remainder)
@pytest.mark.parametrize("n", [2, 45, 46, 91, 92, 256, 257, 362, 363])
@pytest.mark.parametrize("widths", [None, (0, 0), (1, 3)])
def test_assembly_of_a_subset_is_a_sub_matrix(rsd, n, widths):
    from rsd_amd.configs import random_suspension
    N = 400
    pos, rad, edge = random_suspension(N, 0.25, seed=11)
    # one pair in overlap, for the correction and its count
    pos[1] = pos[0] + (rad[0] + rad[1] - 1e-3) * np.array([0.6, 0.0, 0.8])
    lat = rsd.set_lattice_skew(0.3, [edge] * 3, 1.0)
    rsd.calc_lattice_inverse(lat, 1e-4, rad)
    if widths:
        lat.nr, lat.ni = widths
    L = rsd.load_library()
    whole, _ = assemble(L, N, pos, rad, lat)
    G, overlaps = assemble(L, n, pos, rad, lat)
    sub = whole[np.ix_(rows(N, n), rows(N, n))]
    assert overlaps >= 1 and np.all(np.isfinite(G))
    # both sum the same few hundred terms in other orders: terms * eps, times the
    # cancellation between terms of up to a few times the largest entry
    assert np.max(np.abs(G - sub)) <= 1e-13 * np.max(np.abs(sub))
