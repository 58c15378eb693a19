"""The learned preconditioner's kernels at the sizes where their splits end: particles without neighbours, neighbour
lists that leave waves and passes part full, more neighbour columns than one pass of the block products, chunks of
particles with a remainder, and more particles than the smallest chunks cover."""
import numpy as np
import pytest
import torch

from conftest import relerr

pytestmark = pytest.mark.gpu


def reference(p, M, R, nnb, col, dist, radii, Z):
    """Loss and gradient in 64 bits (the network of gnn_reference, the preconditioner applied pair by pair)."""
    import gnn_reference as ref
    N = len(radii)
    n6 = 6 * N
    K = (torch.tensor(R).cuda() @ torch.tensor(M).cuda()).cpu()
    K[:n6] += torch.eye(n6, 11 * N, dtype=torch.float64)
    K[n6:] = torch.tensor(M[n6:])
    g, _, d = ref.edges(nnb, col)
    dof = torch.tensor(np.array([ref.dofs(N, i) for i in range(N)]))
    D = torch.linalg.inv(K[dof[:, :, None], dof[:, None, :]])
    pair = torch.cat([dof[g], dof[d]], 1)
    X = torch.linalg.inv(K[pair[:, :, None], pair[:, None, :]])
    A, B = X[:, :11, :11] - D[g], X[:, :11, 11:]
    pt = torch.tensor(p.astype(np.float64), requires_grad=True)
    feat, xn = ref.features(nnb, col, dist, radii)
    w = ref.network(ref.unpack_t(pt), xn, feat, g, d, N, nnb)
    rr, zz = 0.0, 0.0
    for z in torch.tensor(np.asarray(Z)).reshape(-1, 11 * N):
        zl = z[dof]
        per = torch.einsum("nij,nj->ni", D, zl)
        pairs = w[:, None] * (torch.einsum("eij,ej->ei", A, zl[g]) + torch.einsum("eij,ej->ei", B, zl[d]))
        per = per.index_add(0, torch.as_tensor(g), pairs)
        y = torch.zeros(11 * N, dtype=torch.float64).index_put((dof.reshape(-1),), per.reshape(-1))
        r = K @ y - z
        rr, zz = rr + r @ r, zz + z @ z
    loss = rr / zz
    loss.backward()
    return float(loss.detach()), pt.grad.numpy()


@pytest.mark.parametrize("nz", [1, 2, 4, 5, 8])
def test_numbers_of_vectors(rsd, nz):
    """The products for several vectors at once, in groups of up to four, and vectors of odd length (11 * 33)."""
    from rsd_amd.configs import random_suspension
    conf, radii, L = random_suspension(33, 0.35, 22)
    sus = rsd.Suspension(conf, radii, rsd.default_config(L))
    sus.prepare_iterative(0.0)
    M, R, nnb, col, dist, cap = sus.iterative_system()
    gnn = rsd.Gnn(seed=4)
    p = gnn.params()
    p[-133:] = (0.05 * np.random.default_rng(6).standard_normal(133)).astype(np.float32)
    gnn.set_params(p)
    loss, grad, Z = sus.gnn_loss(gnn, nz=nz, seed=12)
    want, gwant = reference(p, M, R, nnb, col, dist, radii, Z)
    only, _, _ = sus.gnn_loss(gnn, nz=nz, seed=12, grad=False)
    assert only == loss
    # bounds as below
    assert abs(loss - want) <= 5.5e-5 * want
    assert relerr(gwant, grad) < 1e-3
    gnn.close()
    sus.close()


@pytest.mark.parametrize("n,phi", [(1, 0.01), (5, 0.01), (9, 0.05), (17, 0.4), (72, 0.5), (530, 0.3)])
def test_loss_and_gradient(rsd, n, phi):
    from rsd_amd.configs import random_suspension
    conf, radii, L = random_suspension(n, phi, 21)
    sus = rsd.Suspension(conf, radii, rsd.default_config(L))
    sus.prepare_iterative(0.1)
    M, R, nnb, col, dist, cap = sus.iterative_system()
    gnn = rsd.Gnn(seed=3)
    p = gnn.params()
    p[-133:] = (0.05 * np.random.default_rng(4).standard_normal(133)).astype(np.float32)
    gnn.set_params(p)
    loss, grad, Z = sus.gnn_loss(gnn, nz=3, seed=11)
    want, gwant = reference(p, M, R, nnb, col, dist, radii, Z)
    print(f"N={n}: {nnb.min()} to {nnb.max()} neighbours, loss {loss:.6e} (64 bits {want:.6e})", flush=True)
    # one particle: the preconditioner is the inverse and the loss |K P z - z|^2 / |z|^2 only FP64 rounding, two products
    # with 11 x 11 blocks, (2 * 121 * 2^-53)^2.  Else 7 stages of sums of up to 132 terms in FP32: 7 * 132 * 2^-24 = 5.5e-5 forward; forward and backward twice that,
    # and units whose pre-activation is that close to zero may switch: 1e-3 of a group's norm
    assert abs(loss - want) <= 5.5e-5 * want + (2 * 121 * 2.0 ** -53) ** 2
    off = [0, 192, 192 + 16768, 192 + 2 * 16768, 192 + 3 * 16768, len(p)]
    for a, b in zip(off[:-1], off[1:]):
        if np.linalg.norm(gwant[a:b]) > 0.0:
            assert relerr(gwant[a:b], grad[a:b]) < 1e-3, (a, b)
        else:
            assert np.all(grad[a:b] == 0.0), (a, b)
    gnn.close()
    sus.close()
