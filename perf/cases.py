"""The work that programs give this framework, as cases that can be timed.

Every case is one call, or the few calls that belong together, of the public Python interface: a step of a sheared
suspension on each of the routes that a program can choose, a batch of suspensions, the dense routines that a Fortran
program links in place of its own, and a training pass of the learned preconditioner.

  listed()             the cases, each a dict of plain values with a name of its own
  draw(rng)            another case of the same ranges
  prepare(case, seed)  what a program holds before the call: positions and radii on the host, contexts on the GPU
  run(state)           one pass; returns all that a program reads from it
  work(case)           the bytes and operations that one pass cannot do without
  exact(case, seed)    the pass's result in 64 bits by numpy, where the pass is plain linear algebra
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "regularized-stokesian-dynamics_amd"))

import rsd_amd  # noqa: E402

DT = 5e-4


# ------------------------------------------------------------------ the cases
def step_case(n, phi, **kw):
    """One step of one suspension.  contact: some spheres touch, as they do from the first few steps of a dense run on,
    so that the step takes its five collision sub-steps; without it the step has one.  images "config": the explicit
    Ewald image set (4 real images, |k| <= 6 2pi/L) in place of the truncation rule."""
    case = {"kind": "step", "n": n, "phi": phi, "bidisperse": False, "contact": False, "images": "rule",
            "route": "schur", "geometry": "periodic", "gravity": 0.0, "kbt": 0.0}
    case.update(kw)
    return case


def listed():
    return [
        # the smallest suspension anybody steps, as the smoke check does: launches and latency
        dict(step_case(16, 0.3), name="step_n16"),
        # a small dilute run of many steps (N=64, phi=0.2), once spheres have met
        dict(step_case(64, 0.2, contact=True), name="step_n64_contact"),
        # a Brownian suspension: a Cholesky factor of the mobility and two more assemblies in each step
        dict(step_case(240, 0.3, kbt=0.05), name="step_n240_brownian"),
        # a cloud settling under gravity in unbounded fluid: no periodic images, two right-hand sides
        dict(step_case(200, 0.2, geometry="free", gravity=1.0), name="step_n200_free_gravity"),
        # an odd, dense bidisperse suspension with the explicit image set
        dict(step_case(333, 0.45, bidisperse=True, contact=True, images="config"), name="step_n333_bidisperse_images"),
        # the headline suspension (N=512, phi=0.4) in the state that it is in through most of a run
        dict(step_case(512, 0.4, contact=True), name="step_n512_contact"),
        # the same by the iterative route: GMRES with FP32 inner iterations and the learned preconditioner
        dict(step_case(512, 0.4, contact=True, route="iterative"), name="step_n512_iterative"),
        # a ragged size, settling under gravity: two right-hand sides, one sub-step
        dict(step_case(997, 0.3, gravity=1.0), name="step_n997_gravity"),
        # the largest configuration: N=4096, bidisperse, phi=0.5
        dict(step_case(4096, 0.5, bidisperse=True), name="step_n4096_bidisperse"),
        # many independent suspensions of uneven sizes stepped together
        {"name": "batch_12", "kind": "batch", "count": 12, "n_lo": 108, "n_hi": 640, "phi": 0.4, "contact": True},
        # the resistance algebra behind a Fortran stepper: host matrices in, host matrices out
        {"name": "dense_host_n100", "kind": "dense", "n": 100},
        # the learned preconditioner's training: assemble a system, loss and gradient
        {"name": "train_n256", "kind": "train", "n": 256, "phi": 0.42, "nz": 4},
    ]


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["step", "options", "iterative", "batch", "dense", "train"], [8, 4, 2, 2, 2, 1])[0]
    if kind == "step":
        phi = round(rng.uniform(0.1, 0.5), 3)
        return step_case(log_int(rng, 12, 2500), phi, bidisperse=rng.random() < 0.4, contact=rng.random() < 0.6,
                         images="config" if rng.random() < 0.2 else "rule",
                         gravity=1.0 if rng.random() < 0.2 else 0.0)
    if kind == "options":
        phi = round(rng.uniform(0.1, 0.35), 3)
        if rng.random() < 0.5:
            return step_case(log_int(rng, 12, 700), phi, kbt=round(rng.uniform(0.01, 0.1), 3))
        # above a wall: few spheres, as the wall's images correct the translations alone
        wall = rng.random() < 0.3
        return step_case(log_int(rng, 12, 40 if wall else 700), min(phi, 0.2) if wall else phi,
                         geometry="wall" if wall else "free", gravity=rng.choice([0.0, 1.0]),
                         contact=rng.random() < 0.3)
    if kind == "iterative":
        return step_case(log_int(rng, 50, 600), round(rng.uniform(0.2, 0.4), 3), contact=rng.random() < 0.5,
                         route="iterative")
    if kind == "batch":
        lo = log_int(rng, 20, 200)
        return {"kind": "batch", "count": rng.randint(3, 12), "n_lo": lo, "n_hi": lo + rng.randint(50, 450),
                "phi": round(rng.uniform(0.2, 0.45), 3), "contact": rng.random() < 0.5}
    if kind == "dense":
        return {"kind": "dense", "n": log_int(rng, 8, 200)}
    return {"kind": "train", "n": log_int(rng, 40, 300), "phi": round(rng.uniform(0.35, 0.48), 3),
            "nz": rng.randint(2, 6)}


# ---------------------------------------------------------------- suspensions
def lees_edwards(d, L, strain):
    """Minimum image of the separations d (..., 3) in a cubic box sheared by `strain`."""
    nz = torch.round(d[..., 2] / L)
    x = d[..., 0] - nz * strain * L
    return torch.stack([x - L * torch.round(x / L), d[..., 1] - L * torch.round(d[..., 1] / L), d[..., 2] - L * nz], -1)


def suspension(n, phi, seed, bidisperse=False, contact=False, strain=0.0):
    """(positions, radii, L): spheres at random in a sheared cubic box with every surface gap >= 1e-3; with `contact` a
    few of the closest pairs overlap by up to 1.5e-3, as they do in a run (the steps carry no contact force).

    Spheres start on a random part of a face-centred lattice, are displaced at random, and are pushed apart along their
    lines of centres until none is closer than the gap."""
    rng = np.random.default_rng(seed)
    radii = np.ones(n)
    if bidisperse:
        radii = np.where(np.arange(n) < n // 2, 1.0, 1.4)
        rng.shuffle(radii)
    L = float((np.sum(4.0 / 3.0 * np.pi * radii ** 3) / phi) ** (1.0 / 3.0))
    m = int(math.ceil((n / 4.0) ** (1.0 / 3.0) - 1e-9))
    base = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])
    sites = (np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 1, 3) + base).reshape(-1, 3)
    sites = sites[rng.permutation(len(sites))[:n]] * (L / m)
    sites = sites + rng.uniform(-0.4, 0.4, (n, 3))
    sites[:, 0] += strain * sites[:, 2]  # into the sheared box
    gap = 1e-3
    pos = torch.tensor(sites, device="cuda")
    a = torch.tensor(radii, device="cuda")
    reach = a[:, None] + a[None, :] + gap
    reach.fill_diagonal_(0.0)
    for it in range(4000):
        d = lees_edwards(pos[:, None, :] - pos[None, :, :], L, strain)
        r = torch.sqrt((d * d).sum(-1))
        r.fill_diagonal_(1e9)
        if it % 8 == 0 and not bool((r < reach).any()):
            break
        push = (reach * (1.0 + 1e-3) - r).clamp_(min=0.0) * (r < reach * (1.0 + 5e-4))
        pos = pos + ((0.55 * push / r)[..., None] * d).sum(1)
    else:
        raise RuntimeError("the suspension did not relax")
    pos = pos.cpu().numpy()
    # into the box, as a run's wrap leaves them
    nz = np.floor(pos[:, 2] / L)
    pos[:, 2] -= nz * L
    pos[:, 0] -= nz * strain * L
    pos[:, :2] -= L * np.floor(pos[:, :2] / L)
    if contact:
        touch(pos, radii, rng)
    return np.ascontiguousarray(pos), radii, L


def touch(pos, radii, rng):
    """Moves one sphere of each of the closest separate pairs into its partner."""
    p, a = torch.tensor(pos, device="cuda"), torch.tensor(radii, device="cuda")
    r = torch.sqrt(((p[:, None, :] - p[None, :, :]) ** 2).sum(-1)) - a[:, None] - a[None, :]
    n = len(radii)
    r = torch.where(torch.ones_like(r).triu(1) > 0, r, torch.full_like(r, 1e9)).reshape(-1)
    close = torch.argsort(r, stable=True)[:4 * n].cpu().numpy()
    used, left = set(), max(1, n // 100)
    for k in close:
        i, j = int(k) // n, int(k) % n
        if left == 0 or i >= j:
            break
        if i in used or j in used:
            continue
        used |= {i, j}
        left -= 1
        d = pos[j] - pos[i]
        pos[j] = pos[i] + d / np.linalg.norm(d) * (radii[i] + radii[j] - rng.uniform(2e-4, 1.5e-3))


# -------------------------------------------------------------------- prepare
def make_step(case, seed):
    rng = np.random.default_rng(seed + 7919)
    periodic = case["geometry"] == "periodic"
    t = float(rng.uniform(0.05, 0.95)) if periodic else 0.0
    conf, radii, L = suspension(case["n"], case["phi"], seed, case["bidisperse"], case["contact"], t)
    if case["geometry"] == "wall":
        conf[:, 2] += 4.0  # above the wall z = 0
    sus = rsd_amd.Suspension(conf, radii, rsd_amd.default_config(L, gravity=case["gravity"]))
    if not periodic:
        sus.set_geometry(is_period=False, wall=case["geometry"] == "wall")
    if case["images"] == "config":
        sus.set_ewald_images(4, 6, 36)
    if case["kbt"]:
        sus.set_brownian(case["kbt"], seed=seed)
    if case["route"] == "iterative":
        sus.set_resistance_route(sus.RESIST_ITERATIVE)
        sus.set_iterative(sus.PRECOND_MIXED_LEARNED)
        sus.set_gnn(rsd_amd.Gnn.load(rsd_amd.GNN_PARAMS_PATH))
    return {"sus": sus, "conf": conf, "radii": radii, "t": t}


def make_batch(case, seed):
    rng = np.random.default_rng(seed + 104729)
    sizes = [int(v) for v in np.linspace(case["n_lo"], case["n_hi"], case["count"])]
    members, times = [], []
    for k, n in enumerate(sizes):
        t = float(rng.uniform(0.05, 0.95))
        conf, radii, L = suspension(n, case["phi"], seed * 64 + k, False, case["contact"], t)
        members.append((rsd_amd.Suspension(conf, radii, rsd_amd.default_config(L)), conf, radii))
        times.append(t)
    return {"members": members, "t": np.array(times), "batch": rsd_amd.Batch([m[0] for m in members])}


def dense_inputs(case, seed):
    """A grand mobility and a lubrication resistance of n spheres' shape and conditioning, as host matrices: the first
    decays with distance and is positive definite, the second couples neighbours by stiff symmetric blocks."""
    n = case["n"]
    rng = np.random.default_rng(seed)
    L = (4.0 / 3.0 * np.pi * n / 0.3) ** (1.0 / 3.0)
    pos = rng.uniform(0.0, L, (n, 3))
    d = pos[:, None, :] - pos[None, :, :]
    r = np.sqrt(np.einsum("ijk,ijk->ij", d, d))
    q = np.linalg.qr(rng.standard_normal((11, 11)))[0]
    block = (q * rng.uniform(0.3, 1.5, 11)) @ q.T
    M = np.kron(np.exp(-r / 1.5), block)
    M = 0.5 * (M + M.T) + 0.2 * np.eye(11 * n)
    near = np.triu((r < 2.6).astype(np.float64), 1) * rng.uniform(0.5, 40.0, (n, n))
    lap = np.diag(near.sum(0) + near.sum(1)) - near - near.T
    q = np.linalg.qr(rng.standard_normal((11, 11)))[0]
    R = np.kron(lap, (q * rng.uniform(0.1, 1.0, 11)) @ q.T)
    first = (np.arange(n)[:, None] * 11 + np.arange(6)).reshape(-1)
    rest = (np.arange(n)[:, None] * 11 + np.arange(6, 11)).reshape(-1)

    def blocks(A):
        return [np.asfortranarray(A[np.ix_(x, y)]) for x, y in ((first, first), (first, rest), (rest, rest))]

    return blocks(M), blocks(0.5 * (R + R.T)), rng.standard_normal(6 * n), rng.standard_normal(5 * n)


def prepare(case, seed):
    rsd_amd.init(0)
    if case["kind"] == "step":
        state = make_step(case, seed)
    elif case["kind"] == "batch":
        state = make_batch(case, seed)
    elif case["kind"] == "dense":
        M, R, fe, ein = dense_inputs(case, seed)
        state = {"M": M, "R": R, "fe": fe, "ein": ein}
    else:
        conf, radii, L = suspension(case["n"], case["phi"], seed)
        state = {"sus": rsd_amd.Suspension(conf, radii, rsd_amd.default_config(L)), "conf": conf, "radii": radii,
                 "gnn": rsd_amd.Gnn.load(rsd_amd.GNN_PARAMS_PATH), "nz": case["nz"], "seed": seed}
    state["kind"] = case["kind"]
    return state


# ------------------------------------------------------------------------ run
def outputs(sus):
    conf, u_pos = sus.state()
    u_par, s_hyd, nt = sus.last()
    return {"conf": conf, "u_pos": u_pos, "u_par": u_par, "s_hyd": s_hyd, "nt_dem": nt}


def run(state):
    if state["kind"] == "step":
        sus = state["sus"]
        sus.set_state(state["conf"], state["radii"])
        yeta, info = sus.step(DT, state["t"])
        return dict(outputs(sus), yeta=yeta, info=info)
    if state["kind"] == "batch":
        for sus, conf, radii in state["members"]:
            sus.set_state(conf, radii)
        yeta, info = state["batch"].step(DT, state["t"])
        per = [outputs(m[0]) for m in state["members"]]
        out = {k: np.concatenate([p[k].reshape(-1) for p in per]) for k in ("conf", "u_pos", "u_par", "s_hyd")}
        return dict(out, nt_dem=np.array([p["nt_dem"] for p in per]), yeta=yeta, info=info)
    if state["kind"] == "dense":
        # what the linked routines of a Fortran stepper do in one sub-step
        u_par, s_hyd, rpp = rsd_amd.stepper_nogmres(*state["M"], *state["R"], state["fe"], state["ein"])
        return {"u_par": u_par, "s_hyd": s_hyd, "rpp": rpp}
    sus = state["sus"]
    sus.set_state(state["conf"], state["radii"])
    sus.prepare_iterative(0.0)
    loss, grad, z = sus.gnn_loss(state["gnn"], nz=state["nz"], seed=state["seed"])
    return {"loss": loss, "grad": grad, "z": z}


# ----------------------------------------------------------------------- work
def images(n, phi, kind):
    """(real images, wave vectors) of one pair: the reference's truncation rule at LINERR = 1e-4 gives half-widths 2
    and 2 in a cubic box."""
    return (9 ** 3, 924) if kind == "config" else (5 ** 3, 5 ** 3 - 1)


def step_flops(n, phi, case_images="rule", periodic=True, contact=False, kbt=0.0):
    """The dense algebra that a step cannot do without: a Cholesky factor of the 11N mobility with the inverse of its
    6N Schur complement, a factor of the 6N resistance and a few products in each sub-step; and the pair sums."""
    real, recip = images(n, phi, case_images) if periodic else (1, 0)
    pairs = 0.5 * n * (n - 1) * (1000.0 * real + 250.0 * recip)
    n11, n6, n3 = 11.0 * n, 6.0 * n, 3.0 * n
    dense = n11 ** 3 / 3 + 2 * n6 ** 3 / 3 + n6 ** 3 / 3 + 10 * n11 ** 2
    if contact:  # four more sub-steps, each solved again
        dense += 4 * 10 * 2 * n6 ** 2
    if kbt:
        dense += n3 ** 3 / 3 + 6 * n3 ** 2
        pairs *= 3
    return pairs + dense


def work(case):
    n = case.get("n", 0)
    if case["kind"] == "step":
        if case["route"] == "iterative":
            # assembly, and per sub-step some 40 products with the 11N mobility
            subs = 5 if case["contact"] else 1
            flops = 0.5 * n * (n - 1) * (1000.0 * 125 + 250.0 * 124) + subs * 40 * 2 * (11.0 * n) ** 2
        else:
            flops = step_flops(n, case["phi"], case["images"], case["geometry"] == "periodic", case["contact"],
                               case["kbt"])
        return {"bytes": 8.0 * (4 * n + 3 * n + 6 * n + 6 * n + 5 * n + 5), "flops": flops}
    if case["kind"] == "batch":
        sizes = [int(v) for v in np.linspace(case["n_lo"], case["n_hi"], case["count"])]
        return {"bytes": 8.0 * sum(24 * m + 5 for m in sizes),
                "flops": sum(step_flops(m, case["phi"], contact=case["contact"]) for m in sizes)}
    if case["kind"] == "dense":
        n6, n5, n11 = 6.0 * n, 5.0 * n, 11.0 * n
        return {"bytes": 8.0 * (2 * (n6 * n6 + n6 * n5 + n5 * n5) + n6 * n6 + 2 * n11),
                "flops": n11 ** 3 + n6 ** 3 / 3 + 4 * n6 ** 2}
    pair_sums = 0.5 * n * (n - 1) * (1000.0 * 125 + 250.0 * 124)
    return {"bytes": 8.0 * (4 * n + case["nz"] * 11 * n) + 4.0 * rsd_amd.GNN_PARAMS * 2,
            "flops": pair_sums + case["nz"] * 4 * 2 * (11.0 * n) ** 2}


# ---------------------------------------------------------------------- exact
def exact(case, seed):
    """The dense case is plain linear algebra.  The other cases sum lattice series and tabulated forces over pairs, in
    64 bits already; there is no short numpy form of them."""
    if case["kind"] != "dense":
        return None
    (app, apq, aqq), (rfu, rfe, rse), fe, ein = dense_inputs(case, seed)
    n6 = len(fe)
    W = np.linalg.inv(np.block([[app, apq], [apq.T, aqq]]))
    rpp, rpq, rqq = W[:n6, :n6] + rfu, W[:n6, n6:] + rfe, W[n6:, n6:] + rse
    u = np.linalg.solve(rpp, fe + rpq @ ein)
    s = rpq.T @ np.linalg.solve(rpp, rpq @ ein) - rqq @ ein
    return {"u_par": u, "s_hyd": s, "rpp": np.asfortranarray(rpp)}
