"""Performance cases of the engine's public entry points (atomnn_amd.nnp, atomnn_amd.serve).

listed() names the cases, draw(rng) makes one more of the same ranges, prepare(case, seed) builds
what a program holds before the call (model handle, structures, resident batch, MD state, server,
training set), run(state) is one pass through the entry point, exact(case, seed) is the same result
from plain torch in 64 bits (direct sums over neighbours and triplets, gradients by autograd),
and work(case) counts the bytes and operations a pass cannot do without.

Models (atomnn_amd.synth): "one" (the 64-atom workload: 1 species, rc 6, 8 G2 + 8 G4), "two" (the
4096-atom workload: 2 species, rc 6, 32 G2 + 48 G4, 80-32-32-1), "three" (the precision and serving
workloads: 3 species, rc 6.5, 36 G2 + 48 G4, 84-64-64-1) and "zeta16" (2 species, rc 6, the angular
exponents zeta = 1, 2, 4, 16 of the usual G4 sets, 16 G2 + 48 G4, 64-32-32-1).

A "mixed" case returns its results as float32, the precision that form computes in.
"""
from __future__ import annotations

import atexit
import functools
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from atomnn_amd import synth
from atomnn_amd.nnp import (LOSS_MSE, MD, NNP, NNP_ATOM_ENERGY, NNP_FORCE, NNP_PREC_MIXED, NNP_VACUUM_ENERGY, Train)
from atomnn_amd.serve import Server

DENSITY = {"one": 0.05, "two": 0.05, "three": 0.06, "zeta16": 0.05}
FRACTIONS = {"one": [1.0], "two": [0.5, 0.5], "three": [0.4, 0.3, 0.3], "zeta16": [0.5, 0.5]}
VACUUM = [-3.1, -4.7, -2.2]  # eV per atom, the species' reference energies a potential file carries
MASSES = {"two": [30.0, 60.0], "three": [12.0, 30.0, 60.0]}
MD_DT = 0.1         # fs: the synthetic cells are far from equilibrium, a long run must stay a liquid
MV2E = 103.642696   # eV per amu A^2 / fs^2
KB = 8.617333262e-5  # eV / K
BETA = 1.0          # force weight of the energy + force loss


def listed():
    return [
        # one call on a small unit cell (27 images per pair): what a relaxation or a single-point
        # driver does thousands of times, all latency
        _case("single_64", "compute", "one", 64),
        # the headline structure through the synchronous call a C or C++ driver makes
        _case("single_4096", "compute", "two", 4096),
        # one large, odd-sized strained cell in the precision form, as a screening program sends it
        _case("single_11003_mixed", "compute", "three", 11003, triclinic=True, mixed=True),
        # the classical angular set with zeta up to 16, which the moment expansion does not cover
        _case("single_1500_zeta16", "compute", "zeta16", 1500),
        # the headline metric: a resident structure evaluated again, results fetched
        _case("resident_4096", "resident", "two", 4096),
        # a resident batch of large cells in the precision form, the throughput case
        _case("resident_16x4096_mixed", "resident", "three", 4096, count=16, mixed=True),
        # uneven small triclinic cells in one call: a data set evaluated batch by batch
        _case("batch_20_uneven", "batch", "two", 512, count=20, uneven=True, triclinic=True),
        # descriptors alone, as a program that builds a training database takes them
        _case("descriptors_3001", "symm", "three", 3001),
        # molecular dynamics: 25 steps on the device, then positions, velocities and forces
        _case("md_4096", "md", "two", 4096, steps=25),
        # a burst of requests of very different sizes at the continuous-batching server
        _case("serve_20_mixed", "serve", "three", 8000, count=20, uneven=True, triclinic=True, mixed=True),
        # one optimiser step of energy training: loss and gradient over a batch
        _case("train_16x2048", "train", "three", 2048, count=16),
        # one optimiser step of energy + force training on small, uneven cells
        _case("train_force_24_uneven", "train_force", "two", 700, count=24, uneven=True),
    ]


def draw(rng):
    path = rng.choice(["compute", "compute", "compute", "resident", "resident", "batch", "symm", "md", "serve",
                       "train", "train_force", "compute_zeta16"])
    if path == "compute_zeta16":
        return _case(None, "compute", "zeta16", _size(rng, 24, 1500), triclinic=rng.random() < 0.5)
    if path == "compute":
        model = rng.choice(["one", "two", "three"])
        n = _size(rng, 8, {"one": 2000, "two": 8192, "three": 16000}[model])
        mixed = rng.random() < 0.4
        cluster = n <= 400 and rng.random() < 0.25
        return _case(None, "compute", model, n, triclinic=not cluster and rng.random() < 0.5, mixed=mixed,
                     cluster=cluster)
    if path == "resident":
        if rng.random() < 0.5:
            return _case(None, "resident", rng.choice(["two", "three"]), _size(rng, 300, 16384),
                         mixed=rng.random() < 0.5)
        return _case(None, "resident", rng.choice(["two", "three"]), _size(rng, 256, 4096), count=rng.randint(2, 16),
                     uneven=rng.random() < 0.5, triclinic=rng.random() < 0.5, mixed=True)
    if path == "batch":
        return _case(None, "batch", rng.choice(["two", "three"]), _size(rng, 24, 1024), count=rng.randint(2, 20),
                     uneven=rng.random() < 0.7, triclinic=True, mixed=rng.random() < 0.3)
    if path == "symm":
        return _case(None, "symm", rng.choice(["one", "two", "three"]), _size(rng, 32, 4096))
    if path == "md":
        return _case(None, "md", rng.choice(["two", "three"]), _size(rng, 300, 6000), steps=rng.randint(5, 40))
    if path == "serve":
        return _case(None, "serve", rng.choice(["two", "three"]), _size(rng, 500, 10000), count=rng.randint(3, 20),
                     uneven=True, triclinic=True, mixed=rng.random() < 0.7)
    if path == "train":
        return _case(None, "train", rng.choice(["two", "three"]), _size(rng, 48, 2048), count=rng.randint(4, 16),
                     uneven=rng.random() < 0.5)
    return _case(None, "train_force", rng.choice(["two", "three"]), _size(rng, 48, 800), count=rng.randint(2, 20),
                 uneven=rng.random() < 0.5)


def _size(rng, lo, hi):
    """An atom count spread over the logarithm of [lo, hi], most of them odd or ragged."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _case(name, path, model, atoms, count=1, uneven=False, triclinic=False, mixed=False, cluster=False, steps=0):
    """atoms: of each structure (of the largest one with uneven); steps: MD steps of a pass."""
    c = dict(path=path, model=model, atoms=atoms, count=count, uneven=uneven, triclinic=triclinic, mixed=mixed,
             cluster=cluster, steps=steps)
    return c if name is None else dict(name=name, **c)


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=None)
def _folder():
    d = tempfile.mkdtemp(prefix="atomnn_cases_")
    atexit.register(shutil.rmtree, d, True)
    return d


@functools.lru_cache(maxsize=None)
def _potential(model):
    """(potential as a reader of its file sees it, path of the file)."""
    if model == "zeta16":
        rng = np.random.default_rng(synth.SEED0 + 16)
        pot = synth.make_potential(["A", "B"], 6.0, 8, [0.005, 0.05], [1.0, 2.0, 4.0, 16.0], [1, -1], [32, 32], rng)
        cell = synth.cubic_cell(128, 0.05)
        pot = synth.precondition(pot, synth.Structure(synth.species_exact(128, [0.5, 0.5], rng),
                                                      synth.random_positions(128, cell, 2.0, synth.SEED0 + 116), cell))
    else:
        pot = synth.workload_potential({"one": "plain64", "two": "plain4096", "three": "mixed64x4096"}[model])
    pot.evac = {t: VACUUM[t] for t in range(pot.ntypes)}
    path = os.path.join(_folder(), model + ".ann")
    pot.write(path)
    return pot.quantized(), path


def _sizes(case):
    """Atom counts of the case's structures (the same for every seed)."""
    n, k = case["atoms"], case["count"]
    if not case["uneven"]:
        return [n] * k
    lo, rng = min(8, n), np.random.default_rng(1000 * n + k)
    return [n] + [int(round(math.exp(rng.uniform(math.log(lo), math.log(n))))) for _ in range(k - 1)]


def _structures(case, seed):
    rng = np.random.default_rng([seed, case["atoms"], case["count"]])
    rho, out = DENSITY[case["model"]], []
    for n in _sizes(case):
        cell = synth.strained_cell(n, rho, 0.05, rng) if case["triclinic"] else synth.cubic_cell(n, rho)
        types = synth.species_exact(n, FRACTIONS[case["model"]], rng)
        pos = synth.random_positions(n, cell, 1.8, int(rng.integers(0, 2**62)))
        out.append(synth.Structure(types, pos, None if case["cluster"] else cell))
    return out


def _velocities(case, s, seed):
    """Maxwell-Boltzmann at 300 K without centre-of-mass motion."""
    rng = np.random.default_rng([seed, 17])
    m = np.array(MASSES[case["model"]])[s.types]
    v = rng.normal(0.0, 1.0, (s.natoms, 3)) * np.sqrt(KB * 300.0 / (m * MV2E))[:, None]
    return v - v.mean(axis=0)


def _targets(strucs, seed):
    """Reference energies and forces of a training set."""
    rng = np.random.default_rng([seed, 29])
    e = np.array([rng.normal(-3.0, 0.2) * s.natoms for s in strucs])
    return e, [rng.normal(0.0, 0.5, (s.natoms, 3)) for s in strucs]


def _file_params(pot):
    """The potential's parameters, species by species: the biases, then each weight matrix column-major."""
    parts = []
    for t in range(pot.ntypes):
        parts += [b for b in pot.biases[t]] + [W.reshape(-1, order="F") for W in pot.weights[t]]
    return np.concatenate(parts)


def _train_params(pot, seed):
    """Parameters an optimiser is at: the file's, moved a little."""
    x = _file_params(pot)
    return x + 0.02 * np.random.default_rng([seed, 41]).normal(size=x.shape[0])


def _flags(case):
    return NNP_FORCE | NNP_ATOM_ENERGY | NNP_VACUUM_ENERGY | (NNP_PREC_MIXED if case["mixed"] else 0)


# ------------------------------------------------------------------ the measured passes
def prepare(case, seed):
    pot, path = _potential(case["model"])
    strucs = _structures(case, seed)
    st = {"case": case, "model": NNP.read(path), "structures": strucs, "flags": _flags(case)}
    kind = case["path"]
    if kind == "compute":
        st["call"] = st["model"].compute_into(strucs[0], st["flags"])
    elif kind == "resident":
        st["resident"] = st["model"].resident(strucs, st["flags"])
    elif kind == "md":
        st["md"] = MD(st["model"], strucs[0], MASSES[case["model"]], _velocities(case, strucs[0], seed), dt=MD_DT)
        st["md"].model = st["model"]  # outlives the MD state
    elif kind == "serve":
        st["server"] = Server(st["model"], st["flags"])
    elif kind in ("train", "train_force"):
        e, f = _targets(strucs, seed)
        st["train"] = Train(st["model"], strucs, e)
        st["train"].model = st["model"]  # outlives the training set
        st["x"], st["batch"] = _train_params(pot, seed), np.arange(len(strucs), dtype=np.int32)
        if kind == "train_force":
            st["train"].set_forces(f)
    return st


def run(state):
    case = state["case"]
    kind = case["path"]
    if kind == "compute":
        return _results([state["call"]()], case["mixed"])
    if kind == "resident":
        state["resident"].run()
        return _results(state["resident"].fetch(), case["mixed"])
    if kind == "batch":
        return _results(state["model"].compute_batch(state["structures"], state["flags"]), case["mixed"])
    if kind == "symm":
        return state["model"].symm(state["structures"][0])
    if kind == "md":
        state["md"].step(case["steps"])
        s = state["md"].state()
        return {k: s[k] for k in ("pos", "vel", "force", "epot", "ekin")}
    if kind == "serve":
        pending = [state["server"].submit(s) for s in state["structures"]]
        return _results([p.wait() for p in pending], case["mixed"])
    if kind == "train":
        return state["train"].error(state["x"], state["batch"], LOSS_MSE)
    return state["train"].error_force(state["x"], state["batch"], LOSS_MSE, 1.0, BETA)


def _results(res, mixed):
    """(energy, per-atom energies, forces) of each structure; the precision form's as float32."""
    if not mixed:
        return res
    return [(np.float32(e), ea.astype(np.float32), f.astype(np.float32)) for e, ea, f in res]


# ------------------------------------------------------------------ the same results in 64 bits
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=_dev())


def _neighbours(pos, cell, rc):
    """Padded neighbour entries (r_i - r_j - T [N,P,3], j [N,P], real [N,P], nearest image of j [N,P])."""
    n = pos.shape[0]
    if cell is None:
        shifts, fro = torch.zeros((1, 3), dtype=torch.float64, device=pos.device), 0.0
    else:
        c = cell.cpu().numpy()
        vol = abs(np.linalg.det(c))
        h = [vol / np.linalg.norm(np.cross(c[(d + 1) % 3], c[(d + 2) % 3])) for d in range(3)]
        # with fractional offsets in [-1/2, 1/2], image m is at least (m - 1/2) h away
        m = [max(0, int(math.floor(rc / h[d] + 0.5))) for d in range(3)]
        g = [(a, b, d) for a in range(-m[0], m[0] + 1) for b in range(-m[1], m[1] + 1) for d in range(-m[2], m[2] + 1)]
        shifts = torch.tensor(g, dtype=torch.float64, device=pos.device) @ cell
        fro, inv = float(np.linalg.norm(c)), torch.linalg.inv(cell)
    step = max(1, int(8e6 // (n * shifts.shape[0])))
    rows = []
    for i0 in range(0, n, step):
        d0 = pos[i0:i0 + step, None, :] - pos[None, :, :]
        if cell is not None:
            f = d0 @ inv
            d0 = (f - torch.round(f)) @ cell
        r = d0[:, :, None, :] - shifts
        d2 = (r * r).sum(-1)
        own = torch.arange(i0, min(n, i0 + step), device=pos.device)[:, None] == torch.arange(n, device=pos.device)
        near = torch.zeros_like(d2, dtype=torch.bool)
        near.scatter_(2, d2.argmin(2, keepdim=True), True)
        near &= ~own[:, :, None] & (d2 < fro * fro)
        i, j, k = torch.nonzero((d2 <= rc * rc) & (d2 > 1e-6), as_tuple=True)
        rows.append((i + i0, j, r[i, j, k], near[i, j, k]))
    i, j, r, near = (torch.cat([x[q] for x in rows]) for q in range(4))
    count = torch.bincount(i, minlength=n)
    width = max(1, int(count.max()) if n else 1)
    slot = torch.arange(i.shape[0], device=pos.device) - (torch.cumsum(count, 0) - count)[i]
    R = torch.full((n, width, 3), 2.0 * rc, dtype=torch.float64, device=pos.device)
    J = torch.zeros((n, width), dtype=torch.int64, device=pos.device)
    real = torch.zeros((n, width), dtype=torch.bool, device=pos.device)
    mn = torch.zeros_like(real)
    R[i, slot], J[i, slot], real[i, slot], mn[i, slot] = r, j, True, near
    return R, J, real, mn


def _symmetry(pot, ti, R, tj, real):
    """Descriptors [n, nG] of centres of species ti by direct sums over entries and pairs."""
    T, rc = pot.ntypes, pot.rc
    d = torch.sqrt((R * R).sum(-1))
    fc = 0.5 * (torch.cos(d * (math.pi / rc)) + 1.0)
    of = [(real & (tj == b)).double() for b in range(T)]
    G = []
    for b in range(T):
        for rs, eta in pot.radial[(ti, b)]:
            G.append((torch.exp(-eta * (d - rs) ** 2) * fc * of[b]).sum(1))
    u = R / d[:, :, None]
    cos = (u[:, :, None, :] * u[:, None, :, :]).sum(-1)
    upper = torch.triu(torch.ones(R.shape[1], R.shape[1], dtype=torch.float64, device=R.device), 1)
    leg, term = {}, {}
    for bb in range(T):
        for a in range(bb + 1):
            alpha, fns = pot.angular[(ti, a, bb)]
            for eta, zeta, lam in fns:
                e, c = (eta, alpha), (zeta, lam)
                if e not in leg:
                    leg[e] = torch.exp(-((1.0 / eta) ** alpha) * d ** alpha) * fc
                if c not in term:
                    term[c] = (0.5 * (1.0 + lam * cos)).abs() ** int(zeta)
                A = term[c] * upper if a == bb else term[c]
                G.append(((A * (leg[e] * of[bb])[:, None, :]).sum(2) * (leg[e] * of[a])).sum(1))
    return torch.stack(G, 1)


def _network(pot, ti, G, W, b):
    a = _t(pot.inpw[ti]) * (G + _t(pot.inpb[ti]))
    for l in range(len(W)):
        a = a @ W[l].T + b[l]
        if l < len(W) - 1:
            a = torch.tanh(a)
    return pot.outb.get(ti, 0.0) + pot.outw.get(ti, 1.0) * a[:, 0]


def _net_tensors(pot):
    return ([[_t(W) for W in pot.weights[t]] for t in range(pot.ntypes)],
            [[_t(b) for b in pot.biases[t]] for t in range(pot.ntypes)])


def _by_species(types, ti, width):
    """Centres of species ti in pieces whose pair tables stay below about 1 GB each."""
    idx = torch.nonzero(types == ti)[:, 0]
    return torch.split(idx, max(1, int(2e6 // (width * width)))) if idx.numel() else []


def _evaluate(pot, types, pos, cell, W, b, vacuum=True):
    """Energy, per-atom energies and forces with the reference's reactions (minimum image only)."""
    R, J, real, mn = _neighbours(pos, cell, pot.rc)
    ea = torch.zeros(pos.shape[0], dtype=torch.float64, device=pos.device)
    F = torch.zeros_like(pos)
    for ti in range(pot.ntypes):
        for idx in _by_species(types, ti, R.shape[1]):
            r = R[idx].clone().requires_grad_(True)
            e = _network(pot, ti, _symmetry(pot, ti, r, types[J[idx]], real[idx]), W[ti], b[ti])
            X = -torch.autograd.grad(e.sum(), r)[0] * real[idx][:, :, None]
            ea[idx] = e.detach() + (pot.evac.get(ti, 0.0) if vacuum else 0.0)
            F[idx] += X.sum(1)
            F.index_add_(0, J[idx].reshape(-1), -(X * mn[idx][:, :, None]).reshape(-1, 3))
    return ea.sum(), ea, F


def _np(*xs):
    return tuple(x.detach().cpu().numpy() for x in xs)


def _split_params(pot, x):
    """The parameter vector's tensors: per species weights and biases (views, so gradients reach x)."""
    Ws, bs, at = [], [], 0
    for t in range(pot.ntypes):
        bt, wt = [], []
        for b in pot.biases[t]:
            bt.append(x[at:at + b.size])
            at += b.size
        for W in pot.weights[t]:
            wt.append(x[at:at + W.size].reshape(W.shape[1], W.shape[0]).T)
            at += W.size
        Ws.append(wt)
        bs.append(bt)
    return Ws, bs


def _training(case, pot, seed):
    """Loss sums and the gradient: 0.5 dE^2 per structure with dE = (E - E_ref) / N, and with
    forces beta/2 |(F - F_ref) / N|^2 per atom."""
    strucs = _structures(case, seed)
    eref, fref = _targets(strucs, seed)
    forces = case["path"] == "train_force"
    x = _t(_train_params(pot, seed)).requires_grad_(True)
    err, grad = np.zeros(3 if forces else 2), torch.zeros_like(x)
    for s, e0, f0 in zip(strucs, eref, fref):
        types, n = _t(s.types).long(), s.natoms
        R, J, real, mn = _neighbours(_t(s.pos), _t(s.cell), pot.rc)
        W, b = _split_params(pot, x)
        E, F, parts = 0.0, torch.zeros((n, 3), dtype=torch.float64, device=x.device), []
        for ti in range(pot.ntypes):
            for idx in _by_species(types, ti, R.shape[1]):
                r = R[idx].clone().requires_grad_(forces)
                G = _symmetry(pot, ti, r, types[J[idx]], real[idx])
                # the networks see a leaf copy, so that dE/dG and its gradients stay in the network
                g = G.detach().requires_grad_(forces)
                e = _network(pot, ti, g, W[ti], b[ti]).sum()
                E = E + e
                if forces:
                    y = torch.autograd.grad(e, g, create_graph=True)[0]
                    X = -torch.autograd.grad(G, r, y.detach(), retain_graph=True)[0] * real[idx][:, :, None]
                    F[idx] += X.sum(1)
                    F.index_add_(0, J[idx].reshape(-1), -(X * mn[idx][:, :, None]).reshape(-1, 3))
                    parts.append((ti, idx, r, G, y))
        dE = (E - float(e0)) / n
        loss = 0.5 * dE * dE
        err[0] += float(loss.detach())
        err[1] += float(dE.detach()) ** 2
        if forces:
            fd = (F - _t(f0)) / n
            err[0] += 0.5 * BETA * float((fd * fd).sum())
            err[2] += float((fd * fd).sum())
            gF = BETA * fd / n  # dL/dF; X enters F_i, and -X enters F_j where the entry reacts
            for ti, idx, r, G, y in parts:
                phi = (gF[idx][:, None, :] - gF[J[idx]] * mn[idx][:, :, None]) * real[idx][:, :, None]
                # sum_ij phi . X = -y . (dG/dr phi): the directional derivative by the double-vjp form
                v = torch.zeros_like(G).requires_grad_(True)
                back = torch.autograd.grad(G, r, v, create_graph=True)[0]
                V = torch.autograd.grad(back, v, phi)[0]
                loss = loss - (y * V).sum()
        grad += torch.autograd.grad(loss, x)[0]
    return err, grad.detach().cpu().numpy()


def _trajectory(case, pot, seed):
    """Velocity Verlet from the same start: half kick, drift, return to the cell, forces, half kick."""
    s = _structures(case, seed)[0]
    types, x, cell, v = _t(s.types).long(), _t(s.pos), _t(s.cell), _t(_velocities(case, s, seed))
    m = _t(np.array(MASSES[case["model"]]) * MV2E)[types][:, None]
    W, b = _net_tensors(pot)
    inv = torch.linalg.inv(cell)
    F = _evaluate(pot, types, x, cell, W, b, vacuum=False)[2]
    for _ in range(case["steps"]):
        v = v + 0.5 * MD_DT * F / m
        f = (x + MD_DT * v) @ inv
        x = (f - torch.floor(f)) @ cell
        E, _, F = _evaluate(pot, types, x, cell, W, b, vacuum=False)
        v = v + 0.5 * MD_DT * F / m
    return {"pos": x.cpu().numpy(), "vel": v.cpu().numpy(), "force": F.cpu().numpy(), "epot": float(E),
            "ekin": float((0.5 * m * v * v).sum())}


def exact(case, seed):
    pot, _ = _potential(case["model"])
    kind = case["path"]
    if kind in ("train", "train_force"):
        return _training(case, pot, seed)
    if kind == "md":
        return _trajectory(case, pot, seed)
    W, b = _net_tensors(pot)
    strucs = _structures(case, seed)
    if kind == "symm":
        s = strucs[0]
        types = _t(s.types).long()
        R, J, real, _ = _neighbours(_t(s.pos), None if s.cell is None else _t(s.cell), pot.rc)
        G = torch.zeros((s.natoms, max(pot.ninput(t) for t in range(pot.ntypes))), dtype=torch.float64, device=_dev())
        for ti in range(pot.ntypes):
            for idx in _by_species(types, ti, R.shape[1]):
                g = _symmetry(pot, ti, R[idx], types[J[idx]], real[idx])
                G[idx, :g.shape[1]] = g
        return G.cpu().numpy()
    return [_np(*_evaluate(pot, _t(s.types).long(), _t(s.pos), None if s.cell is None else _t(s.cell), W, b))
            for s in strucs]


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    """Bytes: positions and species in, results out, parameters once.  Operations: per neighbour
    entry the radial functions and, where the angular exponents allow it, the moment form of the
    angular sums (35 monomials); with zeta = 16 every triplet; per atom the networks."""
    pot, _ = _potential(case["model"])
    kind, N = case["path"], float(sum(_sizes(case)))
    P = DENSITY[case["model"]] * 4.0 / 3.0 * math.pi * pot.rc ** 3  # entries per atom
    nR = len(pot.radial[(0, 0)])
    fns = pot.angular[(0, 0, 0)][1]
    NE, NC = len({f[0] for f in fns}), len({f[1:] for f in fns})
    if max(f[1] for f in fns) <= 4:
        sums, grads = 35.0 * (2 + 2 * NE) + 13 * NE, 64.0 + 216 * NE
    else:
        sums, grads = 0.5 * P * (8 + 5 * NC + 2 * NE * NC), 0.5 * P * (30 + 4 * NC + 4 * NE * NC)
    descr, force = P * (20 + 6 * nR + sums), P * (10 + 8 * nR + grads)
    w = float(np.mean([sum(W.size for W in pot.weights[t]) for t in range(pot.ntypes)]))
    nG = float(np.mean([pot.ninput(t) for t in range(pot.ntypes)]))
    params = 8.0 * pot.ntypes * w
    if kind == "symm":
        return {"bytes": N * (28 + 8 * nG), "flops": N * descr}
    if kind == "train":  # forward, back-propagation and gradient rows over the resident descriptors
        return {"bytes": N * 8 * nG + 2 * params, "flops": N * 6 * w}
    if kind == "train_force":  # resident descriptors; forces, then their tangents and both network passes
        return {"bytes": N * (8 * nG + 24 + 28) + 2 * params, "flops": N * (2 * force + 16 * w)}
    steps = max(1, case["steps"])
    return {"bytes": N * (28 + 32) * steps + params, "flops": N * (descr + force + 4 * w) * steps}
