"""Timed cases of the framework's work, through its public entry points.

Each case is one of the things a user of the framework has it do:

  calc   the ASE-style calculator on small silicon structures: energy, forces
         and stress of one new geometry after another (geometry optimisation,
         point defects).  Latency and launches count.
  eval   the engine's evaluation of silicon: new coordinates, neighbor lists,
         energy, forces and virial (a force call of an outside driver).
  md     device-resident velocity-Verlet molecular dynamics of silicon, lists
         rebuilt every step, from a few thousand atoms to a million.
  batch  many independent amorphous silicon cells of 64 to 2048 atoms
         evaluated together (screening).
  ewald  Coulomb energy, forces and stress of rocksalt by Ewald summation to
         1e-6, from 512 to 262,144 ions.
  relax  damped charge dynamics of electronegativity equalisation on
         amorphous silica, from zero charges.
  warm   the same charges to 1e-6 eV/e from the learned start.
  lj     Lennard-Jones argon dynamics, lists rebuilt every 10 steps.
  comb   dynamics of COMB's local silica terms (angles, charge-dependent
         pairs, bond-order attraction) at fixed charges.

A pass of `calc`, `eval` and `ewald` evaluates two geometries in turn, as a
driver that moves the atoms does.  exact() restates every model in plain
torch in 64 bits.
"""
import itertools
import math

import numpy as np
import torch

from pysic_amd import structures as st

EWALD = dict(rc=10.0, sigma=2.0443, kc=2.5713, eps=0.00552635)
LIST_SI = 3.5        # Tersoff cutoff 3.0 + skin 0.5
LIST_COMB = 3.55
LJ_RC, LJ_SKIN = 2.5 * 3.405, 0.5


# --- the cases ------------------------------------------------------------------

def listed():
    return [
        # a point defect in a 3x3x3 supercell: the smallest call, all latency
        {"name": "calc_si_215", "kind": "calc", "nx": 3, "ny": 3, "nz": 3, "vacancies": 1},
        # the 8x8x8 supercell that the parity tests use
        {"name": "eval_si_4096", "kind": "eval", "nx": 8, "ny": 8, "nz": 8, "vacancies": 0},
        # an ordinary simulation cell with defects, run for a while
        {"name": "md_si_5757", "kind": "md", "nx": 8, "ny": 9, "nz": 10, "vacancies": 3,
         "steps": 200},
        # the headline workload
        {"name": "md_si_1048576", "kind": "md", "nx": 64, "ny": 64, "nz": 32, "vacancies": 0,
         "steps": 50},
        # the batched workload
        {"name": "batch_asi_512", "kind": "batch", "cells": 512, "nmin": 64, "nmax": 2048},
        # a small ionic crystal
        {"name": "ewald_nacl_1000", "kind": "ewald", "nx": 5, "ny": 5, "nz": 5},
        # the large ionic crystal
        {"name": "ewald_nacl_262144", "kind": "ewald", "nx": 32, "ny": 32, "nz": 32},
        # charge relaxation from zero on a small cell (labels for training)
        {"name": "relax_sio2_768", "kind": "relax", "n_si": 256, "steps": 60},
        # charges of a large cell from the learned start
        {"name": "warm_sio2_24576", "kind": "warm", "n_si": 8192},
        # pair-potential dynamics, ordinary and large
        {"name": "lj_ar_13500", "kind": "lj", "nx": 15, "ny": 15, "nz": 15, "steps": 100},
        {"name": "lj_ar_1048576", "kind": "lj", "nx": 64, "ny": 64, "nz": 64, "steps": 40},
        # many-body charge-dependent dynamics
        {"name": "comb_sio2_24576", "kind": "comb", "n_si": 8192, "steps": 20},
    ]


def _reps(rng, per_cell, lo, hi, least):
    """Repeats per axis of a box of about exp(uniform) atoms."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    edge = (n / per_cell) ** (1.0 / 3.0)
    r = [max(least, round(edge * rng.uniform(0.8, 1.25))) for _ in range(2)]
    r.append(max(least, int(n / per_cell / (r[0] * r[1]))))
    return {"nx": r[0], "ny": r[1], "nz": r[2]}


def draw(rng):
    kind = rng.choice(["calc", "eval", "md", "batch", "ewald", "relax", "warm", "lj", "comb"])
    c = {"kind": kind}
    if kind == "calc":
        c.update(_reps(rng, 8, 100, 1000, 2), vacancies=rng.randint(0, 3))
    elif kind == "eval":
        c.update(_reps(rng, 8, 512, 131072, 3), vacancies=rng.randint(0, 7))
    elif kind == "md":
        c.update(_reps(rng, 8, 2000, 1000000, 4), vacancies=rng.randint(0, 7))
        c["steps"] = max(20, min(200, int(4e7 / (8 * c["nx"] * c["ny"] * c["nz"]))))
    elif kind == "batch":
        c.update(cells=int(math.exp(rng.uniform(math.log(8), math.log(512)))), nmin=64,
                 nmax=rng.randint(400, 2048))
    elif kind == "ewald":
        c.update(_reps(rng, 8, 512, 200000, 4))
    elif kind == "relax":
        c["n_si"] = int(math.exp(rng.uniform(math.log(128), math.log(4096))))
        c["steps"] = rng.randint(30, 80)
    elif kind == "warm":
        c["n_si"] = int(math.exp(rng.uniform(math.log(256), math.log(8000))))
    elif kind == "lj":
        c.update(_reps(rng, 4, 2000, 1000000, 6))
        c["steps"] = max(20, min(100, 10 * int(4e6 / (4 * c["nx"] * c["ny"] * c["nz"]))))
    else:
        c["n_si"] = int(math.exp(rng.uniform(math.log(512), math.log(8000))))
        c["steps"] = 20
    return c


# --- inputs -----------------------------------------------------------------------

def _silicon(case, seed, temperature=600.0):
    """Diamond silicon with thermal displacements, a few vacancies and
    Maxwell-Boltzmann momenta."""
    s = st.diamond_si((case["nx"], case["ny"], case["nz"]), sigma=0.1, seed=seed)
    if case["vacancies"]:
        gone = np.random.default_rng(seed + 7).choice(len(s), case["vacancies"], replace=False)
        keep = np.setdiff1d(np.arange(len(s)), gone)
        s = st.Structure(["Si"] * len(keep), s.positions[keep], s.cell)
    return st.maxwell_boltzmann(s, temperature, seed + 1)


def _two(positions, seed, step=0.02):
    """The geometry and the next one: every atom moved by about `step` A."""
    rng = np.random.default_rng(seed + 3)
    return [positions, positions + rng.normal(0.0, step, positions.shape)]


def _silica(case, seed):
    s = st.amorphous_sio2(case["n_si"], 2.2, seed=seed)
    rng = np.random.default_rng(seed + 1)
    q = np.where(np.array(s.symbols) == "Si", rng.uniform(0.5, 2.2, len(s)),
                 rng.uniform(-1.3, -0.2, len(s)))
    return s, q


def _rocksalt(case, seed):
    return st.rocksalt((case["nx"], case["ny"], case["nz"]), sigma=0.08, seed=seed)


def _argon(case, seed):
    s = st.fcc((case["nx"], case["ny"], case["nz"]), a=5.26, sigma=0.05, seed=seed)
    return st.maxwell_boltzmann(s, 80.0, seed + 1)


def _amorphous_cells(case, seed, dmin=2.1):
    """Amorphous silicon cells (random addition, minimum separation dmin), all
    grown together from the seed; sizes and densities belong to the case."""
    rng = np.random.default_rng([case["cells"], case["nmin"], case["nmax"]])
    sizes = rng.integers(case["nmin"], case["nmax"] + 1, size=case["cells"])
    dens = rng.uniform(2.25, 2.35, size=case["cells"])
    box = (sizes * st.AMU_SI / st.AVOGADRO / dens * 1e24) ** (1.0 / 3.0)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(seed))
    m, tries = int(sizes.max()), 64
    want = torch.tensor(sizes, device=dev)
    edge = torch.tensor(box, device=dev)
    pos = torch.full((len(sizes), m, 3), 1e6, device=dev, dtype=torch.float64)
    count = torch.zeros(len(sizes), device=dev, dtype=torch.int64)
    lower = torch.ones(tries, tries, device=dev).tril(-1).bool()
    while bool((count < want).any()):
        new = torch.rand((len(sizes), tries, 3), generator=gen, device=dev,
                         dtype=torch.float64) * edge[:, None, None]
        top = int(count.max())

        def near(a, b):
            hit = 0.0
            for x in range(3):
                d = (a[:, :, None, x] - b[:, None, :, x]).float()
                e = edge.float()[:, None, None]
                d = d - e * torch.round(d / e)
                hit = hit + d * d
            return hit < (dmin + 1e-4) ** 2

        ok = ~near(new, new).logical_and(lower).any(2)
        if top:
            there = torch.arange(top, device=dev)[None, :] < count[:, None]
            ok &= ~near(new, pos[:, :top]).logical_and(there[:, None, :]).any(2)
        slot = count[:, None] + ok.cumsum(1) - 1
        ok &= slot < want[:, None]
        c, t = torch.nonzero(ok, as_tuple=True)
        pos[c, slot[c, t]] = new[c, t]
        count += ok.sum(1)
    pos = pos.cpu().numpy()
    return [st.Structure(["Si"] * n, pos[k, :n], np.diag([box[k]] * 3))
            for k, n in enumerate(sizes)]


def _kcells(cell, kc):
    rec = 2.0 * np.pi * np.linalg.inv(cell).T
    vol = rec[0] @ np.cross(rec[1], rec[2])
    return [int(kc * np.linalg.norm(np.cross(rec[(a + 1) % 3], rec[(a + 2) % 3])) / vol + 0.5)
            for a in range(3)]


def _system(s, species, potentials, charges=None, radius=0.0, ewald=None, capacity=None):
    """An engine holding the structure, its model and its neighbor lists."""
    from pysic_amd.engine import Engine
    from pysic_amd.interactions import build_descriptors
    pd, bd, _ = build_descriptors(potentials, {x: k for k, x in enumerate(species)})
    eng = Engine(0)
    eng.create_atoms(np.array([species.index(x) for x in s.symbols], np.int32), s.positions,
                     masses=s.masses, charges=charges, momenta=s.momenta)
    eng.create_cell(s.cell, s.pbc)
    eng.set_potentials(pd)
    eng.set_bond_order_factors(bd)
    if ewald:
        eng.set_ewald(ewald["rc"], ewald["kc"], _kcells(s.cell, ewald["kc"]), ewald["sigma"],
                      ewald["eps"])
    else:
        eng.ewald_off()
    if capacity:
        eng.set_neighbor_capacity(capacity)
    eng.generate_neighbor_lists(np.full(len(s), radius))
    return eng


def prepare(case, seed):
    kind = case["kind"]
    out = {"case": case}
    if kind == "calc":
        from pysic_amd import Pysic, tersoff_si
        s = _silicon(case, seed)
        out["steps"] = []
        for p in _two(s.positions, seed):
            t = s.copy()
            t.set_positions(p)
            out["steps"].append(t)
        out["calc"] = Pysic(potentials=tersoff_si())
    elif kind in ("eval", "md"):
        from pysic_amd.interactions import tersoff_si
        s = _silicon(case, seed)
        out["eng"] = _system(s, ["Si"], tersoff_si(), radius=LIST_SI)
        out["n"] = len(s)
        out["positions"] = _two(s.positions, seed)
    elif kind == "batch":
        from pysic_amd.batch import BatchedCells
        from pysic_amd.interactions import tersoff_si
        out["batch"] = BatchedCells(_amorphous_cells(case, seed), tersoff_si())
    elif kind == "ewald":
        s = _rocksalt(case, seed)
        out["eng"] = _system(s, ["Cl", "Na"], [], charges=s.charges, radius=EWALD["rc"] + 0.5,
                             ewald=EWALD)
        out["positions"] = _two(s.positions, seed)
    elif kind in ("relax", "warm"):
        import os

        import pysic_amd
        from pysic_amd.learned import ChargePredictor, EEMSystem
        s, _ = _silica(case, seed)
        out["system"] = EEMSystem(0).load(s)
        out["zero"] = np.zeros(len(s))
        if kind == "warm":
            out["predictor"] = ChargePredictor.load(
                os.path.join(os.path.dirname(pysic_amd.__file__), "data", "sio2_eem_mlp.npz"), 0)
    elif kind == "lj":
        from pysic_amd.interactions import lj_argon
        s = _argon(case, seed)
        out["eng"] = _system(s, ["Ar"], lj_argon(cutoff=LJ_RC), radius=LJ_RC + LJ_SKIN,
                             capacity=112)
    elif kind == "comb":
        from pysic_amd.interactions import comb_sio2
        s, q = _silica(case, seed)
        st.maxwell_boltzmann(s, 300.0, seed + 2)
        out["eng"] = _system(s, ["O", "Si"], comb_sio2(), charges=q, radius=LIST_COMB)
        out["start"] = (s.positions, s.momenta)
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "calc":
        calc, out = state["calc"], []
        for s in state["steps"]:
            out.append((calc.get_potential_energy(s), calc.get_forces(s), calc.get_stress(s)))
        return out
    if kind == "eval":
        eng, out = state["eng"], []
        for p in state["positions"]:
            eng.update_coordinates(p)
            eng.generate_neighbor_lists(np.full(state["n"], LIST_SI))
            out.append((eng.energy(),) + eng.forces())
        return out
    if kind == "md":
        state["eng"].md_run(case["steps"], st.ASE_FS, rebuild=1)
        return state["eng"].state()
    if kind == "batch":
        state["batch"].evaluate(use_graph=True)
        return state["batch"].results()
    if kind == "ewald":
        eng, out = state["eng"], []
        for p in state["positions"]:
            eng.update_coordinates(p)
            out.append((eng.energy(),) + eng.forces())
        return out
    if kind == "relax":
        from pysic_amd.learned import TRAIN_RELAX
        sysm, n = state["system"], len(state["zero"])
        p = _relax_settings(n, TRAIN_RELAX)
        return sysm.eng.relax_charges(state["zero"], state["zero"], case["steps"], p["timestep"],
                                      p["inertia"], p["friction"], 1e-10)[:2]
    if kind == "warm":
        sysm = state["system"]
        q0 = state["predictor"].warm_start(sysm.eng)
        return sysm.relax(q0, 1e-6)[0]
    if kind == "lj":
        state["eng"].md_run(case["steps"], 2.0 * st.ASE_FS, rebuild=10)
        return state["eng"].state()
    # comb: every run starts from the prepared configuration
    eng = state["eng"]
    eng.update_coordinates(*state["start"])
    eng.md_run(case["steps"], 0.5 * st.ASE_FS, rebuild=1)
    return eng.state()


def _relax_settings(n, train):
    """The time step stable for the box: 0.1 for the 768-atom training cells,
    falling as one over the edge (the stiffest charge mode grows as its
    square) to 0.03 at 24,576 atoms."""
    return dict(train, timestep=min(0.1, 0.095 * (768.0 / n) ** (1.0 / 3.0)))


# --- work and tolerance ---------------------------------------------------------

def _atoms(case):
    kind = case["kind"]
    if kind in ("calc", "eval", "md"):
        return 8 * case["nx"] * case["ny"] * case["nz"] - case["vacancies"]
    if kind == "ewald":
        return 8 * case["nx"] * case["ny"] * case["nz"]
    if kind == "lj":
        return 4 * case["nx"] * case["ny"] * case["nz"]
    if kind == "batch":
        return case["cells"] * (case["nmin"] + case["nmax"]) // 2
    return 3 * case["n_si"]


def _reciprocal(n, edges):
    """(k-vectors of the half space, flops of one reciprocal pass): the
    direct sum's 8 per ion and k-vector, or, where less, a transform over a
    mesh of 8 points per k-vector and 1000 flops per ion to meet it."""
    kc = EWALD["kc"]
    nk = edges[0] * edges[1] * edges[2] * kc ** 3 / (12.0 * math.pi ** 2)
    mesh = 16.0 * nk
    return nk, min(8.0 * n * nk, 1000.0 * n + 2.5 * mesh * math.log2(max(mesh, 2.0)))


def work(case):
    kind, n = case["kind"], _atoms(case)
    if kind in ("calc", "eval"):     # positions in, forces out, twice
        return {"bytes": 2 * 48.0 * n, "flops": 2 * 2000.0 * n}
    if kind == "md":                 # positions and momenta in and out per step
        return {"bytes": 96.0 * n * case["steps"], "flops": 1000.0 * n * case["steps"]}
    if kind == "batch":
        return {"bytes": 48.0 * n, "flops": 3000.0 * n}
    if kind == "ewald":
        _, rec = _reciprocal(n, [5.64 * case[a] for a in ("nx", "ny", "nz")])
        pairs = 0.5 * n * (n / (n / 8.0 * 5.64 ** 3)) * 4.19 * EWALD["rc"] ** 3
        return {"bytes": 2 * 56.0 * n, "flops": 2 * (2 * rec + 60.0 * pairs)}
    if kind in ("relax", "warm"):
        edge = (n * 15.02) ** (1.0 / 3.0)
        _, rec = _reciprocal(n, [edge] * 3)
        steps = case["steps"] if kind == "relax" else 17
        return {"bytes": 16.0 * n * steps,
                "flops": steps * (2 * rec + 40.0 * 0.5 * n * 279.0)}
    if kind == "lj":
        return {"bytes": 96.0 * n * case["steps"], "flops": 30.0 * 33.0 * n * case["steps"]}
    return {"bytes": 96.0 * n * case["steps"], "flops": 5000.0 * n * case["steps"]}


def tolerance(case):
    """About four times what the path is seen to differ from exact(): 32-bit
    three-body terms in every Tersoff force (64 bits elsewhere), 64-bit sums
    in the others, with what dynamics and relaxation make of the rounding;
    the learned start ends at the relaxation's own 1e-6 eV/e."""
    return {"calc": {"rel": 1e-6, "max": 4e-5}, "eval": {"rel": 1e-6, "max": 4e-5},
            "batch": {"rel": 1e-6, "max": 4e-5}, "md": {"rel": 2e-5, "max": 1e-3},
            "ewald": {"rel": 1e-12, "max": 4e-11}, "relax": {"rel": 1e-9, "max": 4e-8},
            "warm": {"rel": 4e-8, "max": 1e-6}, "lj": {"rel": 1e-12, "max": 4e-11},
            "comb": {"rel": 3e-11, "max": 1e-9}}[case["kind"]]


# --- the models in plain torch, 64 bits -----------------------------------------------

def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _lists(pos, edges, rc):
    """Padded neighbor lists of a periodic orthorhombic box: (j, shift, mask)
    of shape [n, m(, 3)], r_j + shift - r_i within rc."""
    n, dev = len(pos), pos.device
    nb = [max(1, int(e // rc)) for e in edges]
    rows, cols, shifts = [], [], []
    if min(nb) < 3:
        reach = [int(math.ceil(rc / e)) for e in edges]
        home = torch.floor(pos / edges)
        p = pos - home * edges
        step = max(1, int(4e7 // n))
        for o in itertools.product(*(range(-r, r + 1) for r in reach)):
            sh = torch.tensor(o, device=dev, dtype=torch.float64) * edges
            for a in range(0, n, step):
                d2 = sum((p[None, :, c] + sh[c] - p[a:a + step, None, c]) ** 2 for c in range(3))
                hit = d2 < rc * rc
                if not any(o):
                    hit[torch.arange(len(hit), device=dev), torch.arange(a, a + len(hit),
                                                                        device=dev)] = False
                i, j = torch.nonzero(hit, as_tuple=True)
                i = i + a
                rows.append(i)
                cols.append(j)
                shifts.append(sh + (home[i] - home[j]) * edges)
    else:
        nbt = torch.tensor(nb, device=dev)
        home = torch.floor(pos / edges)
        p = pos - home * edges
        b = torch.minimum((p / edges * nbt).long(), nbt - 1)
        key = (b[:, 2] * nb[1] + b[:, 1]) * nb[0] + b[:, 0]
        order = torch.argsort(key, stable=True)
        total = nb[0] * nb[1] * nb[2]
        cnt = torch.bincount(key, minlength=total)
        first = cnt.cumsum(0) - cnt
        m = int(cnt.max())
        slots = torch.arange(m, device=dev)
        for o in itertools.product((-1, 0, 1), repeat=3):
            t = b + torch.tensor(o, device=dev)
            w = torch.div(t, nbt, rounding_mode="floor")
            t = t - w * nbt
            k = (t[:, 2] * nb[1] + t[:, 1]) * nb[0] + t[:, 0]
            for a in range(0, n, 1 << 20):
                kk = k[a:a + (1 << 20)]
                there = slots[None, :] < cnt[kk][:, None]
                j = order[torch.where(there, first[kk][:, None] + slots, 0)]
                sh = w[a:a + (1 << 20)].double() * edges
                d2 = sum((p[:, c][j] + sh[:, None, c] - p[a:a + (1 << 20), None, c]) ** 2
                         for c in range(3))
                i0 = torch.arange(a, a + len(kk), device=dev)
                hit = there & (d2 < rc * rc) & ~((j == i0[:, None]) & (not any(o)))
                i, s = torch.nonzero(hit, as_tuple=True)
                jj = j[i, s]
                rows.append(i0[i])
                cols.append(jj)
                shifts.append(sh[i] + (home[i0[i]] - home[jj]) * edges)
    i, j, s = torch.cat(rows), torch.cat(cols), torch.cat(shifts)
    o = torch.argsort(i, stable=True)
    i, j, s = i[o], j[o], s[o]
    cnt = torch.bincount(i, minlength=n)
    rank = torch.arange(len(i), device=dev) - (cnt.cumsum(0) - cnt)[i]
    m = max(1, int(cnt.max()))
    J = torch.zeros((n, m), dtype=torch.int64, device=dev)
    S = torch.zeros((n, m, 3), dtype=torch.float64, device=dev)
    M = torch.zeros((n, m), dtype=torch.bool, device=dev)
    J[i, rank], S[i, rank], M[i, rank] = j, s, True
    return J, S, M


def _fc(r, hard, soft):
    w = 0.5 * (1.0 + torch.cos(math.pi * (r - soft) / (hard - soft)))
    return torch.where(r < soft, torch.ones_like(r), torch.where(r > hard, torch.zeros_like(r), w))


def _compress(pos, lists, rc):
    """The entries of the lists within rc now, padded again: (j, shift, mask)."""
    J, S, M = lists
    with torch.no_grad():
        d = pos[J] + S - pos[:, None, :]
        M = M & ((d * d).sum(2) < rc * rc)
        m = max(1, int(M.sum(1).max()))
        o = torch.argsort(M.to(torch.int8), dim=1, descending=True, stable=True)[:, :m]
    return J.gather(1, o), S.gather(1, o[..., None].expand(-1, -1, 3)), M.gather(1, o)


def _vectors(pos, lists):
    J, S, M = lists
    d = pos[J] + S - pos[:, None, :]
    d = torch.where(M[..., None], d, torch.ones_like(d))
    return J, d, torch.sqrt((d * d).sum(2)), M


def _tersoff(pos, lists):
    """Tersoff silicon: energy per atom."""
    P = dict(A=1830.8, l1=2.4799, B=471.18, l2=1.7322, beta=1.1e-6, eta=0.78734, c=100390.0,
             d=16.217, h=-0.59825, cut=3.0, soft=2.7)
    J, d, r, M = _vectors(pos, _compress(pos, lists, P["cut"]))
    f = torch.where(M, _fc(r, P["cut"], P["soft"]), torch.zeros_like(r))
    u = d / r[..., None]
    cs = u @ u.transpose(1, 2)
    cc, dd = P["c"] ** 2, P["d"] ** 2
    t2 = (P["h"] - cs) ** 2
    g = 1.0 + cc * t2 / (dd * (dd + t2))
    g = g * (1.0 - torch.eye(g.shape[1], device=g.device, dtype=g.dtype))
    zeta = (g * f[:, None, :]).sum(2)
    safe = torch.where(zeta > 0, zeta, torch.ones_like(zeta))
    b = torch.where(zeta > 0, (1.0 + (P["beta"] * safe) ** P["eta"]) ** (-0.5 / P["eta"]),
                    torch.ones_like(zeta))
    e = f * (P["A"] * torch.exp(-P["l1"] * r) - P["B"] * b * torch.exp(-P["l2"] * r))
    return 0.5 * e.sum(1), (J, M, r)


COMB = {"Si": dict(rmax=-1.658949, rmin=1.651725, qmax=4.0, qmin=-4.0, alpha=1.7322, a=1.0,
                   b=-9.5367431640625e-07, q=0.0, n=10.0, B=471.18, A=1830.8, lam=2.4799,
                   cut=3.0, margin=0.2),
        "O": dict(rmax=-0.00112, rmin=0.00148, qmax=5.5046, qmin=-1.8349, alpha=2.68, a=1.00098,
                  b=-2.26e-6, q=1.83485, n=10.0, B=260.8931, A=3326.699, lam=5.36, cut=3.0,
                  margin=0.4)}
COMB_BOND = {"Si": dict(beta=1.0999e-6, eta=0.78734, mu=3, a=1.7322, c=100390.0, d=16.218,
                        h=-0.59826),
             "O": dict(beta=2.0, eta=1.0, mu=1, a=2.68, c=6.6, d=1.0, h=-0.229)}


def _comb(pos, lists, si, q):
    """COMB's local silica terms (si: which atoms are silicon): energy per atom."""
    J, d, r, M = _vectors(pos, _compress(pos, lists, 3.05))
    dev = pos.device

    def pick(a, b, like):
        return torch.where(like, torch.tensor(float(a), dtype=torch.float64, device=dev),
                           torch.tensor(float(b), dtype=torch.float64, device=dev))

    ci, cj = si[:, None].expand_as(J), si[J]
    same, mixed = ci == cj, ci != cj
    cut = pick(3.0, 3.05, same)
    soft = torch.where(mixed, pick(2.55, 2.55, same), pick(2.8, 2.6, ci))
    f = torch.where(M, 0.5 * (1.0 + torch.cos(math.pi * (r - soft) / (cut - soft))),
                    torch.zeros_like(r))
    f = torch.where(M & (r < soft), torch.ones_like(r), f)
    f = torch.where(r > cut, torch.zeros_like(r), f)

    def screen(name):
        p = COMB[name]
        eta = math.log(p["rmax"] / (p["rmax"] - p["rmin"])) / math.log(
            p["qmax"] / (p["qmax"] - p["qmin"]))
        beta = (p["rmin"] - p["rmax"]) ** (1.0 / eta) / (p["qmax"] - p["qmin"])
        return (p["rmax"] + (beta * (p["qmax"] - q)).abs() ** eta,
                (p["a"] + p["b"] * (q - p["q"]).abs() ** p["n"]).clamp(min=0.0))

    (Ds, fs), (Do, fo) = screen("Si"), screen("O")
    D, fa = torch.where(si, Ds, Do), torch.where(si, fs, fo)
    S, O = COMB["Si"], COMB["O"]

    def per(key, how):
        a, b = S[key], O[key]
        mid = math.sqrt(a * b) if how == "geo" else 0.5 * (a + b)
        return torch.where(mixed, pick(mid, mid, ci), pick(a, b, ci))

    al, lam = pick(S["alpha"], O["alpha"], si), pick(S["lam"], O["lam"], si)
    sa = torch.exp(0.5 * ((al * D)[:, None] + (al * D)[J]))
    sr = torch.exp(0.5 * ((lam * D)[:, None] + (lam * D)[J]))
    absf = torch.sqrt(fa[:, None] * fa[J])
    att = -per("B", "geo") * sa * absf * torch.exp(-per("alpha", "mean") * r)
    rep = per("A", "geo") * sr * torch.exp(-per("lam", "mean") * r)
    # the lone charge_abs term of oxygen pairs, cutoff 3.0 with margin 0.5
    oo = (~ci) & (~cj) & M
    lone = torch.where(oo, absf * _fc(r, 3.0, 2.5), torch.zeros_like(r))
    # bond order: zeta over the third neighbors k of i, partner j
    u = d / r[..., None]
    cs = u @ u.transpose(1, 2)
    ti = ci[:, :1, None]
    pj, tk = cj[:, :, None], cj[:, None, :]
    mono = (ti == pj) & (pj == tk)
    tcut = torch.where(mono, pick(3.0, 3.0, mono), pick(3.05, 3.05, mono))
    tsoft = torch.where(mono, pick(2.8, 2.6, ti), pick(2.55, 2.55, mono))
    rk = r[:, None, :].expand_as(tcut)
    fk = 0.5 * (1.0 + torch.cos(math.pi * (rk - tsoft) / (tcut - tsoft)))
    fk = torch.where(rk < tsoft, torch.ones_like(fk), fk)
    fk = torch.where(rk > tcut, torch.zeros_like(fk), fk)
    eye = torch.eye(J.shape[1], device=dev, dtype=torch.bool)
    valid = M[:, :, None] & M[:, None, :] & ~eye
    bs, bo = COMB_BOND["Si"], COMB_BOND["O"]
    a_mid = 0.5 * (bs["a"] + bo["a"])
    a = torch.where(mixed, pick(a_mid, a_mid, ci), pick(bs["a"], bo["a"], ci))[:, :, None]
    x = a * (r[:, :, None] - r[:, None, :])
    x = torch.where(valid, x, torch.zeros_like(x))
    ex = torch.exp(torch.where(ti, x ** 3, x))
    cc, dd, h = pick(bs["c"] ** 2, bo["c"] ** 2, ti), pick(bs["d"] ** 2, bo["d"] ** 2, ti), \
        pick(bs["h"], bo["h"], ti)
    t2 = (h - cs) ** 2
    z = torch.where(valid, fk * ex * (1.0 + cc * t2 / (dd * (dd + t2))), torch.zeros_like(ex))
    zeta = z.sum(2)
    beta, eta = pick(bs["beta"], bo["beta"], ci), pick(bs["eta"], bo["eta"], ci)
    safe = torch.where(zeta > 0, zeta, torch.ones_like(zeta))
    b = torch.where(zeta > 0, (1.0 + (beta * safe) ** eta) ** (-0.5 / eta), torch.ones_like(zeta))
    e = 0.5 * torch.where(M, f * (att * b + rep) + lone, torch.zeros_like(r)).sum(1)
    # angles Si-O-Si and O-Si-O, every unordered pair of legs once
    leg = torch.where(M & mixed, _fc(r, 3.05, 2.55), torch.zeros_like(r))
    c0 = pick(math.cos(1.910611932), math.cos(2.508561734), ti)
    k0 = pick(0.3122, 2.6, ti)
    ang = k0 * (cs - c0) ** 2 * leg[:, :, None] * leg[:, None, :]
    return e + torch.where(valid, 0.5 * ang, torch.zeros_like(ang)).sum((1, 2))


def _grad(energy, pos):
    """(energy, forces, virial sum r f over list entries) by differentiation."""
    p = pos.clone().requires_grad_(True)
    e = energy(p).sum()
    (g,) = torch.autograd.grad(e, p)
    return e.detach(), -g


def _verlet(pos, mom, mass, dt, steps, forces):
    f = forces(pos)
    for _ in range(steps):
        mom = mom + 0.5 * dt * f
        pos = pos + dt * mom / mass
        f = forces(pos)
        mom = mom + 0.5 * dt * f
    return pos, mom


def _following(edges, rc, skin=1.0):
    """Lists of radius rc + skin for positions that move, built again when an
    atom has moved by half the skin."""
    held = {}

    def lists(pos):
        if not held or float((pos - held["at"]).norm(dim=1).max()) > 0.49 * skin:
            held["at"], held["lists"] = pos.clone(), _lists(pos, edges, rc + skin)
        return held["lists"]
    return lists


def _tersoff_efw(pos, edges):
    """Energy, forces and W = -sum_ij r_ij (x) dU_i/dr_ij (xx yy zz yz xz xy)."""
    lists = _compress(pos, _lists(pos, edges, 3.0), 3.0)
    strain = torch.zeros((3, 3), dtype=torch.float64, device=pos.device, requires_grad=True)
    p = pos.clone().requires_grad_(True)
    one = torch.eye(3, dtype=torch.float64, device=pos.device)
    J, S, M = lists
    e, _ = _tersoff(p @ (one + strain), (J, S @ (one + strain), M))
    f, w = torch.autograd.grad(e.sum(), (p, strain))
    w = -w   # the engine's virial: sum of r (x) f
    w = torch.stack([w[0, 0], w[1, 1], w[2, 2], w[1, 2], w[0, 2], w[0, 1]])
    return e.sum().detach(), -f, w


def _lj_forces(lists):
    eps, sig = 4 * 119.8 * 8.617333262e-5, 3.405

    def forces(pos):
        J, S, M = lists(pos)
        out = torch.empty_like(pos)
        for a in range(0, len(pos), 1 << 18):
            sl = slice(a, a + (1 << 18))
            d = pos[J[sl]] + S[sl] - pos[sl, None, :]
            r2 = (d * d).sum(2)
            on = M[sl] & (r2 < LJ_RC * LJ_RC)
            i2 = 1.0 / torch.where(on, r2, torch.ones_like(r2))
            s6 = (sig * sig * i2) ** 3
            g = torch.where(on, eps * (12.0 * s6 * s6 - 6.0 * s6) * i2, torch.zeros_like(r2))
            out[sl] = -(g[..., None] * d).sum(1)
        return out
    return forces


class _Ewald:
    """Ewald sums of a periodic orthorhombic box of point charges."""

    def __init__(self, pos, edges, lists=None):
        self.pos, self.edges, self.n = pos, edges, len(pos)
        self.K = _kcells(np.diag(edges.cpu().numpy()), EWALD["kc"])
        self.vol = float(edges.prod())
        self.c4 = 1.0 / (4.0 * math.pi * EWALD["eps"])
        self.c2 = 1.0 / (2.0 * self.vol * EWALD["eps"])
        self.lists = _lists(pos, edges, EWALD["rc"]) if lists is None else lists
        u = pos / edges
        self.e = []
        for a in range(3):
            k = torch.arange(0 if a == 2 else -self.K[a], self.K[a] + 1, device=pos.device,
                             dtype=torch.float64)
            x = u[:, a:a + 1] * k
            x = 2.0 * math.pi * (x - torch.round(x))
            self.e.append(torch.complex(torch.cos(x), torch.sin(x)))
        b = 2.0 * math.pi / edges
        g = [torch.arange(0 if a == 2 else -self.K[a], self.K[a] + 1, device=pos.device,
                          dtype=torch.float64) * b[a] for a in range(3)]
        self.g = g
        k2 = g[0][:, None, None] ** 2 + g[1][None, :, None] ** 2 + g[2][None, None, :] ** 2
        on = (k2 < EWALD["kc"] ** 2) & (k2 > 0)
        k2s = torch.where(on, k2, torch.ones_like(k2))
        w = torch.full_like(k2, 2.0)
        w[:, :, 0] = 1.0
        self.coef = torch.where(on, self.c2 * w * torch.exp(-EWALD["sigma"] ** 2 * k2s / 2) / k2s,
                                torch.zeros_like(k2))

    def structure(self, q):
        e1, e2, e3 = self.e
        return torch.stack([(((q * e1[:, a])[:, None]) * e2).t().contiguous() @ e3
                            for a in range(e1.shape[1])])

    def at_atoms(self, z):
        """sum_k z(k) conj(e^{ikr}) at every atom, for each array of z."""
        e1, e2, e3 = self.e
        out = [torch.zeros(self.n, dtype=e1.dtype, device=e1.device) for _ in z]
        for a in range(e1.shape[1]):
            t = e1[:, a:a + 1] * e2
            for y, o in zip(z, out):
                o += ((e3.conj() @ y[a].t().contiguous()) * t.conj()).sum(1)
        return out

    def real(self, q, what):
        J, S, M = self.lists
        out = []
        s2 = 1.0 / (math.sqrt(2.0) * EWALD["sigma"])
        for a in range(0, self.n, 1 << 16):
            sl = slice(a, a + (1 << 16))
            d = self.pos[J[sl]] + S[sl] - self.pos[sl, None, :]
            d = torch.where(M[sl][..., None], d, torch.ones_like(d))
            r = torch.sqrt((d * d).sum(2))
            on = M[sl] & (r < EWALD["rc"])
            er = torch.erfc(r * s2) / r
            if what == "chi":
                out.append(-self.c4 * torch.where(on, q[J[sl]] * er, torch.zeros_like(r)).sum(1))
                continue
            qq = self.c4 * q[sl][:, None] * q[J[sl]]
            e = torch.where(on, 0.5 * qq * er, torch.zeros_like(r))
            g = (er / r + math.sqrt(2.0 / math.pi) / EWALD["sigma"] *
                 torch.exp(-(r * s2) ** 2) / r) / r
            f = torch.where(on, -qq * g, torch.zeros_like(r))[..., None] * d
            # pair virial: half of each end's
            w = -0.5 * torch.stack([(d[..., x] * f[..., y]).sum() for x, y in
                                    ((0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1))])
            out.append((e.sum(), f.sum(1), w))
        if what == "chi":
            return torch.cat(out)
        return (sum(o[0] for o in out), torch.cat([o[1] for o in out]), sum(o[2] for o in out))

    def energy_forces(self, q):
        e, f, w = self.real(q, "forces")
        s = self.structure(q)
        e = e + (self.coef * (s.real ** 2 + s.imag ** 2)).sum()
        e = e - self.c4 / (math.sqrt(2.0 * math.pi) * EWALD["sigma"]) * (q * q).sum()
        e = e - q.sum() ** 2 * 0.5 * self.c2 * EWALD["sigma"] ** 2
        z = self.coef * s
        g = self.g
        t = self.at_atoms([z * g[0][:, None, None], z * g[1][None, :, None],
                           z * g[2][None, None, :]])
        # F = -dE/dr with d|S|^2/dr_i = 2 q k Im(S e^{-ikr})
        fr = torch.stack([-2.0 * q * x.imag for x in t], dim=1)
        p = self.pos
        w = w + torch.stack([(p[:, x] * fr[:, y]).sum() for x, y in
                             ((0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1))])
        return e, f + fr, w

    def chi(self, q):
        c = self.real_matrix @ q if hasattr(self, "real_matrix") else self.real(q, "chi")
        c = c + 2.0 * q * self.c4 / (math.sqrt(2.0 * math.pi) * EWALD["sigma"])
        c = c + self.c2 * EWALD["sigma"] ** 2 * q.sum()
        (t,) = self.at_atoms([self.coef * self.structure(q)])
        return c - 2.0 * t.real


EEM = {"Si": (4.77, 16.0), "O": (8.74, 20.0)}


def _host(v):
    return v.cpu().numpy()


def exact(case, seed):
    kind, dev = case["kind"], _dev()

    def t(x):
        return torch.tensor(np.asarray(x, dtype=np.float64), device=dev)

    if kind in ("calc", "eval"):
        s = _silicon(case, seed)
        edges, out = t(np.diag(s.cell)), []
        for p in _two(s.positions, seed):
            e, f, w = _tersoff_efw(t(p), edges)
            e, f, w = float(e), _host(f), _host(w)
            if kind == "calc":
                v = s.momenta / s.masses[:, None]
                kin = np.array([(s.momenta[:, a] * v[:, b]).sum() for a, b in
                                ((0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1))])
                w = -(kin + w) / s.get_volume()
            out.append((e, f, w))
        return out
    if kind == "batch":
        E, W, F = [], [], []
        for s in _amorphous_cells(case, seed):
            e, f, w = _tersoff_efw(t(s.positions), t(np.diag(s.cell)))
            E.append(float(e))
            W.append(_host(w))
            F.append(_host(f))
        return np.array(E), np.array(W), np.concatenate(F)
    if kind == "md":
        s = _silicon(case, seed)
        lists = _following(t(np.diag(s.cell)), 3.0)
        x, p = _verlet(t(s.positions), t(s.momenta), t(s.masses)[:, None], st.ASE_FS,
                       case["steps"],
                       lambda r: _grad(lambda y: _tersoff(y, lists(r))[0], r)[1])
        return _host(x), _host(p)
    if kind == "lj":
        s = _argon(case, seed)
        x, p = _verlet(t(s.positions), t(s.momenta), t(s.masses)[:, None], 2.0 * st.ASE_FS,
                       case["steps"], _lj_forces(_following(t(np.diag(s.cell)), LJ_RC)))
        return _host(x), _host(p)
    if kind == "comb":
        s, q = _silica(case, seed)
        st.maxwell_boltzmann(s, 300.0, seed + 2)
        lists = _following(t(np.diag(s.cell)), 3.05)
        si = torch.tensor([x == "Si" for x in s.symbols], device=dev)
        x, p = _verlet(t(s.positions), t(s.momenta), t(s.masses)[:, None], 0.5 * st.ASE_FS,
                       case["steps"],
                       lambda r: _grad(lambda y: _comb(y, lists(r), si, t(q)), r)[1])
        return _host(x), _host(p)
    if kind == "ewald":
        s = _rocksalt(case, seed)
        q, edges, out = t(s.charges), t(np.diag(s.cell)), []
        for p in _two(s.positions, seed):
            e, f, w = _Ewald(t(p), edges).energy_forces(q)
            out.append((float(e), _host(f), _host(w)))
        return out
    # charges: damped dynamics, or the equilibrium by conjugate gradients
    s, _ = _silica(case, seed)
    sums = _Ewald(t(s.positions), t(np.diag(s.cell)))
    chi0 = t([EEM[x][0] for x in s.symbols])
    hard = t([EEM[x][1] for x in s.symbols])

    def chi(q):
        return sums.chi(q) - chi0 - hard * q

    n = len(s)
    if kind == "relax":
        from pysic_amd.learned import TRAIN_RELAX
        p = _relax_settings(n, TRAIN_RELAX)
        dt, mq, fr = p["timestep"], p["inertia"], p["friction"]
        q, v = torch.zeros(n, dtype=torch.float64, device=dev), 0.0
        f = chi(q)
        f = f - f.mean()
        for _ in range(case["steps"]):
            q = q + v * dt + (f - fr * v) / mq * dt * dt
            v = (1.0 - 0.5 * fr * dt) * v + 0.5 * f / mq * dt
            f = chi(q)
            f = f - f.mean()
            v = (v + 0.5 * f / mq * dt) / (1.0 + 0.5 * fr * dt)
        return _host(q), _host(v)
    base = chi(torch.zeros(n, dtype=torch.float64, device=dev))

    def hess(x):     # -(chi(x) - chi(0)) on the space of zero sum
        y = base - chi(x)
        return y - y.mean()

    q = torch.zeros(n, dtype=torch.float64, device=dev)
    r = base - base.mean()
    d, rr = r.clone(), float(r @ r)
    for _ in range(200):
        h = hess(d)
        a = rr / float(d @ h)
        q, r = q + a * d, r - a * h
        new = float(r @ r)
        if new < 1e-22 * n:
            break
        d, rr = r + new / rr * d, new
    return _host(q)
