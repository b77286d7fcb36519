"""The work that users of the engine have it do, as cases that can be timed
and checked.

Every case is one pass through the Python host (`molsim_amd.engine`) as a
simulation program drives it: molecular and Brownian dynamics runs, single
force evaluations on the host's positions, batched replicas, Monte Carlo
sweeps, the parameter adjoint and the force-matching gradient.  `listed()`
names twelve of them, `draw()` gives more of the same ranges, `exact()` the
results in 64-bit torch without the engine.

Units are MOLSIM's: A, ps, g/mol, kJ/mol.

A mixed-precision engine evaluates forces, energies and gradients in FP32
arithmetic, so a program that chose it keeps those in 32 bits (`_kept`);
positions are FP64 state on both paths.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from molsim_amd import engine as E

KT = 2.4777                 # kJ/mol at 298 K
RGAS = 8.314472
EFP = E.epsi0_four_pi() / 78.4
FFAC = E.force_unit_fac()
DT_MD, DT_BD = 0.002, 0.005
SIGMA = 4.0
LJCUT = 2.0 ** float(np.float32(1.0 / 6.0))
NKNOT, KNOT_LO = 64, 3.5
SPECIES = {                 # charges and masses per type; composition below
    "salt": ([1.0, -1.0], [23.0, 35.4]),
    "salts": ([1.0, 2.0, -1.0], [22.99, 40.08, 35.45]),
    "chains": ([-1.0, 1.0, -1.0], [30.0, 23.0, 35.4]),
}
CHAIN_LEN, BOND_LEN = 50, 5.0
BOND = (0.4 * KT, 2, BOND_LEN)            # namelist k, p, eq
ANGLE = (0.002, 2, 180.0)                 # namelist k (per degree^2), p, eq


# ------------------------------------------------------------------ cases
def listed():
    return [
        # the smallest system in daily use: 1000 ions in a 50 A box with the
        # standard Ewald sum; a step is bound by launches and latency
        dict(name="md_1k_std", kind="md", prec="mixed", species="salt", n=1000, density=8.0e-3,
             aspect=1.0, rc=15.0, ewald="std", ncut=8, order=0, mesh=0, meshz=0, steps=50),
        # polyelectrolyte solution: 40 chains of 50 beads with bonds and
        # angles, counterions and salt
        dict(name="md_6k_chains", kind="md", prec="mixed", species="chains", n=6000,
             density=3.472e-3, aspect=1.0, rc=18.0, ewald="spm", ncut=0, order=4, mesh=64,
             meshz=64, steps=50),
        # the benchmark's electrolyte on the mixed path and on the FP64 path
        dict(name="md_200k", kind="md", prec="mixed", species="salts", n=200000,
             density=7.527e-4, aspect=1.0, rc=12.0, ewald="spm", ncut=0, order=6, mesh=128,
             meshz=128, steps=50),
        dict(name="md_200k_fp64", kind="md", prec="fp64", species="salts", n=200000,
             density=7.527e-4, aspect=1.0, rc=12.0, ewald="spm", ncut=0, order=6, mesh=128,
             meshz=128, steps=25),
        # the largest runs: a million ions, a mesh that is no power of two
        dict(name="md_1m", kind="md", prec="mixed", species="salts", n=1000035,
             density=7.527e-4, aspect=1.0, rc=12.0, ewald="spm", ncut=0, order=6, mesh=240,
             meshz=240, steps=10),
        # a host program with its own integrator: positions up, UTotal with
        # the cell-list pair semantics, forces and energies back, each step
        dict(name="utotal_31k_fp64", kind="utotal", prec="fp64", species="salts", n=31415,
             density=7.527e-4, aspect=1.5, rc=12.0, ewald="spm", ncut=0, order=5, mesh=54,
             meshz=80, nlist="cell", move=0.02),
        # independent snapshots evaluated again: every call rebuilds the list
        dict(name="snapshots_100k", kind="utotal", prec="mixed", species="salts", n=100000,
             density=7.527e-4, aspect=1.0, rc=12.0, ewald="spm", ncut=0, order=4, mesh=120,
             meshz=120, nlist="vlist", move=-1.0),
        # one Brownian dynamics run of an odd-sized system
        dict(name="bd_20k", kind="bd", prec="mixed", species="salts", n=20005, density=1.2e-3,
             aspect=1.0, rc=14.0, ewald="spm", ncut=0, order=5, mesh=70, meshz=70, steps=50),
        # many small replicas (500 to 4000 ions) stepped together
        dict(name="bd_batch_96", kind="batch", prec="mixed", species="salt", n=4000, replicas=96,
             density=1.2e-3, aspect=1.0, rc=18.0, ewald="spm", ncut=0, order=4, mesh=36,
             meshz=36, steps=100),
        # a Monte Carlo sweep: trial moves, pair and reciprocal changes,
        # Metropolis, accepted moves kept
        dict(name="mc_50k", kind="mc", prec="fp64", species="salts", n=50000, density=7.527e-4,
             aspect=1.0, rc=12.0, ewald="spm", ncut=0, order=6, mesh=80, meshz=80, trials=64),
        # the parameter adjoint of one large polyelectrolyte frame
        dict(name="adjoint_66k", kind="adjoint", prec="mixed", species="chains", n=66000,
             density=3.472e-3, aspect=1.0, rc=18.0, ewald="spm", ncut=0, order=4, mesh=96,
             meshz=96),
        # force matching: loss and gradient over frames of that system
        dict(name="fm_66k", kind="fm", prec="mixed", species="chains", n=66000,
             density=3.472e-3, aspect=1.0, rc=18.0, ewald="spm", ncut=0, order=4, mesh=96,
             meshz=96, frames=4),
    ]


# meshes the engine takes whose bricks stay small: even, primes up to 7
_MESHES = [16, 18, 20, 24, 28, 30, 32, 36, 40, 42, 48, 50, 54, 56, 60, 64, 70, 72, 80, 84, 90,
           96, 100, 108, 112, 120, 126, 128, 140, 144, 150, 160]


def _mesh_for(length, spacing, order):
    want = length / spacing
    return min((m for m in _MESHES if m >= order), key=lambda m: abs(math.log(m / want)))


def draw(rng):
    """One more case: the kind as often as it is listed, sizes spread over
    their logarithm."""
    kind = rng.choice(["md", "md", "md", "utotal", "utotal", "bd", "batch", "mc", "adjoint",
                       "fm"])

    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    c = dict(kind=kind, prec=rng.choice(["mixed", "mixed", "fp64"]), aspect=1.0, ewald="spm",
             ncut=0, order=rng.choice([4, 4, 5, 6, 6, 8]))
    c["species"] = rng.choice(["salt", "salts", "salts", "chains"])
    c["density"] = round(math.exp(rng.uniform(math.log(3e-4), math.log(3.5e-3))), 6)
    c["rc"] = round(rng.uniform(10.0, 16.0), 2)
    if kind == "md":
        c["n"] = size(1000, 300000)
        c["steps"] = 50 if c["n"] < 50000 else 10
        c["aspect"] = rng.choice([1.0, 1.0, 1.4, 2.0])
        if c["n"] < 4000 and rng.random() < 0.5:
            c["ewald"], c["ncut"], c["order"] = "std", rng.randint(5, 10), 0
    elif kind == "utotal":
        c["n"] = size(2000, 200000)
        c["aspect"] = rng.choice([1.0, 1.3, 2.0])
        c["nlist"] = rng.choice(["vlist", "cell"])
        c["move"] = rng.choice([0.02, -1.0])
    elif kind == "bd":
        c["n"], c["steps"] = size(1000, 100000), 40
    elif kind == "batch":
        c.update(prec="mixed", species="salt", n=size(1000, 4000), replicas=rng.randint(8, 96),
                 steps=50, rc=round(rng.uniform(12.0, 20.0), 2), order=rng.choice([4, 5, 6]),
                 density=round(math.exp(rng.uniform(math.log(3e-4), math.log(1.2e-3))), 6))
    elif kind == "mc":
        c["n"], c["trials"] = size(2000, 100000), 48
        c["species"] = rng.choice(["salt", "salts"])
    else:
        c["n"], c["species"] = size(6000, 66000), "chains"
        c["density"], c["rc"] = 3.472e-3, round(rng.uniform(12.0, 18.0), 2)
        c["order"] = rng.choice([4, 5, 6])
        if kind == "fm":
            c["frames"] = rng.randint(1, 4)
    # neutral compositions: an even number of ions, a multiple of five,
    # whole chains with their counterions and salt
    unit = {"salt": 2, "salts": 5, "chains": 150}[c["species"]]
    c["n"] = max(unit, c["n"] // unit * unit)
    box = _box(c)
    c["rc"] = min(c["rc"], round(0.45 * float(box.min()), 2))
    spacing = c["rc"] / 3.0 * rng.uniform(0.8, 1.25) * (1.0 if c["order"] >= 6 else 0.7)
    c["mesh"] = _mesh_for(box[0], spacing, c["order"]) if c["ewald"] == "spm" else 0
    c["meshz"] = _mesh_for(box[2], spacing, c["order"]) if c["ewald"] == "spm" else 0
    return c


# ---------------------------------------------------------------- systems
def _box(case, n=None):
    lx = ((n or case["n"]) / case["density"] / case["aspect"]) ** (1.0 / 3.0)
    return np.array([lx, lx, lx * case["aspect"]])


def _types(case, n):
    """1-based types in order, and the chains (first, length)."""
    if case["species"] == "salt":
        return np.repeat([1, 2], [n // 2, n // 2]).astype(np.int32), []
    if case["species"] == "salts":
        k = n // 5
        return np.repeat([1, 2, 3], [k, k, 3 * k]).astype(np.int32), []
    # a third beads, half counterions and cations, the rest anions
    nchain = n // 150
    beads, salt = nchain * CHAIN_LEN, n // 6
    types = np.repeat([1, 2, 3], [beads, beads + salt, salt]).astype(np.int32)
    return types, [(1 + c * CHAIN_LEN, CHAIN_LEN) for c in range(nchain)]


def _sites(rng, box, nchain, nfree):
    """Distinct sites of a fine grid: self-avoiding walks of CHAIN_LEN steps
    for the chains, uniformly chosen sites for the free particles."""
    pitch = BOND_LEN if nchain else 4.6
    m = np.maximum(np.floor(box / pitch).astype(np.int64), 1)
    total = int(m.prod())
    used = np.zeros(total, bool)
    walk = np.zeros(nchain * CHAIN_LEN, np.int64)
    mx, my, mz = (int(v) for v in m)
    moves = ((1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1))
    order = rng.integers(0, 720, (nchain * 60 + 1000) * 2)
    perms = [p for p in _permutations(6)]
    k = 0
    for c in range(nchain):
        while True:
            start = int(rng.integers(total))
            if used[start]:
                continue
            path = [start]
            used[start] = True
            x, y, z = start // (my * mz), start // mz % my, start % mz
            while len(path) < CHAIN_LEN:
                for d in perms[order[k % order.size]]:
                    a, b, e = (x + moves[d][0]) % mx, (y + moves[d][1]) % my, (z + moves[d][2]) % mz
                    s = (a * my + b) * mz + e
                    if not used[s]:
                        x, y, z = a, b, e
                        used[s] = True
                        path.append(s)
                        break
                else:
                    break
                k += 1
            if len(path) == CHAIN_LEN:
                walk[c * CHAIN_LEN:(c + 1) * CHAIN_LEN] = path
                break
            used[path] = False
    if total < 3 * nfree or nchain:
        free = rng.choice(np.flatnonzero(~used), nfree, replace=False)
    else:
        free = np.unique(rng.integers(0, total, int(1.4 * nfree) + 64))
        free = rng.permutation(free)[:nfree]
        while free.size < nfree:
            free = np.unique(np.concatenate([free, rng.integers(0, total, nfree)]))
            free = rng.permutation(free)[:nfree]
    s = np.concatenate([walk, free])
    return np.stack([s // (my * mz), s // mz % my, s % mz], 1), box / m


def _permutations(n):
    if n == 1:
        return [(0,)]
    return [p[:i] + (n - 1,) + p[i:] for p in _permutations(n - 1) for i in range(n)]


def _wrap(x, box):
    return np.clip(x - box * np.round(x / box), -box / 2, box / 2)


def _system(case, seed, n=None, frames=1):
    """A seeded electrolyte: particles on distinct jittered sites, so no two
    are closer than 3.4 A; `frames` sets of positions on the same sites."""
    rng = np.random.default_rng([seed, n or case["n"], 71])
    n = n or case["n"]
    box = _box(case, n)
    types, chains = _types(case, n)
    zat, mass = (np.array(v) for v in SPECIES[case["species"]])
    sites, pitch = _sites(rng, box, len(chains), n - len(chains) * CHAIN_LEN)
    amp = np.minimum((pitch - 3.4) / 2, 0.75)
    ros = [_wrap((sites + 0.5) * pitch - box / 2 + rng.uniform(-amp, amp, (n, 3)), box)
           for _ in range(frames)]
    sd = np.sqrt(RGAS * 298.0 / (mass / 1000.0)) * 0.01
    rod = rng.standard_normal((n, 3)) * sd[types - 1][:, None]
    npt = zat.size
    return dict(n=n, box=box, types=types, chains=chains, zat=zat, mass=mass,
                sig=np.full(npt, SIGMA), eps=np.full(npt, KT), ros=ros, rod=rod, rng=rng)


def _knots(case, rng):
    return 0.05 * rng.standard_normal((6, NKNOT))


def _replica_case(case, r):
    """Replica r of a batch: sizes from an eighth to the whole of n, the box
    and the mesh with it."""
    f = 0.125 + 0.875 * ((r * 0.6180339887) % 1.0)
    n = max(200, int(case["n"] * f) // 2 * 2)
    c = dict(case, n=n)
    box = _box(c)
    c["rc"] = min(case["rc"], 0.45 * float(box.min()))
    spacing = float(_box(case)[0]) / case["mesh"] * c["rc"] / case["rc"]
    c["mesh"] = c["meshz"] = _mesh_for(box[0], spacing, case["order"])
    return c


# ---------------------------------------------------------------- engines
def _tables(case, s):
    return E.build_tables(s["zat"], s["sig"], s["eps"], rcut=case["rc"], epsi_four_pi=EFP,
                          alpha=3.0 / case["rc"])


def _engine(case, s, ro, tables=None, maxnneigh=0):
    eng = E.ForceEngine(s["n"], case["prec"])
    eng.set_box(s["box"])
    eng.set_particles(s["types"], s["zat"][s["types"] - 1], 1.0 / s["mass"])
    eng.set_tables(tables or _tables(case, s), case["rc"])
    eng.set_ewald(case["ewald"], 3.0 / case["rc"], case["order"],
                  (case["mesh"], case["mesh"], case["meshz"]), case["ncut"], False, False, EFP)
    eng.set_neighbor(case.get("nlist", "vlist"), 2.0, maxnneigh)
    if s["chains"]:
        eng.set_chains(s["chains"], *BOND)
        eng.set_angles(*ANGLE)
    eng.upload_positions(ro)
    eng.upload_velocities(s["rod"])
    return eng


def _bd_factors(npt):
    return E.bd_factors(DT_BD, 298.0, [1.0] * npt)


def _capacity(case, n, box):
    mean = 4.0 / 3.0 * math.pi * (case["rc"] + 2.0) ** 3 * n / float(box.prod())
    return int(min(n - 1, 4 * mean + 64))


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case, kind=kind)
    if kind == "batch":
        reps = [_replica_case(case, r) for r in range(case["replicas"])]
        cache = {}
        st["engines"] = []
        for r, c in enumerate(reps):
            s = _system(c, seed * 1000 + r)
            if c["rc"] not in cache:
                cache[c["rc"]] = _tables(c, s)
            e = _engine(c, s, s["ros"][0], cache[c["rc"]], _capacity(c, c["n"], s["box"]))
            e.set_bd(*_bd_factors(2), seed * 1000 + r)
            st["engines"].append(e)
        st["batch"] = E.Batch(st["engines"])
        st["batch"].compute()
        return st
    s = _system(case, seed, frames=case.get("frames", 1))
    eng = st["engine"] = _engine(case, s, s["ros"][0],
                                 maxnneigh=_capacity(case, s["n"], s["box"]) if kind == "bd" else 0)
    if kind == "utotal":
        st["positions"], st["next"] = _position_sets(case, seed, s), 0
        eng.build_list()
    elif kind in ("md", "bd"):
        if kind == "bd":
            eng.set_bd(*_bd_factors(s["zat"].size), seed)
        eng.utotal()
    elif kind == "mc":
        st.update(ro=s["ros"][0].copy(), box=s["box"], rng=np.random.default_rng([seed, 5]))
        eng.build_list()
    else:
        c = _knots(case, np.random.default_rng([seed, 9]))
        eng.set_pair_params(s["zat"], s["sig"], s["eps"], rcut=case["rc"], epsi_four_pi=EFP,
                            alpha=3.0 / case["rc"])
        eng.set_knots(KNOT_LO, case["rc"], c)
        if kind == "fm":
            eng.fm_set_frames(np.stack(s["ros"]), _targets(case, seed, s))
        else:
            eng.build_list()
    return st


def _position_sets(case, seed, s):
    """What successive calls upload: small steps of a host integrator around
    one configuration, or independent snapshots."""
    rng = np.random.default_rng([seed, 17])
    if case["move"] > 0:
        return [_wrap(s["ros"][0] + case["move"] * rng.standard_normal((s["n"], 3)), s["box"])
                for _ in range(4)]
    return [_system(case, seed + 1000 * (k + 1))["ros"][0] for k in range(3)]


def _kept(case, x):
    """Forces, energies and gradients as a program keeps them: 32 bits on
    the mixed path."""
    return np.asarray(x, np.float32 if case["prec"] == "mixed" else np.float64)


def _energies(case, e):
    return _kept(case, [e.tot, e.twob0, e.rec, e.bond, e.virial])


def run(st):
    case, kind = st["case"], st["kind"]
    if kind == "batch":
        b = st["batch"]
        b.step_bd(case["steps"])
        en = [_energies(case, e) for e in b.energies()]
        return dict(ro=np.concatenate([e.download_state()[0] for e in st["engines"]]),
                    energy=np.stack(en))
    eng = st["engine"]
    if kind == "md":
        eng.step_md(case["steps"], DT_MD)
        ro, rod, rodd = eng.download_state()
        return dict(ro=ro, rod=_kept(case, rod), rodd=_kept(case, rodd),
                    energy=_energies(case, eng.energy()))
    if kind == "bd":
        eng.step_bd(nsteps=case["steps"])
        return dict(ro=eng.download_state()[0], force=_kept(case, eng.download_forces()),
                    energy=_energies(case, eng.energy()))
    if kind == "utotal":
        eng.upload_positions(st["positions"][st["next"] % len(st["positions"])])
        st["next"] += 1
        f, e = eng.utotal()
        return dict(force=_kept(case, f), energy=_energies(case, e))
    if kind == "mc":
        return _sweep(st)
    if kind == "adjoint":
        g = eng.adjoint()
        return {k: _kept(case, v) for k, v in g.items()}
    g = eng.fm_loss_grad()
    return {k: _kept(case, v) for k, v in g.items()}


def _trial(rng, ro, box):
    i = int(rng.integers(ro.shape[0]))
    return i, _wrap(ro[i] + rng.uniform(-0.5, 0.5, 3), box), rng.random()


def _sweep(st):
    """Metropolis trial moves of single particles, the host deciding."""
    eng, ro, box, case = st["engine"], st["ro"], st["box"], st["case"]
    du_pair, du_rec = np.zeros(case["trials"]), np.zeros(case["trials"])
    kept = False
    for t in range(case["trials"]):
        i, new, u = _trial(st["rng"], ro, box)
        du_pair[t], overlap = eng.mc_delta_pair([i + 1], new[None])
        if overlap:
            continue
        du_rec[t] = eng.mc_delta_rec([i + 1], new[None], reuse_current=kept)
        kept = True
        if u < math.exp(min(0.0, -(du_pair[t] + du_rec[t]) / KT)):
            eng.mc_accept([i + 1], new[None])
            ro[i] = new
    return dict(du_pair=_kept(case, du_pair), du_rec=_kept(case, du_rec), ro=ro.copy())


# ------------------------------------------------------------------- work
def work(case):
    """Bytes and operations of one pass: per force evaluation the particle
    data read and the forces written, the pair list read, the mesh written
    by the spreading, transformed there and back and read by the gather;
    per step the FP64 state read and written."""
    kind = case["kind"]
    if kind == "batch":
        parts = [_evaluation(_replica_case(case, r)) for r in range(case["replicas"])]
        ns = [_replica_case(case, r)["n"] for r in range(case["replicas"])]
        return dict(bytes=case["steps"] * (sum(p[0] for p in parts) + 96 * sum(ns)),
                    flops=case["steps"] * sum(p[1] for p in parts))
    n = case["n"]
    b, f = _evaluation(case)
    if kind in ("md", "bd"):
        state = 144 if kind == "md" else 96
        return dict(bytes=case["steps"] * (b + state * n), flops=case["steps"] * f)
    if kind == "utotal":
        rebuild = 4.0 * _entries(case) if case["move"] < 0 else 0.0
        return dict(bytes=b + 48 * n + rebuild, flops=f)
    if kind == "mc":
        # the kept spectrum read once per trial, and once more transformed
        # and accepted moves added (about two thirds of the trials)
        spec = 8.0 * case["mesh"] ** 2 * (case["mesh"] + 2) * case["meshz"] / case["mesh"]
        return dict(bytes=spec * case["trials"] * 5 / 3, flops=3 * spec * case["trials"])
    if kind == "adjoint":
        return dict(bytes=b + 4.0 * _entries(case) + 32 * n, flops=f + 60 * _entries(case))
    return dict(bytes=case["frames"] * (2 * b + 4.0 * _entries(case) + 72 * n),
                flops=case["frames"] * (2 * f + 120 * _entries(case)))


def _entries(case):
    """Stored list entries: both directions, radius rc + 2 A."""
    return 4.0 / 3.0 * math.pi * (case["rc"] + 2.0) ** 3 * case["density"] * case["n"]


def _evaluation(case):
    real = 4 if case["prec"] == "mixed" else 8
    n, pairs = case["n"], _entries(case)
    nbytes, flops = n * (4 * real + 24) + 4 * pairs, 30 * pairs
    if case["ewald"] == "std":
        nk = 4.0 / 3.0 * math.pi * case["ncut"] ** 3 / 2
        return nbytes + 24 * n, flops + 16 * nk * n
    m = case["mesh"] ** 2 * case["meshz"]
    mc = m / 2 + m / case["mesh"]
    # spreading 1 mesh out; five passes in and out; gather 1 mesh in
    nbytes += real * (2 * m + 2 * m + 14 * mc) + 2 * 4 * real * n
    flops += 10 * m * math.log2(m) / 2 + n * case["order"] ** 3 * 10
    return nbytes, flops


# -------------------------------------------------- results in 64-bit torch
class _Model:
    """The energy that the engine evaluates, in torch FP64, differentiable:
    table potential (its analytic form), SPME or standard Ewald sum with the
    self term, bonds and angles, the spline pair term."""

    def __init__(self, case, s):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.case, self.n = case, s["n"]
        self.box = self._t(s["box"])
        self.types = torch.as_tensor(s["types"].astype(np.int64) - 1, device=self.dev)
        self.mass = self._t(s["mass"])[self.types]
        self.alpha = 3.0 / case["rc"]
        self.zat, self.sig, self.eps = (self._t(s[k]) for k in ("zat", "sig", "eps"))
        self.knots = None
        beads = len(s["chains"]) * CHAIN_LEN
        idx = torch.arange(beads, device=self.dev)
        self.bond_i = idx[idx % CHAIN_LEN < CHAIN_LEN - 1]
        self.angle_i = idx[(idx % CHAIN_LEN > 0) & (idx % CHAIN_LEN < CHAIN_LEN - 1)]

    def _t(self, x):
        return torch.as_tensor(np.asarray(x, np.float64), device=self.dev)

    def wrap(self, x):
        y = x - self.box * torch.round(x / self.box)
        return torch.where(x.abs() > self.box / 2, y, x)

    @torch.no_grad()
    def pairs(self, x):
        """Indices of the pairs within rc."""
        rc2 = self.case["rc"] ** 2
        m = [int(v) for v in torch.floor(self.box / self.case["rc"])]
        if min(m) < 3:
            i, j = torch.triu_indices(self.n, self.n, 1, device=self.dev)
            d = self.minimum(x[i] - x[j])
            near = (d * d).sum(1) <= rc2
            return i[near], j[near]
        mt = torch.tensor(m, device=self.dev)
        c = torch.minimum(((x / self.box + 0.5) * mt).floor().long().clamp(min=0), mt - 1)
        cell = (c[:, 0] * m[1] + c[:, 1]) * m[2] + c[:, 2]
        count = torch.bincount(cell, minlength=m[0] * m[1] * m[2])
        depth = int(count.max())
        order = torch.argsort(cell, stable=True)
        start = torch.cumsum(count, 0) - count
        slot = torch.empty_like(cell)
        slot[order] = torch.arange(self.n, device=self.dev) - start[cell[order]]
        table = torch.full((count.numel(), depth), -1, dtype=torch.int64, device=self.dev)
        table[cell, slot] = torch.arange(self.n, device=self.dev)
        grid = table.reshape(m[0], m[1], m[2], depth)
        chunk = max(1, int(6e7 / depth / depth))
        out_i, out_j = [], []
        for off in [(a, b, e) for a in (-1, 0, 1) for b in (-1, 0, 1) for e in (-1, 0, 1)
                    if (a, b, e) >= (0, 0, 0)]:
            other = torch.roll(grid, [-v for v in off], (0, 1, 2)).reshape(-1, depth)
            for k in range(0, table.shape[0], chunk):
                i, j = torch.broadcast_tensors(table[k:k + chunk, :, None],
                                               other[k:k + chunk, None, :])
                ok = (i >= 0) & (j >= 0)
                if off == (0, 0, 0):
                    ok &= i < j
                i, j = i[ok], j[ok]
                d = self.minimum(x[i] - x[j])
                near = (d * d).sum(1) <= rc2
                out_i.append(i[near])
                out_j.append(j[near])
        return torch.cat(out_i), torch.cat(out_j)

    def minimum(self, d, scale=1.0):
        return d - self.box * scale * torch.round((d / (self.box * scale)).detach())

    def pair_energy(self, x, i, j, q, scale):
        d = self.minimum(x[i] * scale - x[j] * scale, scale)
        r = torch.sqrt((d * d).sum(1))
        u = EFP * q[i] * q[j] * torch.erfc(self.alpha * r) / r
        ti, tj = self.types[i], self.types[j]
        sig = 0.5 * (self.sig[ti] + self.sig[tj])
        near = r < LJCUT * sig
        eps = torch.sqrt(self.eps[ti] * self.eps[tj])
        s6 = (sig / r)[near] ** 6
        u = u.sum() + (4.0 * eps[near] * (s6 * s6 - s6) + eps[near]).sum()
        if self.knots is not None:
            h = (self.case["rc"] - KNOT_LO) / (NKNOT - 3)
            y = (r - KNOT_LO) / h
            on = (y >= 0) & (y < NKNOT - 3)
            y = y[on]
            k = y.detach().floor()
            f, k = y - k, k.long()
            g = 1.0 - f
            w = (g ** 3 / 6, (3 * f ** 3 - 6 * f ** 2 + 4) / 6,
                 (-3 * f ** 3 + 3 * f ** 2 + 3 * f + 1) / 6, f ** 3 / 6)
            lo, hi = torch.minimum(ti, tj)[on], torch.maximum(ti, tj)[on]
            p = lo * self.zat.numel() - lo * (lo - 1) // 2 + hi - lo
            u = u + sum((w[m] * self.knots[p, k + m]).sum() for m in range(4))
        return u

    def _weights(self, f):
        """Cardinal B-spline weights M(f + i), i = 0..order-1."""
        v = [f, 1.0 - f]
        for n in range(3, self.case["order"] + 1):
            last = v + [torch.zeros_like(f)]
            v = [((f + i) * last[i] + (n - i - f) * (last[i - 1] if i else 0.0)) / (n - 1)
                 for i in range(n)]
        return v

    def _influence(self, scale):
        """G(k) of E = 1/2 sum G |Q(k)|^2 over the whole spectrum."""
        order, axes, k2 = self.case["order"], [], 0.0
        knot = [float(v) for v in self._weights(torch.zeros((), dtype=torch.float64))]
        s = self.mesh
        for a in range(3):
            m = torch.arange(s[a] // 2 + 1 if a == 2 else s[a], device=self.dev,
                             dtype=torch.float64)
            m = torch.where(m > s[a] / 2, m - s[a], m)
            acc = sum(knot[k + 1] * torch.exp(2j * math.pi * m * k / s[a])
                      for k in range(order - 1))
            b2 = 1.0 / (acc.real ** 2 + acc.imag ** 2)
            if order % 2:
                b2 = torch.where(2 * m.abs() == s[a], torch.zeros_like(b2), b2)
            shape = [1, 1, 1]
            shape[a] = -1
            axes.append(b2.reshape(shape))
            k2 = k2 + ((2.0 * math.pi * m / (self.box[a] * scale)) ** 2).reshape(shape)
        k2 = torch.where(k2 == 0, torch.full_like(k2, float("inf")), k2)
        g = 4.0 * math.pi / (self.box * scale).prod() * torch.exp(-k2 / (4.0 * self.alpha ** 2)) / k2
        return g * axes[0] * axes[1] * axes[2]

    @property
    def mesh(self):
        return (self.case["mesh"], self.case["mesh"], self.case["meshz"])

    def charge_mesh(self, x, q):
        s, order = self.mesh, self.case["order"]
        u = x / self.box * torch.tensor(s, dtype=torch.float64, device=self.dev)
        base = u.detach().floor()
        w = [self._weights((u - base)[:, a]) for a in range(3)]
        base = base.long()
        at = [[(base[:, a] - i) % s[a] for i in range(order)] for a in range(3)]
        mesh = torch.zeros(s[0] * s[1] * s[2], dtype=torch.float64, device=self.dev)
        wz, az = torch.stack(w[2], 1), torch.stack(at[2], 1)
        for i in range(order):
            for j in range(order):
                k = ((at[0][i] * s[1] + at[1][j]) * s[2])[:, None] + az
                mesh = mesh.index_add(0, k.reshape(-1),
                                      ((q * w[0][i] * w[1][j])[:, None] * wz).reshape(-1))
        return mesh.reshape(s)

    def spectrum_energy(self, spec, g):
        wt = torch.full((spec.shape[2],), 2.0, dtype=torch.float64, device=self.dev)
        wt[0] = wt[-1] = 1.0
        return 0.5 * EFP * (g * wt * (spec.real ** 2 + spec.imag ** 2)).sum()

    def rec_energy(self, x, q, scale):
        self_term = -EFP * self.alpha / math.sqrt(math.pi) * (q * q).sum()
        if self.case["ewald"] == "spm":
            spec = torch.fft.rfftn(self.charge_mesh(x, q))
            return self.spectrum_energy(spec, self._influence(scale)) + self_term
        m = torch.arange(-self.case["ncut"], self.case["ncut"] + 1, device=self.dev,
                         dtype=torch.float64)
        m = torch.cartesian_prod(m, m, m)
        m2 = (m * m).sum(1)
        m = m[(m2 > 0) & (m2 <= self.case["ncut"] ** 2)]
        k2 = ((2.0 * math.pi * m / (self.box * scale)) ** 2).sum(1)
        ph = 2.0 * math.pi * (x / self.box) @ m.T
        s2 = (q @ torch.cos(ph)) ** 2 + (q @ torch.sin(ph)) ** 2
        vol = (self.box * scale).prod()
        return EFP * 2.0 * math.pi / vol * (torch.exp(-k2 / (4.0 * self.alpha ** 2)) / k2
                                            * s2).sum() + self_term

    def chain_energies(self, x, scale):
        if not self.bond_i.numel():
            z = torch.zeros((), dtype=torch.float64, device=self.dev)
            return z, z
        k, p, eq = BOND
        d = self.minimum((x[self.bond_i] - x[self.bond_i + 1]) * scale, scale)
        bond = (k / p * (torch.sqrt((d * d).sum(1)) - eq) ** p).sum()
        k, p, eq = ANGLE
        a = self.minimum(x[self.angle_i] - x[self.angle_i - 1])
        b = self.minimum(x[self.angle_i] - x[self.angle_i + 1])
        cs = (a * b).sum(1) / torch.sqrt((a * a).sum(1) * (b * b).sum(1))
        theta = torch.acos(cs.clamp(-1.0, 1.0)) * 180.0 / math.pi
        return bond, (k / p * (theta - eq) ** p).sum()

    def terms(self, x, q=None, scale=1.0):
        """(two-body, reciprocal, bond, angle) energies."""
        q = self.zat[self.types] if q is None else q
        i, j = self.pairs(x.detach())
        bond, angle = self.chain_energies(x, scale)
        return self.pair_energy(x, i, j, q, scale), self.rec_energy(x, q, scale), bond, angle

    def forces(self, x):
        x = x.detach().requires_grad_()
        return -torch.autograd.grad(sum(self.terms(x)), x)[0]

    def energies(self, x):
        scale = torch.ones((), dtype=torch.float64, device=self.dev, requires_grad=True)
        t = self.terms(x, scale=scale)
        virial = torch.autograd.grad(t[0] + t[1] + t[2], scale)[0]
        return np.array([float(v) for v in (sum(t), t[0], t[1], t[2], virial)])


def _targets(case, seed, s):
    """Target forces of the frames: the model's with other parameters."""
    m = _Model(case, s)
    rng = np.random.default_rng([seed, 23])
    m.knots = m._t(_knots(case, np.random.default_rng([seed, 9]))
                   + 0.02 * rng.standard_normal((6, NKNOT)))
    m.zat = m.zat * m._t([1.03, 0.98, 1.02])
    m.sig = m.sig * m._t([1.02, 0.99, 1.01])
    m.eps = m.eps * m._t([0.95, 1.06, 1.03])
    return np.stack([m.forces(m._t(x)).cpu().numpy() for x in s["ros"]])


def _deviates(seed, n, step):
    """The engine's noise stream: Philox4x32-10 with counter (i, step, 0, 0)
    and key seed (Salmon et al., SC'11), three Box-Muller deviates."""
    c = [np.arange(n, dtype=np.uint64), np.full(n, step, np.uint64), np.zeros(n, np.uint64),
         np.zeros(n, np.uint64)]
    k, low = [seed & 0xFFFFFFFF, seed >> 32], np.uint64(0xFFFFFFFF)
    for _ in range(10):
        a, b = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(b >> np.uint64(32)) ^ c[1] ^ np.uint64(k[0]), b & low,
             (a >> np.uint64(32)) ^ c[3] ^ np.uint64(k[1]), a & low]
        k = [(k[0] + 0x9E3779B9) & 0xFFFFFFFF, (k[1] + 0xBB67AE85) & 0xFFFFFFFF]
    u = [(v.astype(np.float64) + 0.5) * 2.0 ** -32 for v in c]
    r0, r1 = np.sqrt(-2.0 * np.log(u[0])), np.sqrt(-2.0 * np.log(u[2]))
    return np.stack([r0 * np.cos(2 * np.pi * u[1]), r0 * np.sin(2 * np.pi * u[1]),
                     r1 * np.cos(2 * np.pi * u[3])], 1)


def _exact_bd(case, s, seed):
    m = _Model(case, s)
    fac1, fac2 = (float(v[0]) for v in _bd_factors(1))
    x = m._t(s["ros"][0])
    f = m.forces(x) * FFAC
    for step in range(case["steps"]):
        x = m.wrap(x + fac1 * f + fac2 * m._t(_deviates(seed, s["n"], step)))
        f = m.forces(x) * FFAC
    return x.cpu().numpy(), f.cpu().numpy(), m.energies(x)


def _exact_md(case, s):
    m = _Model(case, s)
    x, v = m._t(s["ros"][0]), m._t(s["rod"])
    a = torch.zeros_like(x)
    for _ in range(case["steps"]):
        x = m.wrap(x + DT_MD * v + 0.5 * DT_MD ** 2 * a)
        new = m.forces(x) * FFAC / m.mass[:, None]
        v = v + 0.5 * DT_MD * (new + a)
        a = new
    return dict(ro=x.cpu().numpy(), rod=v.cpu().numpy(), rodd=a.cpu().numpy(),
                energy=m.energies(x))


def _exact_mc(case, s, seed):
    m = _Model(case, s)
    ro, rng = s["ros"][0].copy(), np.random.default_rng([seed, 5])
    q = m.zat[m.types]
    g = m._influence(1.0)
    mesh = m.charge_mesh(m._t(ro), q)
    old_rec = m.spectrum_energy(torch.fft.rfftn(mesh), g)
    du_pair, du_rec = np.zeros(case["trials"]), np.zeros(case["trials"])
    for t in range(case["trials"]):
        i, new, u = _trial(rng, ro, s["box"])
        x = m._t(np.concatenate([ro, new[None]]))
        both = []
        for at in (s["n"], i):
            d = m.minimum(x[:s["n"]] - x[at])
            r2 = (d * d).sum(1)
            j = torch.nonzero((r2 <= case["rc"] ** 2)
                              & (torch.arange(s["n"], device=m.dev) != i))[:, 0]
            y = m._t(ro)
            y[i] = x[at]
            both.append(m.pair_energy(y, torch.full_like(j, i), j, q, 1.0))
        du_pair[t] = float(both[0] - both[1])
        pair = torch.stack([x[s["n"]], x[i]])
        trial = mesh + m.charge_mesh(pair, torch.stack([q[i], -q[i]]))
        rec = m.spectrum_energy(torch.fft.rfftn(trial), g)
        du_rec[t] = float(rec - old_rec)
        if u < math.exp(min(0.0, -(du_pair[t] + du_rec[t]) / KT)):
            ro[i], mesh, old_rec = new, trial, rec
    return dict(du_pair=du_pair, du_rec=du_rec, ro=ro)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        out = []
        # thousands of small evaluations one after another take too long
        if case["replicas"] * case["steps"] > 2000:
            return None
        for r in range(case["replicas"]):
            c = _replica_case(case, r)
            out.append(_exact_bd(c, _system(c, seed * 1000 + r), seed * 1000 + r))
        return dict(ro=np.concatenate([o[0] for o in out]),
                    energy=np.stack([o[2] for o in out]))
    if kind in ("md", "bd") and case["n"] * case["steps"] > 1.2e7:
        return None
    s = _system(case, seed, frames=case.get("frames", 1))
    if kind == "md":
        return _exact_md(case, s)
    if kind == "bd":
        ro, f, en = _exact_bd(case, s, seed)
        return dict(ro=ro, force=f, energy=en)
    if kind == "mc":
        return _exact_mc(case, s, seed)
    m = _Model(case, s)
    if kind == "utotal":
        x = m._t(_position_sets(case, seed, s)[0])
        return dict(force=(m.forces(x) * FFAC).cpu().numpy(), energy=m.energies(x))
    m.knots = m._t(_knots(case, np.random.default_rng([seed, 9]))).requires_grad_()
    par = [m.zat, m.sig, m.eps]
    for p in par:
        p.requires_grad_()
    if kind == "adjoint":
        x = m._t(s["ros"][0]).requires_grad_()
        q = m.zat[m.types].detach().requires_grad_()
        t = m.terms(x, q)
        # the engine's model energy leaves the angle term to u%angle
        gx, gq, gs, ge, gk = torch.autograd.grad(sum(t), [x, q, m.sig, m.eps, m.knots])
        zat = torch.zeros_like(m.zat).detach().index_add(0, m.types, gq)
        return dict(dq=gq.cpu().numpy(), dzat=zat.cpu().numpy(), dsigat=gs.cpu().numpy(),
                    depsat=ge.cpu().numpy(), dknot=gk.cpu().numpy(), dro=gx.cpu().numpy(),
                    E=float(t[0] + t[1] + t[2]))
    targets = _targets(case, seed, s)
    total, grads = 0.0, None
    for ro, tgt in zip(s["ros"], targets):
        x = m._t(ro).requires_grad_()
        f = -torch.autograd.grad(sum(m.terms(x)), x, create_graph=True)[0]
        loss = ((f - m._t(tgt)) ** 2).sum()
        g = torch.autograd.grad(loss, par + [m.knots])
        grads = g if grads is None else [a + b for a, b in zip(grads, g)]
        total += float(loss)
    return dict(loss=total, **{k: v.cpu().numpy() for k, v in
                               zip(("dzat", "dsigat", "depsat", "dknot"), grads)})
