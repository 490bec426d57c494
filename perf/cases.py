"""The work whose time and accuracy are tracked: batched energy / force evaluations, batched
minimizations and the served-minimization pool, each through the package's Python entry points.

A case describes a batch of molecules (a library of `molecules` seeded branched molecules of
`lo`..`hi` atoms, each with `conformers` conformers) and what is done with it.  The library
belongs to the case; the conformers (coordinates) come from the seed given to prepare().

  listed()            the tracked cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) device-resident inputs and handles, as a program holds them before a call
  run(state)          one pass; returns its outputs
  work(case)          bytes and flops a pass cannot do without
  exact(case, seed)   an evaluation's outputs in 64 bits by plain torch
"""
import ctypes
import functools
import math

import numpy as np
import torch

from stormm_amd import _lib, restraints, serving, synthetic
from stormm_amd import synthesis as S
from stormm_amd.topology import AMBER_COULOMB, AMBER_SCEE, AMBER_SCNB, Topology

# Fixed-precision bits (coordinates, forces, energies) of the two precision models.
BITS = {"single": (32, 23, 26), "double": (32, 40, 32)}
FLOAT = {"single": torch.float32, "double": torch.float64}
IGB_OBC2 = 5
NEW_POSITIONS = 0.05   # A, conformers of an evaluated batch: thermal spread around the molecule
STRAINED = 0.3         # A, conformers to be minimized
SD_CYCLES, DX0 = 10, 0.01
CLASH_CYCLES = 5


# ------------------------------------------------------------------------------------------
# Cases
# ------------------------------------------------------------------------------------------
def _case(name, kind, molecules, conformers, lo, hi, precision="single", forces=True, gb=True,
          salt=0.0, tables=False, restrained=False, separate=False, cycles=0, library=0):
    """kind: "evaluate", "minimize" or "serve".  forces: energies only when false.  tables:
    AMBER-style stored Lennard-Jones tables of 16 types instead of combining rules.  separate:
    the non-bonded and valence launches one after the other instead of the fused evaluation.
    cycles: minimization cycles."""
    c = {"name": name, "kind": kind, "molecules": molecules, "conformers": conformers, "lo": lo,
         "hi": hi, "precision": precision, "forces": forces, "gb": gb, "salt": salt,
         "tables": tables, "restrained": restrained, "separate": separate, "cycles": cycles,
         "library": library}
    if name is None:
        del c["name"]
    return c


def listed():
    return [
        # The smallest call: 32 copies of one 48-atom molecule in vacuum, where launches count.
        _case("vacuum_32", "evaluate", 1, 32, 48, 48, gb=False),
        # One request of a serving program: conformers of a single large molecule (odd size),
        # far fewer systems than compute units.
        _case("conformers_24x487", "evaluate", 1, 24, 487, 487, library=1),
        # The benchmark's batch: 1024 heterogeneous molecules of 24-256 atoms in GB solvent.
        _case("batch_1024", "evaluate", 1024, 1, 24, 256, library=2),
        # Energies of the same batch, the line-search trial of a minimizer.
        _case("batch_1024_energy", "evaluate", 1024, 1, 24, 256, forces=False, library=2),
        # The double-precision model on the same batch.
        _case("batch_1024_double", "evaluate", 1024, 1, 24, 256, precision="double", library=2),
        # A screening library: many drug-sized molecules.
        _case("library_16384", "evaluate", 16384, 1, 32, 96, library=3),
        # Energies of a library at physiological salt (Debye screening) in double precision.
        _case("library_4096_salt_double", "evaluate", 4096, 1, 32, 96, precision="double",
              forces=False, salt=0.15, library=4),
        # AMBER topologies: stored Lennard-Jones tables.
        _case("tables_1024", "evaluate", 1024, 1, 24, 256, tables=True, library=5),
        # Positionally restrained molecules, non-bonded and valence launched separately as the
        # reference's callers do.
        _case("restrained_300", "evaluate", 300, 1, 40, 200, restrained=True, separate=True,
              library=6),
        # Minimization of one request's conformers: a chain of small launches.
        _case("minimize_33x149", "minimize", 1, 33, 149, 149, cycles=20, library=7),
        # Minimization of a whole batch.
        _case("minimize_4096", "minimize", 4096, 1, 16, 128, cycles=12, library=8),
        # Served minimization: requests of several conformers each admitted to the pool,
        # advanced in ticks of ten cycles, read back and released.
        _case("serve_8x20", "serve", 8, 20, 16, 512, cycles=20, library=9),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """Batches over the whole range: 1 to 16384 systems of 8 to 512 atoms, either precision,
    every option; at most the pair work of the largest listed case."""
    most = max(_pair_work(c) for c in listed())
    while True:
        kind = rng.choice(["evaluate"] * 6 + ["minimize"] * 3 + ["serve"])
        lo = _log_int(rng, 8, 512)
        hi = min(512, max(lo, int(lo * rng.uniform(1.0, 5.0))))
        if kind == "serve":
            c = _case(None, kind, _log_int(rng, 2, 12), _log_int(rng, 1, 40), lo, hi,
                      cycles=rng.choice([10, 20]))
        elif kind == "minimize":
            # Single precision: a long double-precision trajectory magnifies its last bits.
            c = _case(None, kind, _log_int(rng, 1, 2048), _log_int(rng, 1, 64), lo, hi,
                      gb=rng.random() < 0.8, tables=rng.random() < 0.3,
                      cycles=_log_int(rng, 5, 20))
        else:
            restrained = rng.random() < 0.15
            c = _case(None, kind, _log_int(rng, 1, 16384), _log_int(rng, 1, 64), lo, hi,
                      precision=rng.choice(["single", "single", "double"]),
                      forces=rng.random() < 0.7, gb=rng.random() < 0.8,
                      salt=rng.choice([0.0, 0.0, 0.15]), tables=rng.random() < 0.3,
                      restrained=restrained, separate=rng.random() < 0.2)
        c["library"] = rng.randrange(10, 1 << 20)
        systems = c["molecules"] * c["conformers"]
        if systems <= 16384 and 1.0e4 <= _pair_work(c) <= 0.6 * most and \
                c["molecules"] * (lo + hi) <= 2500000:
            return c


# ------------------------------------------------------------------------------------------
# Molecules
# ------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=16)
def _skeletons(size):
    """Four grown molecules of `size` atoms.  A molecule grows atom by atom, each bonded to an
    earlier one, so the first m atoms of one are themselves a molecule of m atoms."""
    return [synthetic.branched_molecule(max(size, 4), seed=5000 + k) for k in range(4)]


def _sizes(case):
    rng = np.random.default_rng([case["library"], 1])
    if case["kind"] == "serve":
        return synthetic.log_uniform_sizes(rng, case["molecules"], case["lo"], case["hi"])
    return rng.integers(case["lo"], case["hi"] + 1, case["molecules"])


def _charges(rng, n):
    """Charges on the 2^-23 e grid that sum to zero exactly."""
    q = rng.normal(0.0, 0.3, n)
    iq = np.rint((q - q.mean()) * 2.0 ** 23).astype(np.int64)
    resid = int(iq.sum())
    k = np.argsort(-np.abs(iq), kind="stable")[:abs(resid)]
    iq[k] -= 1 if resid > 0 else -1
    return iq * 2.0 ** -23


@functools.lru_cache(maxsize=4)
def _cached_library(key):
    case = dict(key)
    rng = np.random.default_rng([case["library"], 2])
    topos, shapes = [], []
    sizes = _sizes(case)
    skeletons = _skeletons(int(max(case["hi"], 4)))
    for n, pick in zip(sizes, rng.integers(0, len(skeletons), len(sizes))):
        n = int(n)
        t, x = skeletons[pick]
        b_in = (t.bonds < n).all(axis=1)
        b = t.bonds[b_in]
        a_in = (t.angles < n).all(axis=1)
        d = t.dihedrals[(t.dihedrals < n).all(axis=1)]
        a = t.angles[a_in]
        nb, na, nd = len(b), len(a), len(d)
        sig, eps = rng.uniform(2.0, 3.8, n), rng.uniform(0.02, 0.2, n)
        lj = {"lj_idx": np.arange(n, dtype=np.int32), "n_lj_types": n, "lj_sigma": sig,
              "lj_epsilon": eps}
        if case["tables"]:
            # Types in turn; one pair of types 5 % off the combining rule, as NBFIX pairs are.
            m = min(16, n)
            s6 = (0.5 * (sig[:m, None] + sig[None, :m])) ** 6
            lb = 4.0 * np.sqrt(eps[:m, None] * eps[None, :m]) * s6
            la = lb * s6
            la[0, m - 1] *= 1.05
            la[m - 1, 0] = la[0, m - 1]
            lj = {"lj_idx": (np.arange(n) % m).astype(np.int32), "n_lj_types": m,
                  "lja": la.ravel(), "ljb": lb.ravel(), "lja14": la.ravel().copy(),
                  "ljb14": lb.ravel().copy()}
        topos.append(Topology(
            natom=n, charge=_charges(rng, n), bonds=b, bond_k=rng.uniform(200.0, 400.0, nb),
            bond_r0=t.bond_r0[b_in], angles=a, angle_k=rng.uniform(40.0, 80.0, na),
            angle_theta=t.angle_theta[a_in], dihedrals=d, dihe_amp=rng.uniform(0.0, 2.0, nd),
            dihe_phase=np.where(rng.random(nd) < 0.5, 0.0, math.pi),
            dihe_freq=rng.integers(1, 4, nd).astype(np.float64),
            dihe_improper=np.zeros(nd, dtype=np.int32), dihe_scee=np.full(nd, AMBER_SCEE),
            dihe_scnb=np.full(nd, AMBER_SCNB), pb_radii=rng.uniform(1.2, 2.0, n),
            gb_screen=rng.uniform(0.7, 0.9, n), igb=IGB_OBC2 if case["gb"] else 0,
            dielectric=78.5, salt=case["salt"], coulomb=AMBER_COULOMB, **lj))
        shapes.append(x[:n])
    return topos, shapes


def _library(case):
    keys = ("kind", "molecules", "lo", "hi", "gb", "salt", "tables", "library")
    return _cached_library(tuple((k, case[k]) for k in keys))


def _conformers(case, seed):
    """Topologies and coordinates of every system, and the restraints (or None).  Coordinates
    lie on the 2^-32 A grid the synthesis stores."""
    topos, shapes = _library(case)
    rng = np.random.default_rng([seed, case["library"], 3])
    spread = NEW_POSITIONS if case["kind"] == "evaluate" else STRAINED
    reps = case["conformers"]
    flat = np.concatenate([x for x in shapes for _ in range(reps)])
    flat = flat + rng.normal(0.0, spread, flat.shape)
    flat = np.rint(flat * 2.0 ** 32) * 2.0 ** -32
    every = [t for t in topos for _ in range(reps)]
    cuts = np.cumsum([t.natom for t in every])[:-1]
    coords = np.split(flat, cuts)
    held = None
    if case["restrained"]:
        # Every third atom held to its place in the molecule, flat within 0.05 A.
        held = []
        for t, x in zip(topos, shapes):
            plan = restraints.apply_positional_restraints(x, range(0, t.natom, 3), 20.0, 0.05)
            held += [plan] * reps
    return every, coords, held


# ------------------------------------------------------------------------------------------
# Programs
# ------------------------------------------------------------------------------------------
class _DeviceWords:
    def __init__(self, pointer, shape):
        self.__cuda_array_interface__ = {"data": (int(pointer), False), "shape": shape,
                                         "typestr": "<i8", "version": 2}


def _words(pointer, *shape):
    """A tensor over int64 device memory that a handle owns."""
    return torch.as_tensor(_DeviceWords(pointer, shape), device="cuda")


class _Batch:
    """A batch's handles and tensors over its device arrays."""

    def __init__(self, case, topos, coords, held):
        self.case = case
        self.precision = case["precision"]
        gpos, frc, nrg = BITS[self.precision]
        self.ag = S.AtomGraphSynthesis(topos, restraints=held)
        self.ps = S.PhaseSpaceSynthesis(self.ag, gpos, frc)
        self.sc = S.ScoreCard(self.ag.system_count, nrg)
        self.ps.upload(coords)
        w = self.ps.writer()
        n = int(self.ag.info.padded_atom_count)
        self.positions = [_words(p, n) for p in (w.xcrd, w.ycrd, w.zcrd)]
        self.forces = [_words(p, n) for p in (w.xfrc, w.yfrc, w.zfrc)]
        acc = _lib.load().stormm_scorecard_device_accumulators(self.sc.handle)
        self.energies = _words(acc, self.ag.system_count, S.SCORECARD_STRIDE)[:, :13]
        dtype = FLOAT[self.precision]
        self.position_unit = torch.tensor(2.0 ** -gpos, dtype=dtype)
        self.force_unit = torch.tensor(2.0 ** -frc, dtype=dtype)
        self.energy_unit = torch.tensor(2.0 ** -nrg, dtype=dtype)
        if case["kind"] == "minimize":
            self.controls = S.minimize_controls(case["cycles"], min(SD_CYCLES, case["cycles"]),
                                                DX0, 0.0,
                                                clash_cycles=min(CLASH_CYCLES, case["cycles"]))
            self.start = [p.clone() for p in self.positions]
            self.line = S.LineMinimization(self.ag.system_count, DX0)
            lw = _lib.LinMinWriter()
            _lib.check(_lib.load().stormm_line_min_data(self.line.handle, ctypes.byref(lw)))
            self.line_state = _words(lw.l_move, 9, self.ag.system_count).view(torch.float64)
            self.line_start = self.line_state.clone()


class _Served:
    """A serving pool and the requests that a pass sends through it."""

    def __init__(self, case, topos, coords):
        self.case = case
        # Cycle limit and stop of the service's own workload; nothing stops within a pass.
        self.pool = serving.MinimizationPool(total_cycles=300, conv_rms=0.1)
        reps = case["conformers"]
        self.requests = [(topos[i], coords[i:i + reps]) for i in range(0, len(topos), reps)]


def prepare(case, seed):
    topos, coords, held = _conformers(case, seed)
    if case["kind"] == "serve":
        return _Served(case, topos, coords)
    return _Batch(case, topos, coords, held)


def _evaluate(b):
    forces = b.case["forces"]
    if forces:
        b.ps.initialize_forces()
    b.sc.initialize()
    if b.case["separate"]:
        S.launch_nonbonded(b.precision, b.ag, None, b.ps, b.sc, forces, True)
        S.launch_valence(b.precision, b.ag, None, b.ps, b.sc, forces, True)
    else:
        S.launch_mm_evaluation(b.precision, b.ag, None, b.ps, b.sc, forces, True)
    out = {"energies": b.energies * b.energy_unit}
    if forces:
        out["forces"] = [f * b.force_unit for f in b.forces]
    return out


def _minimize(b):
    for p, s in zip(b.positions, b.start):
        p.copy_(s)
    b.line_state.copy_(b.line_start)
    S.launch_minimization(b.precision, b.ag, b.ps, b.controls, b.sc, b.line)
    return {"energies": b.energies * b.energy_unit,
            "positions": [p * b.position_unit for p in b.positions]}


def _serve(s):
    pool = s.pool
    slots = []
    for topo, confs in s.requests:
        got = pool.admit_conformers(topo, confs)
        slots.append(got)
    every = [k for got in slots for k in got]
    for _ in range(s.case["cycles"] // 10):
        pool.minimize(10)
        steps, done, rms, energies = pool.status(every)
    positions = [pool.coordinates(k, topo.natom)
                 for (topo, _), got in zip(s.requests, slots) for k in got]
    for got in slots:
        pool.release(got)
    # The pool computes in single precision.
    return {"steps": steps, "rms": rms.astype(np.float32),
            "energies": energies.astype(np.float32),
            "positions": np.concatenate(positions).astype(np.float32)}


def run(state):
    if state.case["kind"] == "serve":
        return _serve(state)
    if state.case["kind"] == "minimize":
        return _minimize(state)
    return _evaluate(state)


# ------------------------------------------------------------------------------------------
# Work
# ------------------------------------------------------------------------------------------
def _evaluations(case):
    """(force evaluations, energy evaluations) of a pass: a minimization cycle takes one force
    evaluation and three trial energies, and the run (or tick) ends with one energy."""
    if case["kind"] == "evaluate":
        return (1, 0) if case["forces"] else (0, 1)
    ends = case["cycles"] // 10 if case["kind"] == "serve" else 1
    return case["cycles"], 3 * case["cycles"] + ends


def _pair_work(case):
    n = _sizes(case).astype(np.float64)
    return float((n * (n - 1.0)).sum()) * 0.5 * case["conformers"] * sum(_evaluations(case))


def work(case):
    """Flops: per pair, 24 for Coulomb + Lennard-Jones energies and 14 more for their forces; with
    GB 42 for the Born integrals, 16 for the pair energy, and for forces 16 more for the pair
    and 56 for the radius derivatives; 60 per valence term, 40 per atom.  Bytes: coordinates
    in, forces (or a minimization's coordinates) and energies out, each molecule's parameters
    once (eleven 8-byte values an atom, 40 bytes a valence term)."""
    n = _sizes(case).astype(np.float64)
    reps = case["conformers"]
    pairs = float((n * (n - 1.0)).sum()) * 0.5 * reps
    atoms = float(n.sum()) * reps
    # A branched molecule of n atoms has n - 1 bonds, about 1.7 n angles and 3 n dihedrals.
    terms = 5.7 * atoms
    ef, ee = _evaluations(case)
    energy_pair = 24.0 + ((42.0 + 16.0) if case["gb"] else 0.0)
    force_pair = energy_pair + 14.0 + ((16.0 + 56.0) if case["gb"] else 0.0)
    flops = pairs * ((ef * force_pair) + (ee * energy_pair)) + \
        (ef + ee) * ((60.0 * terms) + (40.0 * atoms))
    moved = 24.0 * (2 if (case["forces"] or case["kind"] != "evaluate") else 1)
    nbytes = atoms * moved + 104.0 * len(n) * reps + float(n.sum()) * (88.0 + 40.0 * 5.7)
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------------------------------------
# An evaluation in 64 bits
# ------------------------------------------------------------------------------------------
def _psi(r, ri, sj):
    """Born-integral term of a sphere of screened radius sj at distance r onto an atom of
    offset radius ri (pairwise descreening), the far field (r > 4 sj) by its series."""
    x = (sj / r) ** 2
    series = 1.0 / 3.0 + x * (0.4 + x * (3.0 / 7.0 + x * (4.0 / 9.0 + x * (5.0 / 11.0))))
    far = -(sj ** 3) / r ** 4 * series
    near = r <= 4.0 * sj
    # Values that keep the unused branches finite.
    rn = torch.where(near, r, 2.0 * sj + ri)
    outside = rn > ri + sj
    crossing = ~outside & (rn > (ri - sj).abs())
    inside = ~outside & ~crossing & (ri < sj)
    rms = torch.where(crossing, torch.ones_like(rn), rn - sj)
    base = -0.5 * sj / (rms * (rn + sj)) - 0.25 / rn * torch.log(rms.abs() / (rn + sj))
    theta = 0.5 / (ri * rn) * (rn ** 2 + ri ** 2 - sj ** 2)
    cross = -0.25 * ((2.0 - theta) / ri - 1.0 / (rn + sj)) - \
        0.25 / rn * torch.log(ri / (rn + sj))
    zero = torch.zeros_like(rn)
    val = torch.where(outside, base, torch.where(crossing, cross,
                                                 torch.where(inside, base - 1.0 / ri, zero)))
    return torch.where(near, val, far)


def _exact_group(case, topos, coords, held, dev):
    """Energies [systems][13] and forces [systems][atoms][3] of systems padded to one size."""
    f8 = torch.float64
    ns, m = len(topos), max(t.natom for t in topos)

    def atoms_of(values, fill):
        a = np.full((ns, m), fill)
        for s, v in enumerate(values):
            a[s, :len(v)] = v
        return torch.tensor(a, dtype=f8, device=dev)

    x = np.zeros((ns, m, 3))
    bonded = np.zeros((ns, m, m), dtype=np.float32)
    for s, (t, c) in enumerate(zip(topos, coords)):
        x[s, :t.natom] = c
        bonded[s, t.bonds[:, 0], t.bonds[:, 1]] = 1.0
        bonded[s, t.bonds[:, 1], t.bonds[:, 0]] = 1.0
    x = torch.tensor(x, dtype=f8, device=dev, requires_grad=True)
    adj = torch.tensor(bonded, device=dev)
    near2 = torch.matmul(adj, adj)
    excluded = (adj + near2 + torch.matmul(near2, adj)) > 0   # within three bonds
    real = atoms_of([np.ones(t.natom) for t in topos], 0.0) > 0
    pair = real[:, :, None] & real[:, None, :]
    pair = pair & ~torch.eye(m, dtype=torch.bool, device=dev)[None]
    energies = torch.zeros((ns, 13), dtype=f8, device=dev)
    root = math.sqrt(AMBER_COULOMB)
    q = atoms_of([t.charge * root for t in topos], 0.0)
    qq = q[:, :, None] * q[:, None, :]
    dx = x[:, :, None, :] - x[:, None, :, :]
    r2 = torch.where(pair, (dx * dx).sum(-1), torch.ones((), dtype=f8, device=dev))
    r = r2.sqrt()
    nb = (pair & ~excluded).to(f8)
    if case["tables"]:
        k = max(t.n_lj_types for t in topos)
        la, lb = np.zeros((ns, k, k)), np.zeros((ns, k, k))
        ty = np.zeros((ns, m), dtype=np.int64)
        for s, t in enumerate(topos):
            la[s, :t.n_lj_types, :t.n_lj_types] = t.lja.reshape(t.n_lj_types, -1)
            lb[s, :t.n_lj_types, :t.n_lj_types] = t.ljb.reshape(t.n_lj_types, -1)
            ty[s, :t.natom] = t.lj_idx
        ty = torch.tensor(ty, device=dev)
        row = torch.arange(ns, device=dev)[:, None, None]
        a12 = torch.tensor(la, device=dev)[row, ty[:, :, None], ty[:, None, :]]
        b6 = torch.tensor(lb, device=dev)[row, ty[:, :, None], ty[:, None, :]]
    else:
        sg = atoms_of([t.lj_sigma for t in topos], 1.0)
        ep = atoms_of([t.lj_epsilon for t in topos], 0.0)
        s6 = (0.5 * (sg[:, :, None] + sg[:, None, :])) ** 6
        b6 = 4.0 * (ep[:, :, None] * ep[:, None, :]).sqrt() * s6
        a12 = b6 * s6
    i6 = r2 ** -3
    parts = {7: 0.5 * (nb * (a12 * i6 - b6) * i6).sum((1, 2)),
             9: 0.5 * (nb * qq / r).sum((1, 2))}
    if case["gb"]:
        rho = atoms_of([t.pb_radii for t in topos], 1.5) - 0.09
        pbr = atoms_of([t.pb_radii for t in topos], 1.5)
        scr = atoms_of([t.gb_screen for t in topos], 0.8) * rho
        psi = (_psi(r, rho[:, :, None], scr[:, None, :]) * pair.to(f8)).sum(2)
        f = -rho * psi
        born = 1.0 / (1.0 / rho - torch.tanh((1.0 - 0.8 * f + 4.85 * f * f) * f) / pbr)
        kappa = 0.73 * math.sqrt(0.10806 * case["salt"])
        rr = born[:, :, None] * born[:, None, :]
        fgb = (r2 + rr * torch.exp(-0.25 * r2 / rr)).sqrt()
        both = qq * (1.0 - torch.exp(-kappa * fgb) / 78.5) / fgb * pair.to(f8)
        own = q * q * (1.0 - torch.exp(-kappa * born) / 78.5) / born
        parts[11] = -0.5 * (both.sum((1, 2)) + own.sum(1))
    # Valence terms of the whole group as one list each.
    first = [s * m for s in range(ns)]
    flat = x.reshape(-1, 3)

    def listed_terms(atoms, *values):
        idx = np.concatenate([np.asarray(atoms(t)) + f for t, f in zip(topos, first)])
        own = np.repeat(np.arange(ns), [len(atoms(t)) for t in topos])
        out = [torch.tensor(np.concatenate([np.asarray(v(t), dtype=np.float64) for t in topos]),
                            device=dev) for v in values]
        return torch.tensor(idx, device=dev).long(), torch.tensor(own, device=dev), out

    def add(slot, own, e):
        parts[slot] = parts.get(slot, 0.0) + torch.zeros(ns, dtype=f8,
                                                         device=dev).index_add(0, own, e)

    idx, own, (k2, r0) = listed_terms(lambda t: t.bonds, lambda t: t.bond_k,
                                      lambda t: t.bond_r0)
    if len(idx):
        d = (flat[idx[:, 1]] - flat[idx[:, 0]]).norm(dim=1)
        add(0, own, k2 * (d - r0) ** 2)
    idx, own, (k2, th0) = listed_terms(lambda t: t.angles, lambda t: t.angle_k,
                                       lambda t: t.angle_theta)
    if len(idx):
        u, v = flat[idx[:, 0]] - flat[idx[:, 1]], flat[idx[:, 2]] - flat[idx[:, 1]]
        th = torch.atan2(torch.linalg.cross(u, v).norm(dim=1), (u * v).sum(1))
        add(1, own, k2 * (th - th0) ** 2)
    idx, own, (amp, phase, freq) = listed_terms(lambda t: t.dihedrals, lambda t: t.dihe_amp,
                                                lambda t: t.dihe_phase, lambda t: t.dihe_freq)
    if len(idx):
        p = [flat[idx[:, c]] for c in range(4)]
        ab, bc, cd = p[1] - p[0], p[2] - p[1], p[3] - p[2]
        u, v = torch.linalg.cross(ab, bc), torch.linalg.cross(bc, cd)
        th = torch.atan2((torch.linalg.cross(u, v) * bc).sum(1) / bc.norm(dim=1),
                         (u * v).sum(1))
        add(2, own, amp * (1.0 + torch.cos(freq * th - phase)))
        # Each proper dihedral carries its attenuated 1:4 pair.
        i14 = (p[3] - p[0]).square().sum(1)
        at = (own, idx[:, 0] - own * m, idx[:, 3] - own * m)
        add(10, own, qq[at] / AMBER_SCEE / i14.sqrt())
        j6 = i14 ** -3
        add(8, own, (a12[at] * j6 - b6[at]) * j6 / AMBER_SCNB)
    if held is not None:
        atom = np.concatenate([h["atoms"][:, 0] + f for h, f in zip(held, first)])
        own = torch.tensor(np.repeat(np.arange(ns), [len(h) for h in held]), device=dev)
        to = torch.tensor(np.concatenate([h["init_target"] for h in held]), device=dev)
        d = (flat[torch.tensor(atom, device=dev).long()] - to).norm(dim=1)
        k3 = torch.tensor(np.concatenate([h["init_k"][:, 1] for h in held]), device=dev)
        r3 = torch.tensor(np.concatenate([h["init_r"][:, 2] for h in held]), device=dev)
        add(12, own, k3 * torch.clamp(d - r3, min=0.0) ** 2)
    for slot, e in parts.items():
        energies[:, slot] = e.detach()
    forces = None
    if case["forces"]:
        total = sum(e.sum() for e in parts.values())
        forces = -torch.autograd.grad(total, x)[0]
    return energies, forces


def exact(case, seed):
    """Evaluations only: a minimization's path has no value of its own in 64 bits."""
    if case["kind"] != "evaluate":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    topos, coords, held = _conformers(case, seed)
    counts = np.array([t.natom for t in topos])
    starts = np.concatenate([[0], np.cumsum((counts + 31) // 32 * 32)])
    energies = torch.zeros((len(topos), 13), dtype=torch.float64)
    forces = torch.zeros((3, int(starts[-1])), dtype=torch.float64)
    order = np.argsort(counts, kind="stable")
    at = 0
    while at < len(order):
        # Systems of like size together, about two million pairs at a time.
        end = at + 1
        while end < len(order) and (end + 1 - at) * int(counts[order[end]]) ** 2 <= 2000000:
            end += 1
        pick = [int(i) for i in order[at:end]]
        e, f = _exact_group(case, [topos[i] for i in pick], [coords[i] for i in pick],
                            None if held is None else [held[i] for i in pick], dev)
        energies[pick] = e.cpu()
        if f is not None:
            f = f.cpu()
            for k, i in enumerate(pick):
                n = int(counts[i])
                forces[:, starts[i]:starts[i] + n] = f[k, :n].T
        at = end
    out = {"energies": energies}
    if case["forces"]:
        out["forces"] = list(forces)
    return out
