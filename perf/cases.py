"""Performance cases: the work a user of this package runs, through its
public entry points (``Engine``, ``ReplicaLadder``, ``BDEngine`` and the
allocation-free factorisation of the C-ABI).

A case is a dict of plain values; ``kind`` says what runs:

force   a host engine that integrates by itself: its coordinates go in, the
        forces come back (neighbour lists included, as after every move)
steps   Langevin dynamics resident on the GPU, then the trajectory frame
energy  the energy terms of every system, as an output interval takes them
remd    Langevin steps of a temperature ladder, then one exchange attempt
factor  the Cholesky factor of a diffusion tensor held on the GPU
bd      Brownian steps with hydrodynamic interaction, tensor refactored on
        the way

``model`` picks the system: ``hairpin`` (Debye-Hueckel chains of lognormal
or given length, extended start), ``coulomb`` (a compact chain, plain
Coulomb), ``ewald`` (a chain with explicit ions in a periodic cube),
``valence`` (compact chains whose every base pair is a hydrogen-bond
candidate, so the valence limit is at work).  ``steps`` with
``rebuild_every`` 0 rebuilds the neighbour lists by the displacement
trigger, otherwise every that many steps.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

from tis_amd import topology as T
from tis_amd.bdhi import bead_spring_chain
from tis_amd.engine import BDEngine, Engine, load_library
from tis_amd.remd import ReplicaLadder
from tis_amd.sysdesc import (E_BANGLE, E_BOND, E_ELE, E_EXV, E_HBOND, E_MAX, E_STACK, E_TOTAL,
                             E_VELO, ELE_COULOMB, ELE_DH, MP_PHOS, MP_SUGAR)
from tis_amd.topology import BOLTZ_KCAL_MOL

TSTEP = 0.05            # tau, the DT15 Langevin step
IONIC = 0.150           # M
TOPOLOGY_SEED = 20261202


def listed():
    return [
        # one call of a host program's force loop on the 64-nt hairpin: the
        # smallest work there is, all latency
        dict(name="force_hairpin", kind="force", model="hairpin", systems=1, nt=64),
        # the same for a compact 320-nt chain with plain Coulomb
        dict(name="force_coulomb", kind="force", model="coulomb", systems=1, nt=320),
        # dynamics of one small molecule
        dict(name="steps_hairpin", kind="steps", model="hairpin", systems=1, nt=64, steps=200, rebuild_every=10),
        # the throughput batch: 512 chains of lognormal length (20-600 nt)
        # and the 64-replica ladder of the 64-nt hairpin
        dict(name="steps_batch", kind="steps", model="hairpin", systems=512, nt=120, ladder=64, steps=500,
             rebuild_every=10),
        # a design screen of 128 chains under the displacement trigger
        dict(name="steps_trigger", kind="steps", model="hairpin", systems=128, nt=120, steps=200, rebuild_every=0),
        # the longest serving job, alone on the GPU
        dict(name="steps_job", kind="steps", model="hairpin", systems=1, nt=2000, steps=200, rebuild_every=10),
        # a chain with 565 explicit ions, Ewald electrostatics
        dict(name="steps_ewald", kind="steps", model="ewald", systems=1, nt=76, ions=565, box=150.0, hmax=10,
             steps=100, rebuild_every=10),
        # chains limited by the hydrogen-bond valence
        dict(name="steps_valence", kind="steps", model="valence", systems=64, nt=40, steps=100, rebuild_every=10),
        # energies of the throughput batch at one output interval
        dict(name="energy_batch", kind="energy", model="hairpin", systems=512, nt=120, ladder=64),
        # replica exchange of the 64-nt hairpin over 64 temperatures
        dict(name="remd_ladder", kind="remd", model="hairpin", systems=64, nt=64, steps=200, rebuild_every=10),
        # the diffusion tensor of 3,000 beads
        dict(name="factor_3000", kind="factor", beads=3000),
        # 300 beads, the tensor refactored at every step as the reference does
        dict(name="bd_300", kind="bd", beads=300, steps=20, refactor_every=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["force", "steps", "steps", "steps", "energy", "remd", "factor", "bd"])
    if kind == "factor":
        return dict(kind=kind, beads=_log_int(rng, 60, 3000))
    if kind == "bd":
        return dict(kind=kind, beads=_log_int(rng, 40, 1200), steps=rng.randint(5, 20),
                    refactor_every=rng.choice([1, 5, 10]))
    if kind == "remd":
        return dict(kind=kind, model="hairpin", systems=_log_int(rng, 4, 64), nt=_log_int(rng, 24, 120),
                    steps=rng.randint(50, 200), rebuild_every=10)
    if kind == "energy":
        return dict(kind=kind, model="hairpin", systems=_log_int(rng, 1, 512), nt=_log_int(rng, 40, 160))
    if kind == "force":
        if rng.random() < 0.4:
            return dict(kind=kind, model="coulomb", systems=1, nt=_log_int(rng, 30, 320))
        return dict(kind=kind, model="hairpin", systems=rng.choice([1, 1, 2, 4]), nt=_log_int(rng, 20, 1000))
    steps = rng.randint(50, 200)
    model = rng.choice(["hairpin", "hairpin", "hairpin", "ewald", "valence", "coulomb"])
    if model == "ewald":
        box = rng.choice([60.0, 90.0, 120.0, 150.0])
        return dict(kind=kind, model=model, systems=1, nt=rng.randint(16, 76), ions=_log_int(rng, 24, 565), box=box,
                    hmax=rng.randint(5, 10), steps=steps, rebuild_every=10)
    if model == "valence":
        return dict(kind=kind, model=model, systems=_log_int(rng, 1, 64), nt=rng.randint(24, 40), steps=steps,
                    rebuild_every=10)
    if model == "coulomb":
        return dict(kind=kind, model=model, systems=1, nt=_log_int(rng, 30, 320), steps=steps, rebuild_every=10)
    n = _log_int(rng, 1, 256)
    return dict(kind=kind, model=model, systems=n, nt=_log_int(rng, 20, 160 if n > 4 else 2000), steps=steps,
                rebuild_every=rng.choice([10, 10, 20, 0]))


# ------------------------------------------------------------------ systems
def _hairpin(rng, n):
    stem, loop = int(rng.integers(4, 11)), int(rng.integers(3, 9))
    while 2 * stem + loop + 2 > n:
        stem, loop = max(2, stem - 1), max(3, loop - 1)
    return T.hairpin_design(rng, n, stem, loop)


def _temperatures(n):
    return [290.0 * (400.0 / 290.0) ** (k / max(n - 1, 1)) for k in range(n)]


@functools.lru_cache(maxsize=4)
def _topology(model, systems, nt, ladder, ions, box, hmax, remd):
    """(systems, compact base coordinates or None per system) of a case; the
    same for every seed, as a user's molecules are."""
    rng = np.random.default_rng(TOPOLOGY_SEED)
    if remd:
        chain = T.config0_chain(TOPOLOGY_SEED) if nt == 64 else _hairpin(rng, nt)
        return [T.build_rna_system([chain], tempk=t, ionic_strength=IONIC) for t in _temperatures(systems)], None
    if model == "coulomb":
        s = T.build_rna_system([(T.random_sequence(rng, nt), [])], ele_form=ELE_COULOMB, cutoff_ele=40.0,
                               phos_charge=-1.0)
        # cube side for the density of 160 nt in 60 A
        return [s], [T.compact_coords(s, rng, box=60.0 * (nt / 160.0) ** (1.0 / 3.0), min_dist=2.6)]
    if model == "ewald":
        n_mg, n_k = max(1, ions // 56), (54 * ions) // 100
        s, x = T.config2_ewald(TOPOLOGY_SEED, n=nt, box=box, n_mg=n_mg, n_k=n_k, n_cl=ions - n_mg - n_k,
                               alpha=0.1 if box >= 90.0 else 0.2, rcut=min(30.0, 0.45 * box), hmax=hmax)
        return [s], [x]
    if model == "valence":
        out, base = [], []
        for _ in range(systems):
            s = T.build_rna_system([(T.random_sequence(rng, nt), [])], all_pair_hbonds=True)
            out.append(s)
            base.append(T.compact_coords(s, rng, box=28.0, min_dist=2.4))
        return out, base
    if systems == 1:
        lengths = [nt]
    else:
        lengths = np.clip(np.rint(rng.lognormal(math.log(nt), 0.7, size=systems)), 20, 600).astype(int)
    chains = [T.config0_chain(TOPOLOGY_SEED) if systems == 1 and nt == 64 else _hairpin(rng, int(n)) for n in lengths]
    out = [T.build_rna_system([c], tempk=310.0, ionic_strength=IONIC) for c in chains]
    rep = T.config0_chain(TOPOLOGY_SEED)
    out += [T.build_rna_system([rep], tempk=t, ionic_strength=IONIC) for t in _temperatures(ladder)[:ladder]]
    return out, None


def _systems(case):
    return _topology(case["model"], case["systems"], case["nt"], case.get("ladder", 0), case.get("ions", 0),
                     case.get("box", 0.0), case.get("hmax", 0), case["kind"] == "remd")


def _coordinates(case, seed):
    """Extended helices near the native distances with noise on every bead
    (a few contacts among them), or the compact base coordinates with a small
    displacement per bead."""
    systems, base = _systems(case)
    rng = np.random.default_rng([seed, 1])
    if base is None:
        return systems, [T.helix_coords(s, rng, jitter=0.25, r_s=9.7, r_b=5.0) for s in systems]
    return systems, [x + rng.normal(0.0, 0.05, size=x.shape) for x in base]


def _rpy(x, radius, tempk, viscosity, device):
    """Rotne-Prager-Yamakawa tensor of equal beads that do not overlap or
    only touch (their overlap form included), (3n, 3n) FP64."""
    x = torch.as_tensor(x, dtype=torch.float64, device=device)
    n = len(x)
    a = float(radius)
    c6 = BOLTZ_KCAL_MOL * tempk / (6.0 * math.pi * viscosity)
    c8 = BOLTZ_KCAL_MOL * tempk / (8.0 * math.pi * viscosity)
    eye = torch.eye(3, dtype=torch.float64, device=device)
    D = torch.empty((n, 3, n, 3), dtype=torch.float64, device=device)
    for i in range(n):
        r = x - x[i]
        r2 = (r * r).sum(1)
        r2[i] = 1.0
        d = r2.sqrt()
        far1 = c8 / d * (1.0 + 2.0 * a * a / (3.0 * r2))
        far2 = c8 / d * (1.0 - 2.0 * a * a / r2) / r2
        near1 = c6 / a * (1.0 - 9.0 * d / (32.0 * a))
        near2 = c6 / a * 3.0 / (32.0 * a * d)
        far = d > 2.0 * a
        p1, p2 = torch.where(far, far1, near1), torch.where(far, far2, near2)
        p1[i], p2[i] = c6 / a, 0.0
        D[i] = (p1[:, None, None] * eye + p2[:, None, None] * r[:, :, None] * r[:, None, :]).permute(1, 0, 2)
    return D.reshape(3 * n, 3 * n)


@functools.lru_cache(maxsize=4)
def _chain(beads):
    return bead_spring_chain(beads, seed=TOPOLOGY_SEED % 1000 + beads)


def _chain_coordinates(case, seed):
    s, x = _chain(case["beads"])
    return s, x + np.random.default_rng([seed, 2]).normal(0.0, 0.1, size=x.shape)


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind == "factor":
        s, x = _chain_coordinates(case, seed)
        lib = load_library()
        fn = lib.tis_bdhi_factor_noalloc
        fn.restype = ctypes.c_int32
        fn.argtypes = [ctypes.c_int32, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int32, ctypes.c_void_p,
                       ctypes.c_void_p]
        D = _rpy(x, s.radius[0], s.tempk, s.viscosity, "cuda")
        return dict(kind=kind, fn=fn, D=D, L=torch.empty_like(D), n3=len(D))
    if kind == "bd":
        s, x = _chain_coordinates(case, seed)
        eng = BDEngine(s, key=case["beads"], seed=seed)
        eng.set_coords(x)
        return dict(kind=kind, eng=eng, steps=case["steps"], refactor_every=case["refactor_every"], done=0)
    systems, coords = _coordinates(case, seed)
    eng = Engine(systems, keys=list(range(len(systems))), seed=seed)
    state = dict(kind=kind, eng=eng, n=len(systems), coords=coords)
    if kind == "force":
        return state
    for k, x in enumerate(coords):
        eng.set_coords(k, x)
    if kind == "energy":
        rng = np.random.default_rng([seed, 3])
        for k, s in enumerate(systems):
            eng.set_state(k, 1, rng.normal(size=(s.nmp, 3)) * np.sqrt(BOLTZ_KCAL_MOL * s.tempk / s.mass)[:, None])
        eng.neighbor(-1)
        eng.force_sumup(0) if len(systems) == 1 else eng.force_all()
        return state
    if kind == "remd":
        state["ladder"] = ReplicaLadder(eng, list(range(len(systems))), systems[0], [s.tempk for s in systems],
                                        ionic_strength=IONIC, seed=seed)
    eng.langevin_init(tstep=TSTEP, rebuild_every=case["rebuild_every"])
    state["steps"] = case["steps"]
    return state


# ------------------------------------------------------------------ run
def run(state):
    kind = state["kind"]
    if kind == "factor":
        rc = state["fn"](0, state["D"].data_ptr(), state["L"].data_ptr(), state["n3"],
                         torch.cuda.current_stream().cuda_stream, None)
        if rc != 0:
            raise RuntimeError(f"factorisation failed ({rc})")
        # column-major on the device: the transposed view is L
        return state["L"].T
    eng = state["eng"]
    if kind == "bd":
        eng.steps(state["steps"], tstep=TSTEP, refactor_every=state["refactor_every"], step0=state["done"])
        state["done"] += state["steps"]
        return eng.coords()
    if kind == "force":
        for k, x in enumerate(state["coords"]):
            eng.set_coords(k, x)
        if state["n"] == 1:
            return eng.force_sumup(0)
        return np.concatenate(eng.force_all())
    if kind == "energy":
        return eng.energy_all()
    eng.langevin_steps(state["steps"])
    frame = np.concatenate([eng.coords(k) for k in range(state["n"])])
    if kind == "steps":
        return frame
    attempt = state["ladder"].attempt()
    return {"frame": frame, "delta": np.array([a[2] for a in attempt]),
            "accepted": np.array([a[3] for a in attempt]), "labels": np.array(state["ladder"].rep2lab)}


# ------------------------------------------------------------------ work
def work(case):
    """Inputs read once, results written once, and the arithmetic of one
    evaluation of every term (about 40 operations per electrostatic pair in
    the list, 30 / 80 / 400 / 600 per bond, angle, stack and hydrogen bond,
    150 per bead for contacts, noise and integrator) times the evaluations."""
    kind = case["kind"]
    if kind in ("factor", "bd"):
        n3 = 3 * case["beads"]
        if kind == "factor":
            return {"bytes": 16.0 * n3 * n3, "flops": n3 ** 3 / 3.0}
        refactors = -(-case["steps"] // case["refactor_every"])
        return {"bytes": 8.0 * 6 * n3 + 16.0 * n3 * n3 * refactors,
                "flops": refactors * (n3 ** 3 / 3.0 + 12.0 * n3 * n3) + 3.0 * n3 * n3 * case["steps"]}
    systems, base = _systems(case)
    beads = sum(s.nmp for s in systems)
    params = flops = 0.0
    for s in systems:
        nq = int((np.abs(s.charge) >= 1.0e-6).sum())
        pairs = nq * (nq - 1) / 2.0
        if case["model"] == "ewald":
            pairs *= min(1.0, 4.0 / 3.0 * math.pi * s.params.cutoff_ele ** 3 / case["box"] ** 3)
            flops += 4.0 / 3.0 * math.pi * case["hmax"] ** 3 * nq * 30.0
        params += 16 * len(s.bd_nat) + 20 * len(s.ba_nat) + 56 * len(s.st_mp) + 76 * len(s.hb_mp) + 32 * s.nmp
        flops += 40.0 * pairs + 30 * len(s.bd_nat) + 80 * len(s.ba_nat) + 400 * len(s.st_mp) + 600 * len(s.hb_mp)
        flops += 150.0 * s.nmp
    times = case.get("steps", 1)
    if kind == "remd":
        times += 2
    state = {"force": 48, "energy": 48}.get(kind, 144)
    return {"bytes": params + state * beads, "flops": flops * times}


# ------------------------------------------------------------------ exact
def _dihedral(a, b, axis, n1, n2):
    """Angle whose tangent is (v . n2) |axis| / (n1 . n2)."""
    return torch.atan2((a * n2).sum(1) * axis.norm(dim=1), (n1 * n2).sum(1))


def _wrapped(d):
    return d - 2.0 * math.pi * torch.round(d / (2.0 * math.pi))


def _angle_force(s, x, i):
    """Forces of the bond angles, sin^2 floored at 1 A^4 of the two bond
    lengths as the force field has it."""
    v21, v32 = x[i[:, 1]] - x[i[:, 0]], x[i[:, 2]] - x[i[:, 1]]
    c11, c22, c21 = (v21 * v21).sum(1), (v32 * v32).sum(1), (v32 * v21).sum(1)
    th = torch.acos(-c21 / (c11 * c22).sqrt())
    sin2 = (c11 * c22 - c21 ** 2).clamp(min=1.0)
    fr = 2.0 * torch.as_tensor(s.ba_coef) * (th - torch.as_tensor(s.ba_nat)) / sin2.sqrt()
    f21 = fr[:, None] * (v21 * (c21 / c11)[:, None] - v32)
    f32 = fr[:, None] * (v32 * (c21 / c22)[:, None] - v21)
    F = torch.zeros_like(x)
    for k, f in enumerate((-f21, f21 - f32, f32)):
        F.index_add_(0, i[:, k], f)
    return F


def _bonded(s, x):
    """Energies of bonds, angles, stacks and hydrogen bonds (FP64)."""
    cross, t = torch.linalg.cross, torch.as_tensor
    zero = x.sum() * 0.0
    e = {E_BOND: zero, E_BANGLE: zero, E_STACK: zero, E_HBOND: zero}
    i = t(s.bd_mp, dtype=torch.long).reshape(-1, 2)
    e[E_BOND] = (t(s.bd_coef) * ((x[i[:, 1]] - x[i[:, 0]]).norm(dim=1) - t(s.bd_nat)) ** 2).sum()
    i = t(s.ba_mp, dtype=torch.long).reshape(-1, 3)
    if len(i):
        v21, v32 = x[i[:, 1]] - x[i[:, 0]], x[i[:, 2]] - x[i[:, 1]]
        th = torch.acos(-(v21 * v32).sum(1) / (v21.norm(dim=1) * v32.norm(dim=1)))
        e[E_BANGLE] = (t(s.ba_coef) * (th - t(s.ba_nat)) ** 2).sum()
    i = t(s.st_mp, dtype=torch.long).reshape(-1, 7)
    if len(i):
        nat, cf = t(s.st_nat).reshape(-1, 3), t(s.st_coef).reshape(-1, 4)
        b1, b2, p1, s1, p2, s2, p3 = (x[i[:, k]] for k in range(7))
        v34, v54, v56, v76 = p1 - s1, p2 - s1, p2 - s2, p3 - s2
        m, n = cross(v34, v54), cross(v54, v56)
        phi1 = _dihedral(v34, v54, v54, m, n)
        phi2 = _dihedral(v76, v56, v56, cross(v76, v56), -n)
        div = (1.0 + cf[:, 1] * ((b2 - b1).norm(dim=1) - nat[:, 0]) ** 2
               + cf[:, 2] * _wrapped(phi1 - nat[:, 1]) ** 2 + cf[:, 3] * _wrapped(phi2 - nat[:, 2]) ** 2)
        e[E_STACK] = (cf[:, 0] / div).sum()
    i = t(s.hb_mp, dtype=torch.long).reshape(-1, 6)
    if len(i):
        d = (x[i[:, 0]] - x[i[:, 1]]).norm(dim=1) - t(s.hb_nat).reshape(-1, 6)[:, 0]
        near = d.abs() <= s.params.hb_cutoff_dist
        i, d = i[near], d[near]
        nat, cf = t(s.hb_nat).reshape(-1, 6)[near], t(s.hb_coef).reshape(-1, 7)[near]
        b1, b2, s1, s2, p1, p2 = (x[i[:, k]] for k in range(6))
        v12, v13, v53, v42, v46 = b1 - b2, b1 - s1, p1 - s1, s2 - b2, s2 - p2
        angle = lambda a, b: torch.acos((a * b).sum(1) / (a.norm(dim=1) * b.norm(dim=1)))  # noqa: E731
        m, n = cross(v42, v12), cross(v12, v13)
        u, w = cross(v53, v13), cross(v42, v46)
        dih = (_dihedral(v42, v12, v12, m, n), _dihedral(v53, v13, v13, u, -n), _dihedral(v12, v42, v42, -m, w))
        ex = -cf[:, 1] * d ** 2 - cf[:, 2] * (angle(v12, v13) - nat[:, 1]) ** 2 \
            - cf[:, 3] * (angle(v12, v42) - nat[:, 2]) ** 2
        for k in range(3):
            ex = ex - cf[:, 4 + k] * _wrapped(dih[k] - nat[:, 3 + k]) ** 2
        e[E_HBOND] = (cf[:, 0] * torch.exp(ex)).sum()
    return e


def _pairs(s, x):
    """(energies, forces) of contacts and electrostatics, every pair once."""
    p, n = s.params, s.nmp
    F = torch.zeros_like(x)
    e = {}
    # contacts: pairs closer than their distance D
    kind = torch.as_tensor(np.asarray(s.mptype), dtype=torch.long)
    sep = torch.full((n,), p.n_sep_B)
    sep[kind == MP_PHOS] = p.n_sep_P
    sep[kind == MP_SUGAR] = p.n_sep_S
    i, j = (torch.cdist(x, x) <= max(p.exv_dist, p.exv_dist_PS) + 1.0e-6).nonzero(as_tuple=True)
    keep = j >= i + sep[i]
    i, j = i[keep], j[keep]
    v = x[j] - x[i]
    d = v.norm(dim=1)
    ps = (kind[i] == MP_PHOS) & (kind[j] == MP_SUGAR) | (kind[i] == MP_SUGAR) & (kind[j] == MP_PHOS)
    D = torch.where(ps, p.exv_dist_PS, p.exv_dist).to(torch.float64)
    keep = d <= D
    i, j, v, d, D = i[keep], j[keep], v[keep], d[keep], D[keep]
    eps = torch.as_tensor(s.exv_eps)
    c = eps[i] * eps[j]
    r = d + p.exv_adjust - D
    q6 = (p.exv_adjust / r) ** 6
    e[E_EXV] = (c * (q6 * q6 - 2.0 * q6 + 1.0)).sum()
    f = (12.0 * c * (q6 * q6 - q6).abs() / r.abs() / d).clamp(max=T.DE_MAX)[:, None] * v
    F.index_add_(0, i, -f)
    F.index_add_(0, j, f)
    # electrostatics of the charged beads
    charge = torch.as_tensor(s.charge)
    qb = (charge.abs() >= 1.0e-6).nonzero()[:, 0]
    i, j = torch.triu_indices(len(qb), len(qb), 1)
    i, j = qb[i], qb[j]
    v = x[j] - x[i]
    d = v.norm(dim=1)
    qq = charge[i] * charge[j] * p.ele_coef
    if p.ele_form == ELE_DH:
        lam = p.ele_cdist
        cut = p.cutoff_ele * lam
        yuk = torch.exp(-d / lam) / d
        e[E_ELE] = torch.where(d <= cut, qq * yuk, 0.0).sum()
        f = (qq * yuk * (1.0 / d + 1.0 / lam) / d).clamp(max=T.DE_MAX)
    else:
        cut = p.cutoff_ele
        e[E_ELE] = torch.where(d <= cut, qq * (1.0 / d - 1.0 / cut), 0.0).sum()
        f = qq / d ** 3
    f = torch.where(d <= cut, f, 0.0)[:, None] * v
    F.index_add_(0, i, -f)
    F.index_add_(0, j, f)
    return e, F


def exact(case, seed):
    """Forces, energies and factors in 64 bits; None for trajectories, whose
    noise and rounding are the program's own."""
    kind = case["kind"]
    if kind == "factor":
        s, x = _chain_coordinates(case, seed)
        return torch.linalg.cholesky(_rpy(x, s.radius[0], s.tempk, s.viscosity, "cpu"))
    if kind not in ("force", "energy"):
        return None
    systems, coords = _coordinates(case, seed)
    rng = np.random.default_rng([seed, 3])
    out = []
    for s, x in zip(systems, coords):
        x = torch.as_tensor(x).requires_grad_(kind == "force")
        terms = _bonded(s, x)
        pair_terms, F = _pairs(s, x.detach())
        if kind == "force":
            F += _angle_force(s, x.detach(), torch.as_tensor(s.ba_mp, dtype=torch.long).reshape(-1, 3))
            smooth = sum(v for k, v in terms.items() if k != E_BANGLE)
            out.append((F - torch.autograd.grad(smooth, x)[0]).numpy())
            continue
        e = np.zeros(E_MAX)
        for k, v in {**terms, **pair_terms}.items():
            e[k] = float(v)
        e[E_TOTAL] = e.sum()
        v = rng.normal(size=(s.nmp, 3)) * np.sqrt(BOLTZ_KCAL_MOL * s.tempk / s.mass)[:, None]
        e[E_VELO] = float((0.5 * s.mass[:, None] * v * v).sum())
        out.append(e)
    return np.concatenate(out) if kind == "force" else np.array(out)
