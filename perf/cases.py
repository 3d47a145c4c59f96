"""The work that users of this framework have it do, as cases that can be timed and compared.

Each case goes through the public front end (``faunus_amd.Engine``, ``Batch`` and ``Server``):
the per-move boundary that a host Metropolis loop calls, single chains on one workgroup and
on several, temperature ladders of ions and of water, a polyelectrolyte, a serving loop and
the resume of a checkpoint with its energy and pair-distance histogram.  The systems are those
of the benchmark and the tests, at their own sizes and over the ranges around them.

``exact`` follows the same moves in 64-bit torch on the host, from the formulas alone: the
Philox proposals, pair energies (with their splines), the Ewald sum and the Metropolis rule.
"""
import itertools
import math

import numpy as np
import torch

import faunus_amd as F

AVOGADRO = 6.022137e23
TEMPERATURE = 298.15
KT = TEMPERATURE * 1.380658e-23


# ---------------------------------------------------------------------------------- cases
def listed():
    return [
        # a host program's own Metropolis loop on the smallest system of the tests (200 ions of
        # the primitive model): one energy change per call, where launch latency is everything
        dict(name="permove_ions_200", kind="permove", system="ions", n=200, moves=192),
        # the same loop on the benchmark's large system (cell list, K = 17328)
        dict(name="permove_nacl_20k", kind="permove", system="nacl", n=20000, moves=128),
        # the same loop with rigid molecules (three moved atoms, group cutoff)
        dict(name="permove_water_1000", kind="permove", system="water", n=1000, moves=128),
        # a short chain of a small system on the device, one workgroup, FP64
        dict(name="chain_ions_200", kind="chain", system="ions", n=200, replicas=1, fp32=False, moves=800),
        # the benchmark's headline: one large chain shared by 16 workgroups, FP64
        dict(name="split_nacl_20k", kind="split", system="nacl", n=20000, groups=16, fp32=False, moves=3000),
        # temperature ladders of a 2:1 salt, free-running with swaps, FP32 pairs: the batched
        # form of the benchmark, four compositions over its range of sizes
        dict(name="ladder_salt_fp32", kind="ladder", system="salt", n=8571, compositions=4, rungs=12, fp32=True,
             moves=800),
        # one small ladder in FP64
        dict(name="ladder_salt_fp64", kind="ladder", system="salt", n=1203, compositions=1, rungs=8, fp32=False,
             moves=400),
        # a ladder of 4096 waters as the reference's example writes them (group cutoff, the finer
        # cell grid that the autotuner picks), FP32 pairs, one round of swaps after the launch
        dict(name="water_ladder_fp32", kind="water", system="water", n=4096, replicas=8, divisions=2, fp32=True,
             moves=300),
        # the tests' splined and cut water in FP64 on the default grid
        dict(name="water_splined_fp64", kind="water", system="water_cut", n=1728, replicas=4, divisions=1, fp32=False,
             moves=200),
        # one polyelectrolyte with ion and bead translations and pivots, shared by 16 workgroups
        dict(name="polymer_split_fp32", kind="polymer", n=10001, beads=350, groups=16, fp32=True, moves=1000),
        # a serving loop: a few polyelectrolyte jobs of the job stream's small sizes, submitted
        # and stepped until all are done
        dict(name="serve_polymer", kind="serve", n=3000, jobs=4, fp32=True, moves=400),
        # a checkpoint resumed (Q(k), cell list and energy rebuilt), its energy checked against a
        # full recompute, and one sample of g(r)
        dict(name="resume_nacl_20k", kind="resume", system="nacl", n=20000, bins=240),
    ]


def _log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["permove", "permove", "chain", "split", "ladder", "water", "polymer", "serve", "resume"])
    if kind == "permove":
        system = rng.choice(["ions", "nacl", "water"])
        n = {"ions": lambda: 2 * _log_size(rng, 20, 1000), "nacl": lambda: 2 * _log_size(rng, 700, 10000),
             "water": lambda: _log_size(rng, 216, 4096)}[system]()
        return dict(kind=kind, system=system, n=n, moves=rng.randint(64, 128))
    if kind == "chain":
        return dict(kind=kind, system=rng.choice(["ions", "nacl"]), n=2 * _log_size(rng, 50, 1500),
                    replicas=rng.randint(1, 6), fp32=rng.random() < 0.5, moves=rng.randint(100, 400))
    if kind == "split":
        return dict(kind=kind, system="nacl", n=2 * _log_size(rng, 1000, 10000), groups=rng.choice([12, 16, 24, 32]),
                    fp32=False, moves=rng.randint(500, 2000))
    if kind == "ladder":
        return dict(kind=kind, system="salt", n=3 * _log_size(rng, 200, 2850), compositions=rng.randint(1, 3),
                    rungs=rng.randint(2, 10), fp32=rng.random() < 0.7, moves=rng.randint(50, 200))
    if kind == "water":
        return dict(kind=kind, system=rng.choice(["water", "water", "water_cut"]), n=_log_size(rng, 400, 4096),
                    replicas=rng.randint(1, 8), divisions=rng.choice([1, 2]), fp32=rng.random() < 0.7,
                    moves=rng.randint(50, 200))
    if kind == "polymer":
        beads = _log_size(rng, 50, 350)
        return dict(kind=kind, n=max(2 * beads + 20, _log_size(rng, 1000, 10000)), beads=beads,
                    groups=rng.choice([1, 2, 4, 8, 16, 32]), fp32=rng.random() < 0.7, moves=rng.randint(100, 400))
    if kind == "serve":
        return dict(kind=kind, n=_log_size(rng, 1000, 3000), jobs=rng.randint(1, 4), fp32=True,
                    moves=rng.randint(100, 400))
    return dict(kind="resume", system="nacl", n=2 * _log_size(rng, 700, 10000), bins=rng.randint(50, 400))


# -------------------------------------------------------------------------------- systems
def _sites(n, box, core, rng):
    """n points no closer than `core`: random sites of a cubic lattice, jittered."""
    m = math.ceil(n ** (1.0 / 3.0))
    a = box / m
    pick = rng.choice(m ** 3, size=n, replace=False)
    ijk = np.stack([pick % m, (pick // m) % m, pick // (m * m)], axis=1) + 0.5
    return ijk * a - box / 2 + max(0.0, a - core) / 2 * (2 * rng.random((n, 3)) - 1)


def _ewald(epsr, cutoff, alpha, kmax):
    return {"coulomb": {"type": "ewald", "epsr": epsr, "cutoff": cutoff, "alpha": alpha, "ncutoff": kmax}}


def _ion_system(name, n, rng, conc=0.1):
    """Ions in one atomic group: `ions` (1:1, hard spheres), `nacl` (Lennard-Jones, splined and
    cut at 11.99 A) or `salt` (2:1, hard spheres, real space cut at half the box)."""
    if name == "salt":
        n -= n % 3
        box = ((n / 3) / (conc * AVOGADRO * 1e-27)) ** (1.0 / 3.0)
        charge, sigma, eps, dp = (2.0, -1.0), (4.0, 4.0), (0.0, 0.0), 0.2 * box
        ids = np.tile(np.array([0, 1, 1], np.int32), n // 3)
        epsr, rc, alpha, kmax = 78.7, box / 2, 5.0 / box, 8
    else:
        ids = np.tile(np.array([0, 1], np.int32), n // 2)
        charge = (1.0, -1.0)
        if name == "ions":
            box, sigma, eps, dp = 118.0 * (n / 200) ** (1.0 / 3.0), (4.0, 4.0), (0.0, 0.0), 10.0
            epsr, rc, alpha, kmax = 78.7, min(30.0, 0.49 * box), 0.2, 7
        else:
            box, sigma, eps, dp = 255.0 * (n / 20000) ** (1.0 / 3.0), (3.3, 4.4), (0.5, 0.4), 2.0
            epsr, rc, alpha, kmax = 78.7, 12.0, 0.25, max(6, round(20 * box / 255.0))
    atoms = [{k: {"q": charge[t], "sigma": sigma[t], "eps": eps[t], "dp": dp}} for t, k in enumerate(("A", "B"))]
    terms = [{"lennardjones": {"mixing": "LB"}} if name == "nacl" else {"hardsphere": {}}]
    terms.append(_ewald(epsr, rc, alpha, kmax))
    nonbonded = {"default": terms}
    if name == "nacl":
        nonbonded.update(rmax=11.99, u_at_rmax=0.1)
    cfg = {"temperature": TEMPERATURE, "geometry": {"type": "cuboid", "length": box}, "atomlist": atoms,
           "moleculelist": [{"salt": {"atoms": ["A", "B"], "atomic": True}}],
           "energy": [{"nonbonded_splined" if name == "nacl" else "nonbonded": nonbonded}]}
    xyz = _sites(n, box, 0.9 * max(sigma) if name == "nacl" else max(sigma), rng)
    q = np.array(charge)[ids]
    phys = dict(box=box, charge=charge, sigma=sigma, eps=eps, epsr=epsr, rc=rc, alpha=alpha, kmax=kmax, dp=dp,
                hard=name != "nacl", cut=11.99 if name == "nacl" else None, g2g=None)
    return dict(system=(cfg, xyz, q, ids, dict(begin=[0], size=[n], molid=[0])), kinds=None, phys=phys)


def _water_system(name, n_mol, rng):
    """Rigid three-site water at liquid density: `water` with the group cutoff of the
    reference's example, `water_cut` with the pair energy splined and cut."""
    box = 49.68 * (n_mol / 4096) ** (1.0 / 3.0)
    large = n_mol > 2000
    alpha, rc, kmax, g2g = (0.28, 10.0, 9, 10.0) if large or name == "water_cut" else (0.2, 9.0, 7, 10.0)
    rc, g2g = min(rc, 0.49 * box), min(g2g, 0.49 * box)
    charge, sigma, eps, mass = (-0.8476, 0.4238), (3.166, 2.0), (0.650, 0.0), (15.999, 1.008)
    pairs = _ewald(1.0, rc, alpha, kmax)
    if name == "water":
        energy = [{"nonbonded_coulomblj": {"lennardjones": {"mixing": "LB"}, **pairs, "cutoff_g2g": g2g}}]
    else:
        energy = [{"nonbonded_splined": {"default": [{"lennardjones": {"mixing": "LB"}}, pairs], "rmax": rc - 0.01,
                                         "u_at_rmax": 0.1}}]
    cfg = {"temperature": TEMPERATURE, "geometry": {"type": "cuboid", "length": box},
           "atomlist": [{k: {"q": charge[t], "sigma": sigma[t], "eps": eps[t], "mw": mass[t]}}
                        for t, k in enumerate(("OW", "HW"))],
           "moleculelist": [{"water": {"atoms": ["OW", "HW", "HW"], "rigid": True}}], "energy": energy}
    theta = math.radians(109.47)
    local = np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [math.cos(theta), math.sin(theta), 0.0]])
    v = rng.normal(size=(n_mol, 2, 3))
    e0 = v[:, 0] / np.linalg.norm(v[:, 0], axis=1)[:, None]
    e1 = v[:, 1] - (v[:, 1] * e0).sum(1)[:, None] * e0
    e1 /= np.linalg.norm(e1, axis=1)[:, None]
    frame = np.stack([e0, e1, np.cross(e0, e1)], axis=1)
    m = math.ceil(n_mol ** (1.0 / 3.0))
    xyz = _sites(n_mol, box, box / m, rng)[:, None, :] + local @ frame
    xyz = (xyz - box * np.round(xyz / box)).reshape(-1, 3)
    ids = np.tile(np.array([0, 1, 1], np.int32), n_mol)
    q = np.array(charge)[ids]
    groups = dict(begin=list(range(0, 3 * n_mol, 3)), size=[3] * n_mol, molid=[0] * n_mol)
    phys = dict(box=box, charge=charge, sigma=sigma, eps=eps, epsr=1.0, rc=rc, alpha=alpha, kmax=kmax, mass=mass,
                hard=False, cut=rc - 0.01 if name == "water_cut" else None, g2g=g2g if name == "water" else None,
                dp=0.5, dprot=0.5)
    kinds = [dict(kind=1, molid=0, weight=1, dp=0.5, dprot=0.5)]
    return dict(system=(cfg, xyz, q, ids, groups), kinds=kinds, phys=phys)


def _polymer_system(n_beads, n_total, rng):
    """A bead-spring chain (q = -1, harmonic bonds) with counterions and 1:1 salt at 5 mM of
    monomer, hard spheres + Ewald; ion and bead translations and pivots."""
    n_salt = max(0, (n_total - 2 * n_beads) // 2)
    n_ions = n_beads + 2 * n_salt
    box = (n_beads / (0.005 * AVOGADRO * 1e-27)) ** (1.0 / 3.0)
    bonds = [{"harmonic": {"index": [i, i + 1], "k": 0.5, "req": 4.0}} for i in range(n_beads - 1)]
    cfg = {"temperature": TEMPERATURE, "geometry": {"type": "cuboid", "length": box},
           "atomlist": [{"P": {"q": -1.0, "sigma": 4.0, "dp": 2.0}}, {"C": {"q": 1.0, "sigma": 4.0, "dp": 10.0}},
                        {"A": {"q": -1.0, "sigma": 4.0, "dp": 10.0}}],
           "moleculelist": [{"chain": {"atoms": ["P"] * n_beads, "bondlist": bonds}},
                            {"ions": {"atoms": ["C", "A"], "atomic": True}}],
           "energy": [{"bonded": {}},
                      {"nonbonded": {"default": [{"hardsphere": {}}, _ewald(78.7, box / 2, 5.0 / box, 8)]}}]}
    chain = np.zeros((n_beads, 3))
    back, i = np.zeros(3), 1
    while i < n_beads:
        v = rng.normal(size=3)
        v /= np.linalg.norm(v)
        p = chain[i - 1] + 4.2 * v
        if v @ back >= -0.25 and (((chain[:i - 1] - p) ** 2).sum(1) >= 4.4 ** 2).all():
            chain[i], back, i = p, v, i + 1
    chain -= chain.mean(axis=0)
    chain -= box * np.round(chain / box)
    free = _sites(min(4 * n_ions, 3 * n_ions + 4000), box, 4.0, rng)
    near = np.zeros(len(free), bool)
    for b in chain:
        d = free - b
        d -= box * np.round(d / box)
        near |= (d * d).sum(1) < 4.4 ** 2
    ions = free[~near][:n_ions]
    ids = np.concatenate([np.zeros(n_beads, np.int32), np.ones(n_beads + n_salt, np.int32),
                          np.full(n_salt, 2, np.int32)])
    q = np.where(ids == 1, 1.0, -1.0)
    groups = dict(begin=[0, n_beads], size=[n_beads, n_ions], molid=[0, 1])
    kinds = [dict(kind=0, molid=1, weight=n_ions, dp=10.0), dict(kind=0, molid=0, weight=n_beads, dp=2.0),
             dict(kind=2, molid=0, weight=max(1, n_beads - 1), dprot=3.0)]
    return dict(system=(cfg, np.concatenate([chain, ions]), q, ids, groups), kinds=kinds)


def _inputs(case, seed):
    """The systems of a case and what else its program has at hand, from the seed alone."""
    rng = np.random.default_rng([seed, 11])
    kind, n = case["kind"], case["n"]
    if kind == "polymer":
        return dict(systems=[_polymer_system(case["beads"], n, rng)])
    if kind == "serve":
        sizes = [max(300, round(n * (0.4 + 0.6 * (j + 1) / case["jobs"]))) for j in range(case["jobs"])]
        return dict(systems=[_polymer_system(50 + 17 * j, s, rng) for j, s in enumerate(sizes)])
    if case["system"].startswith("water"):
        count = min(case.get("replicas", 1), 4)
        systems = [_water_system(case["system"], n, rng) for _ in range(count)]
        if kind == "permove":
            systems[0]["stream"] = _molecule_stream(systems[0], case["moves"], rng)
        return dict(systems=systems)
    if kind == "ladder":
        # compositions from a seventh of n up to n, at 0.01 to 1 M
        sizes = [max(60, int(n * (1 + 6 * c / max(1, case["compositions"] - 1)) / 7)) if case["compositions"] > 1 else n
                 for c in range(case["compositions"])]
        return dict(systems=[_ion_system("salt", s, rng, conc=float(10 ** rng.uniform(-2, 0))) for s in sizes])
    s = _ion_system(case["system"], n, rng)
    if kind == "permove":
        m = case["moves"]
        v = rng.normal(size=(m, 3))
        v *= (s["phys"]["dp"] * rng.random(m) / np.linalg.norm(v, axis=1))[:, None]
        s["stream"] = dict(group=np.zeros(m, np.int32), index=rng.integers(0, n, m).astype(np.int32), shift=v,
                           uniform=rng.random(m))
    if kind == "resume":
        # the configuration to resume: every ion a little away from the replica's own
        xyz = s["system"][1] + 0.4 * (2 * rng.random((n, 3)) - 1)
        s["checkpoint"] = dict(xyz=xyz - s["phys"]["box"] * np.round(xyz / s["phys"]["box"]), mass_center=None,
                               moves=n, accepted=n // 2)
    return dict(systems=[s])


def _molecule_stream(s, m, rng):
    """Trial coordinates of m rigid translate+rotate moves, each of another molecule."""
    _, xyz, _, ids, g = s["system"]
    box, dp, mass = s["phys"]["box"], s["phys"]["dp"], np.array(s["phys"]["mass"])
    m = min(m, len(g["begin"]))
    mol = rng.choice(len(g["begin"]), size=m, replace=False).astype(np.int32)
    atoms = 3 * mol[:, None] + np.arange(3)
    p = xyz[atoms]
    rel = p - p[:, :1]
    rel -= box * np.round(rel / box)
    w = mass[ids[:3]][None, :, None] / mass[ids[:3]].sum()
    cm = p[:, 0] + (w * rel).sum(1)
    rel -= (w * rel).sum(1)[:, None]
    axis = rng.normal(size=(m, 3))
    axis /= np.linalg.norm(axis, axis=1)[:, None]
    angle = (0.5 * (rng.random(m) - 0.5))[:, None, None]
    a = np.broadcast_to(axis[:, None], rel.shape)
    rel = rel * np.cos(angle) + np.cross(a, rel) * np.sin(angle) + a * (a * rel).sum(2)[..., None] * (1 - np.cos(angle))
    shift = rng.normal(size=(m, 3))
    cm = cm + shift * (dp * rng.random(m) / np.linalg.norm(shift, axis=1))[:, None]
    new = cm[:, None] + rel
    return dict(group=mol, offsets=3 * np.arange(m + 1, dtype=np.int64), index=atoms.ravel().astype(np.int32),
                xyz=(new - box * np.round(new / box)).reshape(-1, 3), uniform=rng.random(m),
                mass_center=cm - box * np.round(cm / box), whole=np.ones(m, np.uint8))


# ------------------------------------------------------------------------ prepare and run
def prepare(case, seed):
    given = _inputs(case, seed)
    systems, kind = given["systems"], case["kind"]
    state = dict(case=case, systems=systems, calls=0)
    if kind == "permove":
        cfg, xyz, q, ids, g = systems[0]["system"]
        eng = F.Engine(cfg)
        eng.set_particles(xyz, q, ids)
        eng.set_groups(g["begin"], g["size"], g["molid"])
        eng.init()
        state["engine"] = eng
    elif kind == "serve":
        state["server"] = F.Server(fp32_pairs=case["fp32"], split_atoms=512, max_parts=16)
    else:
        batch = F.Batch(fp32_pairs=case.get("fp32", False), cell_divisions=case.get("divisions", 1))
        for r in _replicas(case, given):
            batch.add(r["system"], beta=r["beta"], seed=r["seed"], ladder=r["ladder"], moves=r["kinds"])
        state["batch"] = batch
        state["moves"] = [r["moves"] for r in _replicas(case, given)]
    return state


def _replicas(case, given):
    """The replicas of a batched case: system, temperature, random stream and moves per launch."""
    systems, kind = given["systems"], case["kind"]
    out = []
    if kind == "ladder":
        # equal work per rung: moves inversely proportional to the cost of one
        top = max(len(s["system"][2]) for s in systems) + 2304.0
        temps = np.linspace(280.0, 360.0, case["rungs"])
        for c, s in enumerate(systems):
            moves = round(case["moves"] * top / (len(s["system"][2]) + 2304.0))
            out += [dict(system=s["system"], phys=s["phys"], kinds=None, beta=TEMPERATURE / t, ladder=c, moves=moves,
                         seed=1000 + 100 * c + k) for k, t in enumerate(temps)]
        return out
    count = case.get("replicas", 1)
    temps = np.linspace(280.0, 360.0, count) if kind == "water" and count > 1 else [TEMPERATURE] * count
    for r in range(count):
        s = systems[r % len(systems)]
        out.append(dict(system=s["system"], phys=s.get("phys"), kinds=s["kinds"], beta=TEMPERATURE / temps[r],
                        ladder=0 if kind == "water" and count > 1 else -1, moves=case.get("moves", 0), seed=9000 + r))
    return out


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    call = state["calls"]
    state["calls"] += 1
    if kind == "permove":
        eng, s = state["engine"], state["systems"][0]["stream"]
        if case["system"] == "water":
            du, acc = eng.replay_moves(s["group"], s["offsets"], s["index"], s["xyz"], s["uniform"], whole=s["whole"],
                                       mass_center=s["mass_center"])
        else:
            du, acc = eng.run_translate(s["group"], s["index"], s["shift"], s["uniform"])
        return dict(du=du, accepted=acc, positions=eng.positions())
    if kind == "serve":
        server = state["server"]
        jobs = [server.submit(s["system"], case["moves"], seed=50 + j, kinds=s["kinds"])
                for j, s in enumerate(state["systems"])]
        while any(server.job(j)["state"] not in (F.Server.DONE, F.Server.FAILED) for j in jobs):
            server.step()
        done = [server.job(j) for j in jobs]
        return dict(energy=np.array([d["energy"] for d in done]), accepted=np.array([d["accepted"] for d in done]),
                    positions=np.concatenate([server.positions(j) for j in jobs]))
    batch = state["batch"]
    if kind == "resume":
        ck = state["systems"][0]["checkpoint"]
        batch.set_state(0, ck)
        total, terms = batch.total_energy(0)
        counts = batch.rdf(0, 0, 1, 24.0 / case["bins"], case["bins"])
        return dict(energy=batch.info(0)["energy"], total=total, terms=terms[:3], rdf=counts.astype(np.int64),
                    positions=batch.positions(0))
    if kind in ("split", "polymer"):
        batch.run_split(case["moves"], groups=case["groups"])
    elif kind == "ladder":
        batch.run_ladders(state["moves"], 2, seed=4242, round0=2 * call)
    else:
        batch.run(state["moves"])
        if kind == "water" and len(state["moves"]) > 1:
            batch.swap(seed=77, rnd=call)
    infos = [batch.info(r) for r in range(len(state["moves"]))]
    return dict(energy=np.array([i["energy"] for i in infos]), beta=np.array([i["beta"] for i in infos]),
                accepted=np.array([i["accepted"] for i in infos], np.int64),
                positions=np.concatenate([batch.positions(r) for r in range(len(infos))]))


def _kcount(kmax):
    r = np.arange(-kmax, kmax + 1)
    n2 = (r * r)[:, None, None] + (r * r)[:, None] + r * r
    return (int((n2 <= kmax * kmax).sum()) - 1 + int(((r * r)[:, None] + r * r <= kmax * kmax).sum()) - 1) // 2


def work(case):
    """One pass: particles (coordinates, charge, type) and structure factors read once and written
    once; per move 27 flops for each pair of a moved atom in both states within the interaction's
    reach and 2m(7 + 20) + 8 per k-vector."""
    kind, n = case["kind"], case["n"]
    if kind in ("polymer", "serve"):
        beads = case.get("beads", 50)
        jobs = case.get("jobs", 1)
        atoms, box = n, (beads / (0.005 * AVOGADRO * 1e-27)) ** (1.0 / 3.0)
        k = _kcount(8)
        moved = (atoms - beads + beads + beads * beads / 2) / (atoms + beads)
        flops = case["moves"] * (2 * moved * atoms * math.pi / 6 * 27 + (54 * moved + 8) * k)
        return {"bytes": jobs * (64.0 * atoms + 32.0 * k), "flops": jobs * flops}
    p = (_water_system if case["system"].startswith("water") else _ion_system)(
        case["system"], n if not case["system"].startswith("water") else min(n, 64), np.random.default_rng(0))["phys"]
    k = _kcount(p["kmax"])
    atoms = n
    if case["system"].startswith("water"):
        p = dict(p, box=49.68 * (n / 4096) ** (1.0 / 3.0), rc=10.0)
        k, atoms = _kcount(9 if n > 2000 or p["cut"] else 7), 3 * n
    reach = atoms * min(1.0, 4 / 3 * math.pi * (p["g2g"] or p["cut"] or p["rc"]) ** 3 / p["box"] ** 3)
    m = 3 if case["system"].startswith("water") else 1
    if kind == "resume":
        return {"bytes": 3 * 32.0 * atoms + 32.0 * k, "flops": 2 * 27 * atoms * reach / 2 + 8.0 * atoms * k}
    replicas, moves = case.get("replicas", 1), case.get("moves", 0)
    if kind == "ladder":
        replicas, moves = case["compositions"] * case["rungs"], 2 * moves
    flops = moves * (2 * m * reach * 27 + (54 * m + 8) * k)
    return {"bytes": replicas * (64.0 * atoms + 32.0 * k), "flops": replicas * flops}


# ---------------------------------------------------------------------------------- exact
def _andrea(f, xmin, xmax, utol, ftol=None):
    """The adaptive quintic spline of f(x) on [xmin, xmax] (Andrea, Swope and Andersen): from
    the top, intervals in sqrt(x) are shrunk until 11 points lie within utol (and the slope
    within ftol).  Returns the knots and six coefficients per interval."""
    h = 1e-4

    def d1(x):
        return (f(x + 0.5 * h) - f(x - 0.5 * h)) / h

    def d2(x):
        return (d1(x + 0.5 * h) - d1(x - 0.5 * h)) / h

    low, top = math.sqrt(xmin), math.sqrt(xmax)
    knots, coeff = [top * top], []
    while True:
        width = top - low
        while True:
            r = max(top - width, low)
            x0, x1 = r * r, top * top
            f0, f1, f2, d = f(x0), d1(x0), d2(x0), x1 - x0
            if abs(f0) < 1e-9 and abs(f1) < 1e-9:
                c = [0.0] * 6
            else:
                a = 6 * (f(x1) - f0 - f1 * d - 0.5 * f2 * d * d) / d ** 3
                b = 2 * (d1(x1) - f1 - f2 * d) / d ** 2
                e = (d2(x1) - f2) / d
                c = [f0, f1, 0.5 * f2, (10 * a - 12 * b + 3 * e) / 6, (-15 * a + 21 * b - 6 * e) / (6 * d),
                     (2 * a - 3 * b + e) / (2 * d * d)]
            good = True
            for j in range(11):
                y = (r + (top - r) / 10.0 * j) ** 2
                z = y - x0
                u = c[0] + z * (c[1] + z * (c[2] + z * (c[3] + z * (c[4] + z * c[5]))))
                s = c[1] + z * (2 * c[2] + z * (3 * c[3] + z * (4 * c[4] + z * 5 * c[5])))
                if abs(u - f(y)) > utol or (ftol is not None and abs(s - d1(y)) > ftol):
                    good = False
                    break
            if good:
                break
            width *= 0.9
        knots.append(r * r)
        coeff.append(c)
        top = r
        if r <= low:
            return torch.tensor(knots[::-1], dtype=torch.float64), torch.tensor(coeff[::-1], dtype=torch.float64)


def _spline(table, x):
    knots, coeff = table
    i = (torch.searchsorted(knots, x) - 1).clamp(0, len(knots) - 2)
    c, z = coeff[i], x - knots[i]
    u = c[..., 5]
    for j in (4, 3, 2, 1, 0):
        u = u * z + c[..., j]
    return u


class _Model:
    """Energies of one system in 64 bits: pairs, the Ewald sum and the self energy."""

    def __init__(self, phys):
        self.p = p = phys
        kj = 1e3 / (AVOGADRO * KT)
        self.lb = 1.602177e-19 ** 2 / (4 * math.pi * 8.85419e-12 * p["epsr"] * 1e-10 * KT)
        s = p["sigma"]
        self.s2 = [[((s[a] + s[b]) / 2) ** 2 for b in (0, 1)] for a in (0, 1)]
        self.e4 = [[0.0 if p["hard"] else 4 * kj * math.sqrt(p["eps"][a] * p["eps"][b]) for b in (0, 1)] for a in (0, 1)]
        self.short = _andrea(lambda x: math.erfc(p["alpha"] * p["rc"] * x), 0.0, 1.0, 0.005 / self.lb)
        self.tables = None
        if p["cut"]:
            self.tables = {}
            for a, b in ((0, 0), (1, 0), (1, 1)):
                self.tables[a, b] = self.tables[b, a] = self._table(a, b)
        n, L, kc = p["kmax"], p["box"], p["kmax"]
        self.n = np.array([v for v in itertools.product(range(0, n + 1), range(-n, n + 1), range(-n, n + 1))
                           if any(v) and v[0] ** 2 + v[1] ** 2 + v[2] ** 2 <= kc * kc])
        k2 = (2 * math.pi / L) ** 2 * (self.n ** 2).sum(1)
        self.ak = np.where(self.n[:, 0] > 0, 2.0, 1.0) * np.exp(-k2 / (4 * p["alpha"] ** 2)) / k2
        self.pref = 2 * math.pi * self.lb / L ** 3

    def _table(self, a, b):
        p = self.p

        def u(r2):
            x = torch.tensor([r2], dtype=torch.float64)
            return float(self.pair(self.s2[a][b], self.e4[a][b], p["charge"][a] * p["charge"][b], x)[0])

        rmin, rmax = (p["sigma"][a] + p["sigma"][b]) / 2, p["cut"]
        while rmin >= 0.01:
            e = abs(u(rmin * rmin))
            if e > 22.0:
                rmin += 0.01
            elif e < 20.0 / 1.1:
                rmin -= 0.01
            else:
                break
        while abs(u(rmax * rmax)) > 0.1:
            rmax += 0.01
        return rmin * rmin, rmax * rmax, _andrea(u, rmin * rmin, rmax * rmax, 1e-3, 1e-2)

    def pair(self, s2, e4, qq, r2):
        """Pair energies at squared distances r2, no tables (s2 and e4: sigma^2 and 4 epsilon)."""
        r = torch.sqrt(r2) + 2.220446049250313e-16
        q = r / self.p["rc"]
        table = tuple(t.to(r2.device) for t in self.short)
        u = torch.where(q < 1, self.lb * qq / r * _spline(table, q.clamp(max=1.0)), 0.0)
        if self.p["hard"]:
            return torch.where(r2 < s2, math.inf, u)
        x = (s2 / r2) ** 3
        return u + e4 * (x * x - x)

    def total_pairs(self, ta, qa, tb, qb, r2):
        """Sum of the pair energies (types and charges elementwise)."""
        if not self.tables and not self.p["g2g"]:
            near = r2 < max(self.p["rc"] ** 2, max(self.s2[0][0], self.s2[1][1]))
            ta, qa, tb, qb, r2 = (v[near] for v in (ta, qa, tb, qb, r2))
        kind = 2 * ta + tb
        s2, e4 = (torch.tensor(sum(v, []), dtype=torch.float64, device=r2.device)[kind] for v in (self.s2, self.e4))
        u = self.pair(s2, e4, qa * qb, r2)
        for (a, b), (lo, hi, table) in (self.tables or {}).items():
            own = kind == 2 * a + b
            u = torch.where(own & (r2 > lo), _spline(tuple(t.to(r2.device) for t in table), r2), u)
            u = torch.where(own & (r2 >= hi), 0.0, u)
        return float(u.sum())

    def phases(self, xyz):
        """e^{ik.r} axis tables of points: three arrays [points, 2 kmax + 1]."""
        m = np.arange(-self.p["kmax"], self.p["kmax"] + 1)
        return [np.exp(2j * math.pi / self.p["box"] * np.outer(xyz[:, d], m)) for d in range(3)]

    def structure(self, xyz, q):
        ex, ey, ez = self.phases(xyz)
        kc, out = self.p["kmax"], np.zeros(len(self.n), complex)
        for nx in range(kc + 1):
            grid = (ey * (q * ex[:, nx + kc])[:, None]).T @ ez
            at = self.n[:, 0] == nx
            out[at] = grid[self.n[at, 1] + kc, self.n[at, 2] + kc]
        return out

    def change_of_q(self, new, old, q):
        kc = self.p["kmax"]
        i, j, k = (self.n + kc).T
        out = np.zeros(len(self.n), complex)
        for sign, xyz in ((1, new), (-1, old)):
            ex, ey, ez = self.phases(xyz)
            for a in range(len(q)):
                out += (sign * q[a]) * ex[a, i] * ey[a, j] * ez[a, k]
        return out

    def image(self, d):
        return d - self.p["box"] * torch.round(d / self.p["box"])


class _Chain:
    """A Metropolis chain followed in 64 bits."""

    def __init__(self, system, phys, seed=0, replica=0, beta=1.0, like=None):
        _, xyz, q, ids, groups = system
        self.m = like.m if like else _Model(phys)
        self.xyz, self.q, self.ids = xyz.copy(), q, ids
        self.tx, self.tq, self.ti = (torch.tensor(v) for v in (self.xyz, q, np.asarray(ids, np.int64)))
        self.size = 1 if len(groups["begin"]) == 1 else 3
        self.seed, self.replica, self.beta, self.moves, self.accepted = seed, replica, beta, 0, 0
        if self.size == 3:
            p = torch.tensor(xyz).view(-1, 3, 3)
            w = torch.tensor([phys["mass"][t] for t in ids[:3]], dtype=torch.float64)
            rel = self.m.image(p - p[:, :1])
            self.cm = self.m.image(p[:, 0] + (w[:, None] / w.sum() * rel).sum(1))
        if like:
            self.qk, self.energy = like.qk.copy(), like.energy
        else:
            self.qk = self.m.structure(xyz, q)
            self.terms = self._terms()
            self.energy = sum(self.terms)

    def _terms(self):
        m, p = self.m, self.m.p
        self_term = -self.m.lb * p["alpha"] / math.sqrt(math.pi) * float((self.q ** 2).sum())
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        x, q, t = self.tx.to(dev), self.tq.to(dev), self.ti.to(dev)
        pairs, n = 0.0, len(q)
        for b in range(0, n, 512):
            d = m.image(x[b:b + 512, None] - x[None])
            r2 = (d * d).sum(2)
            i = torch.arange(b, min(n, b + 512), device=dev)[:, None]
            j = torch.arange(n, device=dev)[None]
            use = (j > i) if self.size == 1 else (j // 3 > i // 3)
            if p["g2g"]:
                c = self.cm.to(dev)
                d = m.image(c[i.ravel() // 3][:, None] - c[None])
                use &= ((d * d).sum(2) < p["g2g"] ** 2).repeat_interleave(3, dim=1)
            elif not p["hard"] and m.tables:
                use &= r2 < max(v[1] for v in m.tables.values())
            i, j = torch.nonzero(use, as_tuple=True)
            pairs += m.total_pairs(t[b + i], q[b + i], t[j], q[j], r2[i, j])
        return [self_term, pairs, m.pref * float((m.ak * abs(self.qk) ** 2).sum())]

    def _pairs(self, first, xyz, cm):
        m, k = self.m, self.size
        out = 0.0
        use = None
        if m.p["g2g"]:
            d = m.image(self.cm - torch.tensor(cm))
            use = ((d * d).sum(1) < m.p["g2g"] ** 2).repeat_interleave(3)
        for a in range(k):
            d = m.image(self.tx - torch.tensor(xyz[a]))
            r2 = (d * d).sum(1)
            ok = torch.ones(len(r2), dtype=torch.bool) if use is None else use.clone()
            ok[first:first + k] = False
            ok &= r2 < (max(v[1] for v in m.tables.values()) if m.tables else math.inf)
            out += m.total_pairs(self.ti[first + a].expand(int(ok.sum())), self.tq[first + a].expand(int(ok.sum())),
                                 self.ti[ok], self.tq[ok], r2[ok])
        return out

    def trial(self, first, new, uniform, cm=None):
        """One move of the atoms first, first + 1, ... to `new`; returns du and the decision."""
        k, m = self.size, self.m
        old = self.xyz[first:first + k]
        e_new = self._pairs(first, new, cm)
        e_old = self._pairs(first, old, None if cm is None else self.cm[first // 3].numpy())
        dq = m.change_of_q(new, old, self.q[first:first + k])
        rec = m.pref * float((m.ak * (2 * (self.qk.conj() * dq).real + abs(dq) ** 2)).sum())
        du = math.inf if math.isinf(e_new) else e_new - e_old + rec
        ok = du <= 0 or uniform <= math.exp(-self.beta * du)
        if ok:
            self.xyz[first:first + k] = new
            self.tx[first:first + k] = torch.tensor(new)
            if cm is not None:
                self.cm[first // 3] = torch.tensor(cm)
            self.qk += dq
            self.energy += du
            self.accepted += 1
        self.moves += 1
        return du, ok

    def step(self):
        """The device chains' own proposal of the next move (Philox4x32-10 blocks of the move)."""
        a, b, c = (_philox((self.moves & 0xffffffff, self.moves >> 32, self.replica, w), self.seed) for w in range(3))
        uniform = ((b[0] >> 5) * 67108864.0 + (b[1] >> 6)) / 2.0 ** 53
        p, box = self.m.p, self.m.p["box"]
        shift = _unit(a[1], a[2]) * (p["dp"] * a[3] / 2.0 ** 32)
        if self.size == 1:
            i = (a[0] * len(self.q)) >> 32
            new = self.xyz[i:i + 1] + shift
            return self.trial(i, new - box * np.round(new / box), uniform)
        g = (a[0] * (len(self.q) // 3)) >> 32
        cm = self.cm[g].numpy() + shift
        cm = cm - box * np.round(cm / box)
        axis, angle = _unit(c[0], c[1]), p["dprot"] * ((c[2] + 0.5) / 2.0 ** 32 - 0.5)
        rel = self.xyz[3 * g:3 * g + 3] + shift - cm
        rel -= box * np.round(rel / box)
        rel = (rel * math.cos(angle) + np.cross(np.broadcast_to(axis, rel.shape), rel) * math.sin(angle) +
               np.outer(rel @ axis, axis) * (1 - math.cos(angle)))
        new = rel + cm
        return self.trial(3 * g, new - box * np.round(new / box), uniform, cm)


def _philox(counter, seed, rounds=10):
    """Philox4x32-10 (Salmon, Moraes, Dror and Shaw 2011)."""
    c = list(counter)
    k0, k1 = seed & 0xffffffff, (seed >> 32) & 0xffffffff
    for _ in range(rounds):
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [(p1 >> 32) ^ c[1] ^ k0, p1 & 0xffffffff, (p0 >> 32) ^ c[3] ^ k1, p0 & 0xffffffff]
        k0, k1 = (k0 + 0x9E3779B9) & 0xffffffff, (k1 + 0xBB67AE85) & 0xffffffff
    return c


def _unit(zw, pw):
    z, phi = 2 * (zw + 0.5) / 2.0 ** 32 - 1, 2 * math.pi * (pw + 0.5) / 2.0 ** 32
    s = math.sqrt(1 - z * z)
    return np.array([s * math.cos(phi), s * math.sin(phi), z])


def _swap(chains, seed, ladder, number):
    """One round of neighbour exchanges along a ladder (chains ordered by decreasing beta)."""
    for k in range(number & 1, len(chains) - 1, 2):
        a, b = chains[k], chains[k + 1]
        x = (a.beta - b.beta) * (a.energy - b.energy)
        r = _philox((number & 0xffffffff, number >> 32, ladder, 0x5a5a0000 + k), seed)
        if x >= 0 or ((r[0] >> 5) * 67108864.0 + (r[1] >> 6)) / 2.0 ** 53 < math.exp(x):
            a.beta, b.beta = b.beta, a.beta
            chains[k], chains[k + 1] = b, a


def exact(case, seed):
    kind = case["kind"]
    if kind in ("polymer", "serve"):
        return None  # pivots of long chains: minutes on the host
    given = _inputs(case, seed)
    if kind == "permove":
        s = given["systems"][0]
        chain, t = _Chain(s["system"], s["phys"]), s["stream"]
        du, acc = [], []
        for i, u in enumerate(t["uniform"]):
            if case["system"] == "water":
                d, ok = chain.trial(3 * int(t["group"][i]), t["xyz"][3 * i:3 * i + 3], u, t["mass_center"][i])
            else:
                j = int(t["index"][i])
                new = chain.xyz[j:j + 1] + t["shift"][i]
                d, ok = chain.trial(j, new - s["phys"]["box"] * np.round(new / s["phys"]["box"]), u)
            du.append(d)
            acc.append(ok)
        return dict(du=np.array(du), accepted=np.array(acc, np.uint8), positions=chain.xyz)
    if kind == "resume":
        s = given["systems"][0]
        ck = s["checkpoint"]["xyz"]
        chain = _Chain((s["system"][0], ck, *s["system"][2:]), s["phys"])
        return dict(energy=chain.energy, total=chain.energy, terms=np.array(chain.terms), rdf=None, positions=ck)
    reps = _replicas(case, given)
    cost = sum(r["moves"] * (8e-4 + 1e-7 * len(r["system"][2]) * (1 if r["kinds"] is None else 4)) for r in reps)
    if cost * (2 if kind == "ladder" else 1) > 15.0:
        return None  # too many moves to follow on the host
    first, chains = {}, []
    for i, r in enumerate(reps):
        c = _Chain(r["system"], r["phys"], r["seed"], i, r["beta"], like=first.get(id(r["system"][1])))
        if id(r["system"][1]) not in first:
            first[id(r["system"][1])] = _Chain(r["system"], r["phys"], like=c)
        chains.append(c)
    ladders = {}
    for r, c in zip(reps, chains):
        ladders.setdefault(r["ladder"], []).append(c)
    for lap in range(2 if kind == "ladder" else 1):
        for r, c in zip(reps, chains):
            for _ in range(r["moves"]):
                c.step()
        for lad, rungs in ladders.items():
            if lad >= 0:
                _swap(rungs, 4242 if kind == "ladder" else 77, lad, lap)
    return dict(energy=np.array([c.energy for c in chains]), beta=np.array([c.beta for c in chains]),
                accepted=np.array([c.accepted for c in chains], np.int64),
                positions=np.concatenate([c.xyz for c in chains]))
