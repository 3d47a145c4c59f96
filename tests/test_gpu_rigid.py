"""Chains of rigid molecules (the kernel that tests mass centres instead of walking a cell
list) against the oracle on the same Philox stream, over the forms that route takes: one
molecule and counts around the workgroup's size, molecules of 1 to 8 atoms in one system,
several move kinds, a cutoff table with unequal entries, splined pairs, the surface term, no
Ewald sum; a launch that mixes such replicas with others; and a fixed cell capacity, which keeps
the cell list."""
import numpy as np
import pytest

import faunus_amd as F
from oracle import oracle as O
from tests import systems
from tests.gpu_helpers import compare_chain

pytestmark = pytest.mark.gpu


def molecules(counts, box, g2g, kmax=5, splined=None, epss=0.0, coulomb="ewald", seed=1):
    """counts: number of molecules of each size; bent chains with 0.8 A steps on a lattice."""
    rng = np.random.default_rng(seed)
    sizes = sorted(counts)
    total = sum(counts.values())
    m = int(np.ceil(total ** (1 / 3)))
    sites = rng.permutation(m ** 3)[:total]
    centre = (np.stack([sites % m, sites // m % m, sites // m ** 2], axis=1) + 0.5) * box / m - box / 2
    xyz, ids, begin, size, molid = [], [], [], [], []
    for t, s in enumerate(sizes):
        for _ in range(counts[s]):
            q, _r = np.linalg.qr(rng.normal(size=(3, 3)))
            chain = np.stack([0.8 * (np.arange(s) % 2), 0.8 * (np.arange(s) // 2 % 2), 0.8 * (np.arange(s) // 4)], axis=1)
            begin.append(len(xyz))
            for p in centre[len(begin) - 1] + (chain - chain.mean(0)) @ q:
                xyz.append(p - box * np.round(p / box))
            ids += [k % 2 for k in range(s)]
            size.append(s)
            molid.append(t)
    if coulomb == "ewald":
        coul = {"type": "ewald", "epsr": 40.0, "cutoff": min(9.0, 0.45 * box), "alpha": 0.25, "ncutoff": kmax, "epss": epss}
    else:
        coul = {"type": "fanourgakis", "epsr": 40.0, "cutoff": min(9.0, 0.45 * box)}
    terms = [{"lennardjones": {"mixing": "LB"}}, {"coulomb": coul}]
    if splined:
        energy = {"nonbonded_splined": {"default": terms, "rmax": splined, "u_at_rmax": 0.3}}
    else:
        energy = {"nonbonded": {"default": terms, "cutoff_g2g": g2g}}
    cfg = {"temperature": 298.15, "geometry": {"type": "cuboid", "length": box},
           "atomlist": [{"A": {"q": 0.4, "sigma": 2.6, "eps": 0.4, "mw": 12.0}},
                        {"B": {"q": -0.4, "sigma": 2.2, "eps": 0.3, "mw": 1.0}}],
           "moleculelist": [{"m%d" % s: {"atoms": ["AB"[k % 2] for k in range(s)], "rigid": True}} for s in sizes],
           "energy": [energy]}
    ids = np.array(ids, np.int32)
    kinds = [dict(kind=1, molid=t, weight=1 + t, dp=0.6 if t != 1 else 0.0, dprot=0.8) for t in range(len(sizes))]
    return (cfg, np.array(xyz), np.where(ids == 0, 0.4, -0.4), ids, dict(begin=begin, size=size, molid=molid)), kinds


def oracle_of(system):
    s = O.System(system[0])
    s.set_particles(*system[1:4])
    s.set_groups(*(system[4][k] for k in ("begin", "size", "molid")))
    return s, s.init()


def check(batch, r, system, kinds, moves, seed, fp32):
    """du within 1e-10 (FP64) or 1e-6 (FP32 pairs) of max(|du|, |E|) and the oracle's decisions."""
    orc, e0 = oracle_of(system)
    rec = orc.run_philox_moves(moves, seed=seed, kinds=kinds, replica=r)
    rep = compare_chain(batch.trace(r, moves), rec, max(1.0, abs(e0)), 1e-6 if fp32 else 1e-10, seed, replica=r)
    assert rep["first_mismatch"] == moves and rep["max_rel"] <= (1e-6 if fp32 else 1e-10), rep
    np.testing.assert_allclose(batch.positions(r), orc.positions(), rtol=0, atol=1e-9)
    assert batch.info(r)["error"] == 0


FORMS = [
    (dict(counts={3: 1}, box=30.0, g2g=9.0), False),
    (dict(counts={3: 511}, box=32.0, g2g=9.0), False),
    (dict(counts={2: 512, 8: 1}, box=33.0, g2g=9.0), False),
    (dict(counts={1: 200, 3: 200, 7: 113}, box=36.0, g2g={"default": 8.0, "m1 m3": 9.5, "m7 m7": 7.0}), False),
    (dict(counts={4: 300}, box=30.0, g2g=0, splined=8.5), False),
    (dict(counts={3: 300}, box=30.0, g2g=9.0, epss=1.0, kmax=4), False),
    (dict(counts={3: 300}, box=30.0, g2g=9.0, coulomb="fanourgakis"), False),
    (dict(counts={3: 300}, box=30.0, g2g=9.0, kmax=12), False),
    (dict(counts={1: 200, 3: 200, 7: 113}, box=36.0, g2g={"default": 8.0, "m1 m3": 9.5, "m7 m7": 7.0}), True),
    (dict(counts={4: 300}, box=30.0, g2g=0, splined=8.5), True),
]


@pytest.mark.parametrize("form,fp32", FORMS)
def test_rigid_molecules(form, fp32):
    system, kinds = molecules(**form)
    b = F.Batch(fp32_pairs=fp32)
    b.add(system, seed=12, moves=kinds)
    b.run([130], trace=130)
    check(b, 0, system, kinds, 130, 12, fp32)
    b.close()


def test_mixed_launch_and_fixed_capacity():
    """A flexible polymer between two rigid replicas in one launch; then the same water with a
    fixed cell capacity (cell list) and without (centres): the same chain."""
    rigid = molecules({3: 120}, 26.0, 9.0)
    cfg, xyz, q, ids, g, kinds = systems.polyelectrolyte(20, 200, seed=7, kmax=5)
    b = F.Batch()
    for system, k in (rigid, ((cfg, xyz, q, ids, g), kinds), rigid):
        b.add(system, seed=5, moves=k)
    b.run([70, 70, 70], trace=70)
    for r, (system, k) in enumerate((rigid, ((cfg, xyz, q, ids, g), kinds), rigid)):
        check(b, r, system, k, 70, 5, False)
    b.close()
    cfg, xyz, q, ids, g, kinds = systems.water(n_mol=1000, seed=3, kmax=4, cutoff=10.0)
    out = []
    for capacity in (0, 400):
        b = F.Batch(cell_capacity=capacity)
        b.add((cfg, xyz, q, ids, g), seed=9, moves=kinds)
        b.run([200])
        out.append((b.positions(0), b.info(0)["accepted"]))
        b.close()
    np.testing.assert_allclose(out[0][0], out[1][0], rtol=0, atol=1e-9)
    assert out[0][1] == out[1][1]
