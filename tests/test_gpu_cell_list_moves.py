"""Move sets on the general kernel's cell-list form, against the oracle on the same Philox
stream: every stencil form on both grids, in FP64 and with FP32 pairs, for the systems that walk
it (rigid molecules with ions, with a larger molecule and a group cutoff, or with a fixed cell
capacity; a flexible chain with pivots).  Each test asserts the kernel it runs on.

du within 1e-10 (FP64) or 1e-6 (FP32 pairs) of max(|du|, |E|), FP64 decisions and positions equal."""
import numpy as np
import pytest

import faunus_amd as F
from oracle import oracle as O
from tests import systems
from tests.gpu_helpers import compare_chain, log, DRIFT_FP32
from tests.test_gpu_rigid import molecules

pytestmark = pytest.mark.gpu


def follow(system, kinds, moves, seed, fp32, telescopes=True, **batch):
    orc = O.System(system[0])
    orc.set_particles(*system[1:4])
    orc.set_groups(*(system[4][k] for k in ("begin", "size", "molid")))
    e0 = orc.init()
    b = F.Batch(fp32_pairs=fp32, **batch)
    b.add(system, seed=seed, moves=kinds)
    assert b.kernel(0) == "general cells"
    b.run([moves], trace=moves)
    rec = orc.run_philox_moves(moves, seed=seed, kinds=kinds, replica=0)
    tol = 1e-6 if fp32 else 1e-10
    rep = compare_chain(b.trace(0, moves), rec, max(1.0, abs(e0)), tol, seed)
    log("cell-list moves", batch, fp32, rep)
    info = b.info(0)
    assert info["error"] == 0 and info["moves"] == moves
    assert rep["max_rel"] <= tol and rep["accepted"] > 0, rep
    if not fp32:
        assert rep["first_mismatch"] == moves, rep
        np.testing.assert_allclose(b.positions(0), orc.positions(), rtol=0, atol=1e-9)
    if telescopes:
        tot, _ = b.total_energy(0)
        assert abs(info["energy"] - tot) <= (DRIFT_FP32 if fp32 else 1e-9) * abs(tot)
    dq, _ = b.check_q(0)
    assert dq < 1e-9
    b.close()


def stencil(box, reach, extent, divisions):
    """Whether one stencil per state serves a molecule of that extent (reach + extent within
    `divisions` cells)."""
    cell = box / np.floor(divisions * box / reach)
    return reach + extent <= divisions * cell


def water_and_ions(cutoff, n_mol=1000, n_ions=20, kmax=5):
    """Waters of which the last n_ions are ions of charge +-0.6, moved by translation."""
    cfg, xyz, q, ids, g, kinds = systems.water(n_mol=n_mol, seed=2, kmax=kmax, cutoff=cutoff)
    keep = 3 * (n_mol - n_ions)
    cfg["atomlist"] += [{"Na": {"q": 0.6, "sigma": 2.5, "eps": 0.3, "dp": 0.5}},
                        {"Cl": {"q": -0.6, "sigma": 3.5, "eps": 0.3, "dp": 0.5}}]
    cfg["moleculelist"] += [{"salt": {"atoms": ["Na", "Cl"], "atomic": True}}]
    xyz = np.concatenate([xyz[:keep], xyz[keep::3]])
    q = np.concatenate([q[:keep], [0.6, -0.6] * (n_ions // 2)])
    ids = np.concatenate([ids[:keep], [2, 3] * (n_ions // 2)]).astype(np.int32)
    waters = n_mol - n_ions
    groups = dict(begin=g["begin"][:waters] + [keep], size=[3] * waters + [n_ions], molid=[0] * waters + [1])
    return (cfg, xyz, q, ids, groups), kinds + [dict(kind=0, molid=1, weight=1, dp=0.5)]


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("rc,divisions,one", [(8.0, 1, True), (10.0, 1, False), (9.0, 2, True), (10.0, 2, False)])
def test_water_with_ions(rc, divisions, one, fp32):
    system, kinds = water_and_ions(rc)
    assert stencil(system[0]["geometry"]["length"], rc, 1.0, divisions) == one
    follow(system, kinds, 400, 17, fp32, cell_divisions=divisions)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("rc,divisions", [(8.0, 1), (10.0, 1), (9.0, 2), (10.0, 2)])
def test_water_with_a_fixed_capacity(rc, divisions, fp32):
    cfg, xyz, q, ids, g, kinds = systems.water(n_mol=1000, seed=3, kmax=5, cutoff=rc)
    follow((cfg, xyz, q, ids, g), kinds, 400, 8, fp32, cell_divisions=divisions, cell_capacity=400)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("divisions", [1, 2])
def test_group_cutoff_with_a_larger_molecule(divisions, fp32):
    """Molecules of nine atoms among triatomic ones, a cutoff per pair of molecule types."""
    system, kinds = molecules({3: 400, 9: 3}, 36.0, {"default": 9.0, "m3 m9": 8.0})
    follow(system, kinds, 300, 23, fp32, cell_divisions=divisions)


@pytest.mark.parametrize("divisions,fp32", [(1, False), (2, False), (1, True), (2, True)])
def test_water_group_cutoff_with_a_fixed_capacity(divisions, fp32):
    cfg, xyz, q, ids, g, kinds = systems.water_g2g(n_mol=1728, seed=4, cutoff=9.0, g2g=9.0, kmax=5)
    follow((cfg, xyz, q, ids, g), kinds, 300, 21, fp32, cell_divisions=divisions, cell_capacity=400)


@pytest.mark.parametrize("divisions,fp32,excluded", [(1, False, 0), (1, True, 1), (2, False, 1), (2, True, 0)])
def test_flexible_chain_with_pivots(divisions, fp32, excluded):
    cfg, xyz, q, ids, g, kinds = systems.polyelectrolyte(20, 300, seed=7, kmax=5, excluded_neighbours=excluded)
    for atom in cfg["atomlist"]:
        for v in atom.values():
            v["eps"] = 0.3
    cfg["energy"][1] = systems.pair_cut([{"lennardjones": {"mixing": "LB"}},
                                         {"coulomb": {"type": "ewald", "epsr": 78.7, "cutoff": 20.0, "alpha": 0.15,
                                                      "ncutoff": 5}}], 19.9)
    kinds = [dict(k, weight=w) for k, w in zip(kinds, (2, 1, 3))]
    follow((cfg, xyz, q, ids, g), kinds, 500, 5, fp32, cell_divisions=divisions)


def test_the_kernel_of_each_kind_of_replica():
    nacl = systems.nacl_lj(n_pairs=300, box=90.0, seed=2, kmax=6)
    many = systems.nacl_lj(n_pairs=300, box=90.0, seed=2, kmax=14)
    chain = systems.polyelectrolyte(20, 200, seed=7, kmax=5)
    water = systems.water_g2g(n_mol=216, seed=3, kmax=5)
    for want, system, kinds in (("translate", nacl, None), ("advance", many, None), ("general", chain[:5], chain[5]),
                                ("rigid", water[:5], water[5])):
        b = F.Batch()
        b.add(system, seed=1, moves=kinds)
        assert b.kernel(0) == want
        b.close()
    with pytest.raises(RuntimeError, match="out of range"):
        b = F.Batch()
        b.add(nacl, seed=1)
        b.kernel(1)
