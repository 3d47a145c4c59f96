"""Pair rows of one moved ion over all others (no cell list) at particle counts around the
lanes' slots, for the forms with straight-line code (hard spheres or Lennard-Jones plus Ewald)
and the general one (both, or an unsplined term), FP64 and FP32 pairs, against the oracle."""
import numpy as np
import pytest

import faunus_amd as F
from oracle import oracle as O
from tests import systems
from tests.gpu_helpers import compare_chain

pytestmark = pytest.mark.gpu

LJ, HS = {"lennardjones": {"mixing": "LB"}}, {"hardsphere": {}}


def ions(n, terms, splined):
    box = 60.0 * (n / 400.0) ** (1 / 3)
    xyz = systems.lattice_positions(n, box, 4.0, np.random.default_rng(n))
    ids = np.arange(n, dtype=np.int32) % 2
    coul = {"coulomb": {"type": "ewald", "epsr": 78.7, "cutoff": box / 2, "alpha": 5 / box, "ncutoff": 4, "splined": splined}}
    cfg = {"temperature": 298.15, "geometry": {"type": "cuboid", "length": box},
           "atomlist": [{"A": {"q": 1.0, "sigma": 3.3, "eps": 0.5, "dp": 5.0}}, {"B": {"q": -1.0, "sigma": 4.0, "eps": 0.4, "dp": 5.0}}],
           "moleculelist": [{"salt": {"atoms": ["A", "B"], "atomic": True}}],
           "energy": [{"nonbonded": {"default": terms + [coul]}}]}
    return cfg, xyz, np.where(ids == 0, 1.0, -1.0), ids, dict(begin=[0], size=[n], molid=[0])


# du within 1e-10 (FP64) or 1e-6 (FP32 pairs) of max(|du|, |E|), the bars of the device chains
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("terms,splined", [([HS], True), ([LJ], True), ([HS, LJ], True), ([HS], False)])
@pytest.mark.parametrize("n", [2, 512, 513, 1025, 1537, 2049])
def test_row_edges(n, terms, splined, fp32):
    system = ions(n, terms, splined)
    orc = O.System(system[0])
    orc.set_particles(*system[1:4])
    orc.set_groups(*(system[4][k] for k in ("begin", "size", "molid")))
    e0 = orc.init()
    b = F.Batch(fp32_pairs=fp32)
    b.add(system, seed=3)
    b.run([40], trace=40)
    rec = orc.run_philox_translate(40, seed=3)
    rep = compare_chain(b.trace(0, 40), rec, max(1.0, abs(e0)), 1e-6 if fp32 else 1e-10, 3)
    b.close()
    assert rep["first_mismatch"] == 40 and rep["max_rel"] <= (1e-6 if fp32 else 1e-10), rep
