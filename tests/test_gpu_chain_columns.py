"""Pivots and bead translations whose slices of particles end in columns of 64, and whose
k-vectors leave room for several groups of threads, against the oracle running the same
Philox stream.  Sizes lie at the edges: slices of 63 to 65 and 511 to 513 particles, just
below four per lane and above; 1 to 16 workgroups; k-spheres of 13 vectors (more groups than
the tables hold sums for) to several hundred; chains around the least moved count.

FP64: du within 1e-10 of max(|du|, E_scale) with every decision equal; FP32: 1e-6 up to the
first near-tie.  These are the bounds that hold for every form of the kernel."""
import numpy as np
import pytest

import faunus_amd as F
from oracle import oracle as O
from tests import systems
from tests.gpu_helpers import compare_chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("beads,total,kmax,groups,excl", [
    (9, 63, 2, 1, 0), (12, 64, 3, 1, 0), (40, 130, 6, 2, 1), (30, 514, 5, 1, 0), (30, 1022, 5, 2, 2),
    (25, 1026, 1, 2, 0), (60, 2046, 4, 1, 0), (60, 2052, 4, 1, 0), (100, 1600, 7, 16, 0),
])
def test_chain_moves_at_the_edges_of_columns_and_groups(beads, total, kmax, groups, excl, fp32):
    cfg, xyz, q, ids, g, kinds = systems.polyelectrolyte(beads, total, seed=beads, kmax=kmax, excluded_neighbours=excl)
    kinds = [dict(k, weight=w) for k, w in zip(kinds, (1, 1, 4))]  # mostly pivots
    orc = O.System(cfg)
    orc.set_particles(xyz, q, ids)
    orc.set_groups(g["begin"], g["size"], g["molid"])
    e0 = orc.init()
    nm = 150
    print("chain columns", beads, total, kmax, groups, excl, fp32, flush=True)
    b = F.Batch(fp32_pairs=fp32)
    b.add((cfg, xyz, q, ids, g), seed=21, moves=kinds)
    if groups > 1:
        b.run_split(nm, groups=groups, trace=nm)
    else:
        b.run([nm], trace=nm)
    b.sync()
    rec = orc.run_philox_moves(nm, seed=21, kinds=kinds, replica=0)
    rep = compare_chain(b.trace(0, nm), rec, max(1.0, abs(e0)), 1e-6 if fp32 else 1e-10, 21)
    assert b.info(0)["error"] == 0 and b.info(0)["moves"] == nm
    assert rep["max_rel"] <= (1e-6 if fp32 else 1e-10), rep
    if not fp32:
        assert rep["first_mismatch"] == nm, rep
        np.testing.assert_allclose(b.positions(0), orc.positions(), rtol=0, atol=1e-9)
    dq, _ = b.check_q(0)
    if rep["first_mismatch"] == nm:
        assert dq < 1e-9
    b.close()
