"""The translation kernel at its edges: k-lists around a thread's share (one to five pairs of
k-vectors per thread, none), cell lists of few and many members at both workgroup sizes, a
system in which most moves follow a move of the same particle, and K on both sides of the route
to the kernel for large K, FP64 and FP32 pairs, against the oracle."""
import numpy as np
import pytest

import faunus_amd as F
from oracle import oracle as O
from tests import systems
from tests.gpu_helpers import compare_chain

pytestmark = pytest.mark.gpu


def ions(n, box, kmax, cut, coulomb="ewald"):
    xyz = systems.lattice_positions(n, box, 2.8, np.random.default_rng(n))
    ids = np.arange(n, dtype=np.int32) % 2
    coul = {"type": coulomb, "epsr": 78.7, "cutoff": cut or 0.5 * box}
    if coulomb == "ewald":
        coul.update(alpha=0.2, ncutoff=kmax)
    cfg = {"temperature": 298.15, "geometry": {"type": "cuboid", "length": box},
           "atomlist": [{"A": {"q": 1.0, "sigma": 2.8, "dp": 6.0}}, {"B": {"q": -1.0, "sigma": 2.8, "dp": 6.0}}],
           "moleculelist": [{"salt": {"atoms": ["A", "B"], "atomic": True}}],
           "energy": [{"nonbonded": {"default": [{"hardsphere": {}}, {"coulomb": coul}]}}]}
    return cfg, xyz, np.where(ids == 0, 1.0, -1.0), ids, dict(begin=[0], size=[n], molid=[0])


# du within 1e-10 (FP64) or 1e-6 (FP32 pairs) of max(|du|, |E|), the bars of the device chains
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("n,box,kmax,cut,coulomb", [
    (3, 40.0, 1, None, "ewald"),          # one k-vector pair or none, the same particle again and again
    (40, 40.0, 8, None, "ewald"),         # two pairs on some threads (512)
    (40, 40.0, 12, None, "ewald"),        # five pairs per thread
    (40, 40.0, 0, None, "fanourgakis"),   # no k-vectors
    (60, 48.0, 6, 12.0, "ewald"),         # 4 x 4 x 4 cells of about one member (256 threads)
    (900, 48.0, 6, 12.0, "ewald"),        # of 14 (512 threads)
    (100, 48.0, 11, 12.0, "ewald"),       # K beyond 8 per thread of 256
    (100, 48.0, 13, 12.0, "ewald"),       # K beyond 8 per thread of 512: the other kernel
])
def test_translations(n, box, kmax, cut, coulomb, fp32):
    system = ions(n, box, kmax, cut, coulomb)
    orc = O.System(system[0])
    orc.set_particles(*system[1:4])
    orc.set_groups(*(system[4][k] for k in ("begin", "size", "molid")))
    e0 = orc.init()
    b = F.Batch(fp32_pairs=fp32)
    b.add(system, seed=4)
    b.run([150], trace=150)
    rec = orc.run_philox_translate(150, seed=4)
    rep = compare_chain(b.trace(0, 150), rec, max(1.0, abs(e0)), 1e-6 if fp32 else 1e-10, 4)
    assert rep["first_mismatch"] == 150 and rep["max_rel"] <= (1e-6 if fp32 else 1e-10), rep
    assert b.info(0)["error"] == 0 and b.info(0)["moves"] == 150
    np.testing.assert_allclose(b.positions(0), orc.positions(), rtol=0, atol=1e-9)
    if coulomb == "ewald":
        assert b.check_q(0)[0] < 1e-9
    b.close()


def test_routes_of_one_launch():
    """Replicas on both sides of the route, in one launch and alone: the same chains."""
    systems_ = [ions(80, 44.0, k, None) for k in (4, 13, 9)]
    alone = []
    for r, s in enumerate(systems_):
        b = F.Batch()
        for q in range(r):
            b.add(systems_[0], seed=1)
        b.add(s, seed=7)
        b.run([0] * r + [100])
        alone.append((b.positions(r), b.info(r)["energy"]))
        b.close()
    b = F.Batch()
    for s in systems_:
        b.add(s, seed=7)
    b.run([100] * 3)
    for r in range(3):
        np.testing.assert_array_equal(b.positions(r), alone[r][0])
        assert b.info(r)["energy"] == alone[r][1]
    b.close()


def test_ladders_of_unlike_replicas_with_cell_lists():
    """Free-running ladders take one launch: replicas with cell lists whose own workgroup sizes
    or kernels differ share one, with the chains of their separate runs."""
    forms = [ions(60, 48.0, 6, 12.0), ions(100, 48.0, 11, 12.0), ions(900, 48.0, 6, 12.0), ions(100, 48.0, 13, 12.0)]
    for pick in (forms[:3], forms):
        a, b = F.Batch(), F.Batch()
        for r, s in enumerate(pick):
            a.add(s, seed=5 + r, ladder=r)
            b.add(s, seed=5 + r)
        a.run_ladders(60, 2, seed=1)
        b.run([120] * len(pick))
        for r in range(len(pick)):
            np.testing.assert_allclose(a.positions(r), b.positions(r), rtol=0, atol=1e-9)
            assert a.info(r)["accepted"] == b.info(r)["accepted"] and a.info(r)["moves"] == 120
        a.close()
        b.close()
