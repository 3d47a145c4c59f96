"""Chains whose tables nearly fill the LDS that a general-kernel workgroup may take (moved
atoms, k-vectors and phase tables), against the oracle on the same Philox stream.  With kmax = 12
(K = 3796) the FP32 form has held chains of up to 698 beads beside its static tables, the FP64 form
of up to 939 within its 96 KB.  Bounds as for every form of the kernel: du within 1e-10 (FP64) or
1e-6 (FP32 pairs) of max(|du|, E_scale)."""
import pytest

import faunus_amd as F
from oracle import oracle as O
from tests import systems
from tests.gpu_helpers import compare_chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("beads,fp32", [(640, True), (698, True), (939, False)])
def test_long_chain_with_many_k_vectors(beads, fp32):
    cfg, xyz, q, ids, g, kinds = systems.polyelectrolyte(beads, 2 * beads + 20, seed=3, kmax=12)
    kinds = [dict(k, weight=w) for k, w in zip(kinds, (1, 1, 2))]
    orc = O.System(cfg)
    orc.set_particles(xyz, q, ids)
    orc.set_groups(g["begin"], g["size"], g["molid"])
    e0 = orc.init()
    nm = 40
    b = F.Batch(fp32_pairs=fp32)
    b.add((cfg, xyz, q, ids, g), seed=4, moves=kinds)
    b.run([nm], trace=nm)
    rec = orc.run_philox_moves(nm, seed=4, kinds=kinds, replica=0)
    tol = 1e-6 if fp32 else 1e-10
    rep = compare_chain(b.trace(0, nm), rec, max(1.0, abs(e0)), tol, 4)
    assert rep["max_rel"] <= tol and (fp32 or rep["first_mismatch"] == nm), rep
    assert b.info(0)["error"] == 0 and b.info(0)["moves"] == nm
    b.close()
