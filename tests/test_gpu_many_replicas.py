"""Batches of more replicas with a cell list than the device has CUs (256): free-running
ladders, for which every workgroup has to be resident, take up to two replicas per CU; they equal
the captured interval replayed as often, bit for bit, and the oracle on the same Philox stream."""
import numpy as np
import pytest

import faunus_amd as F
from oracle import oracle as O
from tests import systems
from tests.gpu_helpers import compare_chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("count,kmax", [(257, 4), (512, 4), (512, 8)])
def test_more_cell_list_replicas_than_cus(count, kmax, fp32):
    system = systems.primitive_model(n_pairs=70, box=66.0, seed=2, cutoff=20.0, kmax=kmax, dp=4.0)

    def batch():
        b = F.Batch(fp32_pairs=fp32)
        for r in range(count):
            b.add(system, beta=1.0 - 0.05 * (r % 4), seed=900 + r, ladder=r // 4)
        return b

    free, captured = batch(), batch()
    moves = np.full(count, 70, np.int64)
    free.run_ladders(moves, np.full(count, 3, np.int32), seed=5)
    captured.capture_interval(moves, seed=5, round0=0)
    for _ in range(3):
        captured.replay(1)
        captured.sync()
    assert free.swap_counts() == captured.swap_counts()
    for r in (0, 3, count // 2, count - 1):
        a, c = free.info(r), captured.info(r)
        assert a == c and a["moves"] == 210 and a["error"] == 0
        assert np.array_equal(free.positions(r), captured.positions(r))
    free.close()
    captured.close()
    # a plain run, replica by replica against the oracle
    b = batch()
    b.run(moves, trace=70)
    for r in (0, count - 1):
        orc = O.System(system[0])
        orc.set_particles(*system[1:4])
        orc.set_groups(*(system[4][k] for k in ("begin", "size", "molid")))
        e0 = orc.init()
        beta = 1.0 - 0.05 * (r % 4)
        rec = orc.run_philox_translate(70, seed=900 + r, replica=r, beta=beta)
        tol = 1e-6 if fp32 else 1e-10
        rep = compare_chain(b.trace(r, 70), rec, max(1.0, abs(e0)), tol, 900 + r, replica=r, beta=beta)
        assert rep["max_rel"] <= tol and (fp32 or rep["first_mismatch"] == 70), rep
    b.close()
