"""Replicas of one batch or server that take different kernels or workgroup sizes run side by
side: a mixed batch takes about as long as its longer half, not as both, every replica follows
the oracle on its own Philox stream, and a captured interval of such a batch equals eager runs,
replay by replay."""
import numpy as np
import pytest

import faunus_amd as F
from oracle import oracle as O
from tests import systems
from tests.gpu_helpers import compare_chain, log

pytestmark = pytest.mark.gpu


def dilute():  # 2.3 members per cell: 256 threads
    return systems.nacl_lj(n_pairs=800, box=255.0 * (1600 / 20000) ** (1 / 3), seed=2, kmax=6), None


def dense():  # 7.4 members per cell: 512 threads
    return systems.primitive_model(n_pairs=100, box=118.0, seed=1), None


def water():
    w = systems.water_g2g(n_mol=64, seed=3, kmax=4, cutoff=6.0, g2g=6.0)
    return w[:5], w[5]


def chain():
    p = systems.polyelectrolyte(20, 200, seed=7, kmax=5)
    return p[:5], p[5]


def batch_of(parts, fp32=False):
    b = F.Batch(fp32_pairs=fp32)
    for r, (system, kinds) in enumerate(parts):
        b.add(system, seed=300 + r, moves=kinds)
    b.set_timing(True)
    return b


def milliseconds(b, moves):
    b.run(moves)
    b.sync()
    best = 1e9
    for _ in range(3):
        b.run(moves)
        best = min(best, b.sync())
    return best


def test_two_workgroup_sizes_overlap():
    count = 60
    halves = [dilute(), dense()]
    alone, moves = [], []
    for h in halves:
        b = batch_of([h] * count)
        per = milliseconds(b, 100) / 100
        moves.append(int(3.0 / per))  # about 3 ms for either half
        alone.append(milliseconds(b, moves[-1]))
        b.close()
    b = batch_of([halves[r % 2] for r in range(2 * count)])
    both = milliseconds(b, np.array([moves[r % 2] for r in range(2 * count)], np.int64))
    b.close()
    log("side by side: alone", alone, "both", both)
    assert both < 0.8 * sum(alone), (alone, both)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("first,second", [(dilute, dense), (water, chain)])
def test_mixed_batch_follows_the_oracle_and_its_capture(first, second, fp32):
    parts = [first(), second(), first(), second(), second()]
    b, g = batch_of(parts, fp32), batch_of(parts, fp32)
    if first is water:
        assert [b.kernel(r) for r in range(2)] == ["rigid", "general"]
    moves = np.array([60, 75, 0, 90, 40], np.int64)
    b.run(moves, trace=90)
    b.sync()
    tol = 1e-6 if fp32 else 1e-10
    for r, (system, kinds) in enumerate(parts):
        nm = int(moves[r])
        assert b.info(r)["moves"] == nm and b.info(r)["error"] == 0
        if nm == 0:
            continue
        orc = O.System(system[0])
        orc.set_particles(*system[1:4])
        orc.set_groups(*(system[4][k] for k in ("begin", "size", "molid")))
        e0 = orc.init()
        rec = (orc.run_philox_moves(nm, seed=300 + r, kinds=kinds, replica=r) if kinds else
               orc.run_philox_translate(nm, seed=300 + r, replica=r))
        rep = compare_chain(b.trace(r, nm), rec, max(1.0, abs(e0)), tol, 300 + r, replica=r)
        assert rep["max_rel"] <= tol and (fp32 or rep["first_mismatch"] == nm), rep
    g.capture_interval(moves, seed=1, round0=0)
    g.replay(1)
    g.sync()
    for step in range(3):
        if step:
            b.run(moves)
            g.replay(1)
            b.sync()
            g.sync()
        for r in range(len(parts)):
            assert b.info(r) == g.info(r)
            assert np.array_equal(b.positions(r), g.positions(r))
    b.close()
    g.close()


@pytest.mark.parametrize("split_atoms", [0, 100])
def test_server_with_jobs_of_every_kernel(split_atoms):
    """The jobs of a mixed server equal the same jobs served alone, also where the chains are
    shared by two workgroups in a cooperative launch."""
    kinds_of_job = [dilute(), dense(), water(), chain()]

    def serve(jobs):
        srv = F.Server(fp32_pairs=False, max_slots=16, split_atoms=split_atoms)
        ids = [srv.submit(s, 500, seed=40 + k, kinds=m) for k, s, m in jobs]
        while srv.step(400) != (0, 0):
            pass
        out = [(srv.job(j)["accepted"], srv.positions(j)) for j in ids]
        srv.close()
        return out
    jobs = [(k, *kinds_of_job[k % 4]) for k in range(8)]
    mixed = serve(jobs)
    for job, (accepted, xyz) in zip(jobs, mixed):
        (alone,) = serve([job])
        assert alone[0] == accepted and np.array_equal(alone[1], xyz)
