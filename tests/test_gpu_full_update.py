"""Full recomputes at the sizes where their tiling can go wrong: Q(k) (whole and broken
particle chunks, one and several column and nz blocks, a k list without its centre column's
neighbours, a box with three lengths) and all pairs (tile edges, short runs, with and without
a cutoff) against the oracle; the pair-distance histogram across tile edges against numpy."""
import numpy as np
import pytest

import faunus_amd as F
from tests import systems
from tests.gpu_helpers import build_pair

pytestmark = pytest.mark.gpu


def ions(n, kmax, box=(60.0, 60.0, 60.0), cut=None, seed=3):
    rng = np.random.default_rng(seed)
    ids = np.arange(n, dtype=np.int32) % 2
    ewald = {"coulomb": {"type": "ewald", "epsr": 78.7, "cutoff": cut or 20.0, "alpha": 0.2, "ncutoff": kmax}}
    terms = [{"hardsphere": {}}] if cut else [{"lennardjones": {"mixing": "LB"}}]
    cfg = {"temperature": 298.15, "geometry": {"type": "cuboid", "length": list(box)},
           "atomlist": [{"A": {"q": 1.0, "sigma": 0.2, "eps": 0.1}}, {"B": {"q": -1.0, "sigma": 0.2, "eps": 0.1}}],
           "moleculelist": [{"salt": {"atoms": ["A", "B"], "atomic": True}}],
           "energy": [{"nonbonded": {"default": terms + [ewald]}}]}
    m = int(np.ceil(n ** (1 / 3)))
    sites = rng.permutation(m ** 3)[:n]
    xyz = np.stack([sites % m, sites // m % m, sites // m ** 2], axis=1) + 0.5 + 0.3 * rng.random((n, 3)) - 0.15
    xyz = (xyz / m - 0.5) * np.array(box)
    return cfg, xyz, np.where(ids == 0, 1.0, -1.0), ids, dict(begin=[0], size=[n], molid=[0])


# FP64 sums of up to n terms of either sign: 1e-10 of the total (at least 1 kT), the bar of
# every FP64 parity test here
@pytest.mark.parametrize("n,kmax,box,cut", [
    (2, 1, (60.0, 60.0, 60.0), None), (31, 7, (60.0, 60.0, 60.0), None), (33, 8, (60.0, 60.0, 60.0), 12.0),
    (257, 11, (60.0, 60.0, 60.0), 12.0), (256, 12.5, (60.0, 45.0, 70.0), None), (1000, 20, (60.0, 60.0, 60.0), 12.0),
    (515, 24, (60.0, 60.0, 60.0), 12.0), (64, 33, (50.0, 60.0, 50.0), None)])
def test_full_energy(n, kmax, box, cut):
    orc, eng, e_cpu, e_gpu = build_pair(ions(n, kmax, box, cut), F.Engine)
    assert abs(e_gpu - e_cpu) <= 1e-10 * max(1.0, abs(e_cpu))
    np.testing.assert_allclose(eng.total_energy()[1], orc.total_energy()[1], rtol=1e-10, atol=1e-10)


@pytest.mark.parametrize("n,a,b,nbins", [(2, 0, 1, 7), (511, 0, 1, 300), (513, 1, 1, 64), (1200, 0, 0, 5)])
def test_rdf_tiles(n, a, b, nbins):
    cfg, xyz, q, ids, g = ions(n, 3, cut=12.0)
    batch = F.Batch()
    batch.add((cfg, xyz, q, ids, g), seed=1)
    dr = 0.11
    d = xyz[ids == a][:, None] - xyz[ids == b][None]
    d = np.where(d > 30.0, d - 60.0, np.where(d < -30.0, d + 60.0, d))
    r = np.sqrt((d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2])
    if a == b:
        r = r[np.triu_indices(len(r), 1)]
    k = np.floor(r * (1.0 / dr)).ravel()
    counts = np.bincount(k[k < nbins].astype(int), minlength=nbins).astype(np.uint64)
    np.testing.assert_array_equal(batch.rdf(0, a, b, dr, nbins), counts)
    batch.close()
