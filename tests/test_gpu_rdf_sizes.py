"""The pair-distance histogram at the sizes where its launch changes: particles with and without
a list of the second type (up to 2048 particles none), tiles of 256, runs of 4 to 32; like and
unlike types, an absent type.  Counts equal those of numpy."""
import numpy as np
import pytest

import faunus_amd as F
from tests.test_gpu_observables import host_rdf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 63, 255, 257, 2048, 2049, 2600])
def test_histogram_at_the_edges(n):
    rng = np.random.default_rng(n)
    box = 40.0
    ids = rng.integers(0, 2, n).astype(np.int32)
    ids[:2] = 0, 1
    xyz = rng.uniform(-box / 2, box / 2, (n, 3))
    cfg = {"temperature": 298.15, "geometry": {"type": "cuboid", "length": box},
           "atomlist": [{"A": {"q": 0.1, "sigma": 0.0}}, {"B": {"q": -0.1, "sigma": 0.0}}, {"C": {"q": 0.0, "sigma": 0.0}}],
           "moleculelist": [{"salt": {"atoms": ["A", "B"], "atomic": True}}],
           "energy": [{"nonbonded": {"default": [{"hardsphere": {}},
                                                 {"coulomb": {"type": "fanourgakis", "epsr": 80.0, "cutoff": 10.0}}]}}]}
    b = F.Batch()
    b.add((cfg, xyz, np.where(ids == 0, 0.1, -0.1), ids, dict(begin=[0], size=[n], molid=[0])), seed=1)
    for a, c in ((0, 1), (1, 0), (0, 0), (1, 1), (0, 2), (2, 1)):
        got = b.rdf(0, a, c, 0.3, 70)
        assert np.array_equal(got, host_rdf(xyz, ids, box, a, c, 0.3, 70)), (n, a, c)
    b.close()
