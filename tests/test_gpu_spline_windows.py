"""Spline tables whose search window holds more than the four knots that are read at once: a long
range puts many of a table's knots into one of its 256 buckets.  The device's pair energies against
the engine's own tables evaluated on the host, over all intervals, at the knots and on either side
of them, the oracle's exact pair energy below the first knot and zero beyond the last: FP64 within
1e-11 of max(|u|, 1 kT), the FP32 form within 1e-6 of max(|u|, 8 kT) (a pair evaluated in a
neighbouring interval is off by about the tables' own tolerance, 1e-4 kT)."""
import numpy as np
import pytest

import faunus_amd as F
from oracle import oracle as O
from tests import systems

pytestmark = pytest.mark.gpu


def window(knots):
    """The longest search window of a table, as the engine lays it out."""
    n, x0, span = len(knots), knots[0], knots[-1] - knots[0]
    first = [int(np.searchsorted(knots, x0 + k * span / 256 - 1e-9 * span)) for k in range(257)]
    return max(min(n, first[k + 1] + 1) - max(0, first[k] - 1) + 1 for k in range(256))


def splined(table, r2):
    """tabulate.h:184-202: interval by lower_bound, Horner from the top coefficient."""
    knots, c = np.asarray(table["knots"]), np.asarray(table["coeff"]).reshape(-1, 6)
    pos = np.clip(np.searchsorted(knots, r2, side="left") - 1, 0, len(knots) - 2)
    z, s = r2 - knots[pos], np.zeros_like(r2)
    for k in (5, 4, 3, 2, 1):
        s = z * (s + c[pos, k])
    return s + c[pos, 0]


@pytest.mark.parametrize("rmax,utol,longest", [(11.99, 1e-3, 4), (30.0, 1e-3, 6), (60.0, 1e-4, 11), (120.0, 1e-4, 13)])
def test_pairs_over_long_search_windows(rmax, utol, longest):
    cfg = systems.ions([{"nonbonded_splined": {
        "default": [{"lennardjones": {"mixing": "LB"}},
                    {"coulomb": {"type": "fanourgakis", "epsr": 78.7, "cutoff": rmax + 0.01}}],
        "rmax": rmax, "u_at_rmax": 0.1, "utol": utol, "ftol": 1e-1}}], n_pairs=10, box=3 * rmax + 20.0)[0]
    orc, eng = O.System(cfg), F.Engine(cfg)
    charge = (1.0, -1.0)
    seen = 0
    for a, b in ((0, 0), (0, 1), (1, 1)):
        table = eng.splined_table(a, b)
        knots = np.asarray(table["knots"])
        seen = max(seen, window(knots))
        inside = np.concatenate([np.linspace(lo, hi, 41)[1:-1] for lo, hi in zip(knots[:-1], knots[1:])])
        edges = knots[1:-1]
        r2 = np.concatenate([inside, edges, edges * (1 - 1e-12), edges * (1 + 1e-12), [0.9 * knots[0], rmax * rmax, 1.1 * rmax * rmax]])
        want = np.where(r2 < knots[-1], splined(table, r2), 0.0)
        below = r2 <= knots[0]
        want[below] = [orc.pair_energy(a, charge[a], b, charge[b], float(x)) for x in r2[below]]
        u64, u32 = eng.pair_probe(a, b, charge[a], charge[b], r2)
        assert (np.abs(u64 - want) <= 1e-11 * np.maximum(np.abs(want), 1.0)).all(), (a, b)
        assert (np.abs(u32 - want) <= 1e-6 * np.maximum(np.abs(want), 8.0)).all(), (a, b)
    assert seen == longest
    eng.close()
