"""The surface pair stream between its count and emit passes: the count pass
keeps 32 partners of every producer and the wave path walks the buckets again
for producers with more.  Two sheets queried with radii that give producers
no partner, a few, exactly 32 and more, at particle and edge counts around
the 16-, 32- and 64-lane groups, must list the oracle's pairs in its order (whole
numbers: no tolerance)."""
import numpy as np
import pytest

import oracle
from avbd_amd import GPUSolver
from conftest import flush_print
from dat_fixtures import sheets_fired

pytestmark = pytest.mark.gpu

KEPT = 32


@pytest.mark.parametrize("n,radius", [(2, 0.031), (3, 0.0237), (4, 0.0305), (8, 0.0101), (8, 0.0293), (13, 0.0123),
                                      (18, 0.0147), (18, 0.0221)])
def test_pair_stream_matches_oracle(n, radius):
    flush_print(f"[gpu case] surface pairs of two {n}x{n} sheets, query radius {radius}")
    scene = sheets_fired(gap=0.009, n=n, speed=0.0)[0]
    g, o = GPUSolver(scene), oracle.OracleSolver(scene)
    g.setDATQueryRadiusForTesting(radius)
    o.setDatTestHooks(queryRadius=radius, pairCapacity=0, softCapacity=0)
    for s in (g, o):
        s.step()
    g.synchronize()
    pg, po = g.datPairs(), o.datPairs()
    _, per = np.unique(po[:, :2], axis=0, return_counts=True)
    flush_print(f"  {len(po)} pairs, {per.min()} to {per.max()} of a producer, {int((per == KEPT).sum())} with {KEPT}")
    assert np.array_equal(pg, po)
    if n == 18 and radius > 0.02:
        assert per.min() < KEPT < per.max() and (per == KEPT).any()
    g.step()  # the second frame starts from a cleared list of large producers
    o.step()
    g.synchronize()
    assert np.array_equal(g.datPairs(), o.datPairs())
