"""Contact adjacency of bodies with many contacts: spheres resting on one
dynamic slab, at counts where the segment sort changes path (one lane's
insertion, a wave's ranking of one, two and four registers, insertion again).
The order of a body's entries is the order of its sums, so runs whose scatter
raced differently are equal bit for bit only if every segment is sorted; and
the first frame agrees with the oracle as every scene's does, 1e-5 m."""
import numpy as np
import pytest

import oracle
from avbd_amd import GPUSolver, PhysicsScene, SimSettings, demos
from conftest import flush_print

pytestmark = pytest.mark.gpu


def _slab(n):
    s = PhysicsScene("slab", SimSettings(iterations=2))
    demos.add_ground(s)
    k = int(np.ceil(np.sqrt(n)))
    s.addBody((0.3 * k, 0.3 * k, 0.2), 1.0, 0.5, (0, 0, 0.1))
    for i in range(n):
        s.addSphere(0.25, 1.0, 0.5, ((i % k - (k - 1) / 2) * 0.28, (i // k - (k - 1) / 2) * 0.28, 0.325))
    return s


@pytest.mark.parametrize("n", [7, 8, 63, 64, 130, 254, 255, 300])
def test_many_contacts_on_one_body(n):
    flush_print(f"[gpu case] {n} spheres on one slab")
    s = _slab(n)
    o = oracle.OracleSolver(s)
    o.step()
    runs = []
    for _ in range(2):
        with GPUSolver(s, lanesPerBody=8, sweepMode=1, maxPairsPerBody=64) as g:
            g.step()
            first = g.positions()
            assert g.stats().num_active_manifolds >= n
            g.step(5)
            runs.append(g.bodyStates())
    assert np.abs(first - o.positions()).max() <= 1e-5
    for x, y in zip(*runs):
        assert np.array_equal(x, y)
