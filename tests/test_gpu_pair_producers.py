"""Pair stream of the hashed producers against the oracle, bit for bit, where
the producer paths change: no partner, one workgroup of eight-lane groups and
one more, more partners than the stash holds (the emit walk), more candidates
than a group takes (the wave path), and collision groups beside globals."""
import numpy as np
import pytest

import oracle
from avbd_amd import GPUSolver, PhysicsScene, SimSettings, demos
from conftest import flush_print

pytestmark = pytest.mark.gpu


def _spheres(n, diameter, pitch, groups=1):
    """n spheres on a cubic lattice of `pitch`, a few in each collision group."""
    s = PhysicsScene("spheres", SimSettings(iterations=1))
    demos.add_ground(s)
    k = int(np.ceil(n ** (1 / 3)))
    for i in range(n):
        s.addBody((diameter,) * 3, 1.0, 0.5, (i % k * pitch, i // k % k * pitch, 0.5 * diameter + i // (k * k) * pitch),
                  shape=1, collisionGroup=i % groups)
    return s


CASES = {
    "apart": (5, 0.5, 2.0, 1), "group_32": (32, 0.5, 0.45, 1), "group_33": (33, 0.5, 0.45, 1),
    "past_stash": (216, 0.9, 0.5, 1), "past_group": (512, 0.06, 0.045, 1), "groups": (125, 0.5, 0.3, 3),
}


@pytest.mark.parametrize("name", list(CASES))
def test_pair_stream(name):
    flush_print(f"[gpu case] pair producers: {name}")
    s = _spheres(*CASES[name])
    o = oracle.OracleSolver(s)
    with GPUSolver(s) as g:
        for _ in range(2):
            g.step()
            o.step()
            po = np.asarray(o.pairs()).reshape(-1, 2)
            assert np.array_equal(g.pairs(), po)
            assert g.stats().pair_candidates == len(po)
    flush_print(f"  {len(po)} pairs, up to {np.bincount(po[:, 0]).max()} from one producer")
