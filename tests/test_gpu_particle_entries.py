"""Particle colors read each adjacency entry's word and cloth slot one pass
ahead: particles with fewer, as many and more springs than their lanes, with
slots (springs between particles) and without any in the scene (springs to a
rigid body, whose entries have no slot), against the oracle.

Bound: ten sweeps, each rounding a coordinate below 2 m a few times (the two
sides sum a particle's springs in different orders): 10 x 2 half-ulps of
1.2e-7 m are 2.4e-6 m."""
import numpy as np
import pytest

import oracle
from avbd_amd import GPUSolver
from avbd_amd.scene import PhysicsScene, SimSettings
from conftest import flush_print

pytestmark = pytest.mark.gpu


def _scene(springs, slots):
    s = PhysicsScene("particle springs", SimSettings(iterations=10))
    fixed = s.addBody((0.5, 0.5, 0.1), 0.0, 0.5, (0.0, 0.0, 1.5))
    rng = np.random.default_rng(springs)
    for p in range(5):
        ids = s.addParticle(0.01, 0.05, (0.3 * p - 0.6, 0.1 * p, 1.0), friction=0.3)
        for k in range(springs):
            at = rng.uniform(-0.2, 0.2, 3)
            if slots:
                other = s.addParticle(0.01, 0.0, (0.3 * p - 0.6 + at[0], 0.1 * p + at[1], 1.3 + at[2]), friction=0.3)
                s.addSpring(ids, other, (0, 0, 0), (0, 0, 0), 40.0)
            else:
                s.addSpring(ids, fixed, (0, 0, 0), (float(at[0]), float(at[1]), 0.0), 40.0)
    return s


@pytest.mark.parametrize("lanes", [4, 32])
@pytest.mark.parametrize("slots", [False, True])
@pytest.mark.parametrize("springs", [1, 4, 5, 33, 65])
def test_particle_springs_match_oracle(springs, slots, lanes):
    flush_print(f"[gpu case] {springs} springs a particle, slots={slots}, lanes={lanes}")
    scene = _scene(springs, slots)
    g, o = GPUSolver(scene, lanesPerBody=lanes, sweepMode=1), oracle.OracleSolver(scene)
    g.step()
    o.step()
    g.synchronize()
    err = float(np.abs(g.positions() - o.positions()).max())
    flush_print(f"  max|x_gpu - x_oracle| = {err:.2e}")
    assert err <= 2.4e-6
