"""The island kernels (one workgroup per group of independent islands: color,
repair and solve) against the grid-wide sweep on the same scenes: states,
colors, color counts and pair streams equal bit for bit over several frames,
at the sizes where the workgroup split changes -- one body, one wave, several
islands per workgroup, an island larger than its workgroup's lane groups, and
islands past the LDS lists of neighbours and contacts."""
import numpy as np
import pytest

from avbd_amd import GPUSolver, PhysicsScene, SceneJoint, SimSettings, demos
from conftest import flush_print

pytestmark = pytest.mark.gpu


def _lattice(n):
    """n^3 touching unit cubes: every inner cube meets six neighbours."""
    s = PhysicsScene("lattice", SimSettings(iterations=4))
    demos.add_ground(s)
    for i in range(n ** 3):
        s.addBody((1, 1, 1), 1.0, 0.5, (i % n - n / 2, i // n % n - n / 2, 0.5 + i // (n * n)))
    return s


def _spheres(n):
    """n^3 overlapping spheres: more neighbours than the LDS list holds."""
    s = PhysicsScene("spheres", SimSettings(iterations=2))
    demos.add_ground(s)
    for i in range(n ** 3):
        s.addSphere(1.9, 1.0, 0.5, (i % n - n / 2, i // n % n - n / 2, 0.95 + i // (n * n)))
    return s


def _loose():
    """Islands of one body, a sprung pair of particles, a pair jointed to each
    other and bodies of two collision groups over shared ground."""
    s = PhysicsScene("loose", SimSettings(iterations=5))
    demos.add_ground(s)
    for g in range(1, 12):
        s.addBody((0.4, 0.4, 0.4), 1.0, 0.5, (2.0 * g, 0, 0.2), collisionGroup=g)
        s.addBody((0.4, 0.4, 0.4), 1.0, 0.5, (2.0 * g, 0.1, 0.61), collisionGroup=g)
    a = s.addBody((0.3, 0.3, 0.3), 1.0, 0.5, (0, 3, 1), collisionEnabled=False)
    b = s.addBody((0.3, 0.3, 0.3), 1.0, 0.5, (0, 3, 2), collisionEnabled=False)
    s.addJoint(SceneJoint(a, b, (0, 0, 0.5), (0, 0, -0.5)))
    c = s.addBody((0.3, 0.3, 0.3), 1.0, 0.5, (0, 5, 1), collisionEnabled=False)
    d = s.addBody((0.3, 0.3, 0.3), 1.0, 0.5, (0, 5, 2), collisionEnabled=False)
    s.addSpring(c, d, (0, 0, 0), (0, 0, 0), 50.0)
    s.addSpring(d, 0, (0, 0, 0), (0, 5, 1), 50.0, hard=True)
    return s


SCENES = {
    "one_cube": lambda: demos.stack_scene(height=1),
    "stack_33": lambda: demos.stack_scene(height=33),
    "stack_128": lambda: demos.stack_scene(height=128, iterations=4),
    "stack_129": lambda: demos.stack_scene(height=129, iterations=4),   # colored by its workgroup, swept by the grid
    "chain_19": lambda: demos.chain_scene(links=19),
    "batch_5": lambda: demos.batched_scene(5)[0],
    "batch_1500": lambda: demos.batched_scene(1500, iterations=4)[0],
    "loose": _loose,
    "lattice_5": lambda: _lattice(5),     # 125 bodies, past the LDS list of contacts
    "lattice_8": lambda: _lattice(8),
    "spheres_8": lambda: _spheres(8),     # past the LDS list of neighbours
    "lattice_9": lambda: _lattice(9),     # 729 bodies in one island: the grid-wide sweep
}


@pytest.mark.parametrize("lanes", [4, 8])
@pytest.mark.parametrize("name", list(SCENES))
def test_islands_equal_the_grid_sweep(name, lanes):
    flush_print(f"[gpu case] islands vs per-color launches: {name}, lanes={lanes}")
    scene = SCENES[name]()
    with GPUSolver(scene, lanesPerBody=lanes) as a, GPUSolver(scene, lanesPerBody=lanes, sweepMode=1) as b:
        rng = np.random.default_rng(1)
        p, r, v, w = a.bodyStates()
        m = a.bodyMass() > 0
        v[m] += rng.normal(0, 0.3, (int(m.sum()), 3)).astype(np.float32)
        idx = np.arange(len(p), dtype=np.uint32)
        a.setBodyStates(idx, p, r, v, w)
        b.setBodyStates(idx, p, r, v, w)
        for _ in range(4):
            a.step()
            b.step()
            sa, sb = a.stats(), b.stats()
            a.synchronize()
            b.synchronize()
            assert np.array_equal(a.debugColors()[m], b.debugColors()[m])
        for x, y in zip(a.bodyStates(), b.bodyStates()):
            assert np.array_equal(x, y)
        sa, sb = a.stats(), b.stats()
        assert list(sa.color_counts) == list(sb.color_counts) and sa.max_color_used == sb.max_color_used
        assert sa.num_pairs == sb.num_pairs and sa.num_active_manifolds == sb.num_active_manifolds
        na, ra = a.stepToResidual(1e-3, 30, 7)
        nb, rb = b.stepToResidual(1e-3, 30, 7)
        assert (na, ra) == (nb, rb)
        for x, y in zip(a.bodyStates(), b.bodyStates()):
            assert np.array_equal(x, y)
        assert a.timePrimal(reps=2)["avg_launch_us"] > 0.0
