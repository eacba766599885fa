"""The lane split of surface scenes of particles follows the bodies of the
largest color and no timing: the same at every create, at the sizes on both
sides of every line, so that two solvers of one scene give the same bits."""
import numpy as np
import pytest

from avbd_amd import GPUSolver, demos
from conftest import flush_print

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,lanes", [(12, 16), (24, 16), (26, 32), (64, 32), (65, 16), (178, 16), (180, 8), (256, 8)])
def test_sheet_split(n, lanes):
    flush_print(f"[gpu case] lane split of an {n}^2 sheet")
    scene = demos.cloth_scene(n=n, iterations=3)
    ends = []
    for _ in range(2):
        with GPUSolver(scene) as g:
            assert g.stats().lanes_per_body == lanes
            g.step(3)
            ends.append(g.bodyStates())
    for x, y in zip(*ends):
        assert np.array_equal(x, y)


def test_the_caller_still_chooses():
    flush_print("[gpu case] lane split given by the caller")
    for lanes in (4, 8, 32):
        with GPUSolver(demos.cloth_scene(n=12), lanesPerBody=lanes) as g:
            assert g.stats().lanes_per_body == lanes
