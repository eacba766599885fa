"""The tile kernel (all sweeps of a tetrahedral scene in one launch, tiles
exchanging versioned positions) against one launch per color at the same 32
lanes, over frames of fall, landing and rest and iterated to a residual: one
tile, a few, an odd number and one per CU; with pinned vertices, with particles
on two static bodies at once, and with particles of the block in contact with
each other, where the frames run the grid-wide sweep.

The two paths evaluate the same expressions in the same order, but the
compiler fuses multiply-adds differently in each: an update may differ by one
rounding, 2^-24 of its step, which Gauss-Seidel contracts.  The bound is eight
units in the last place of the scene's extent on positions, and sixty times
that (1 / dt) on velocities."""
import ctypes as C

import numpy as np
import pytest

from avbd_amd import GPUSolver, _capi, demos
from conftest import flush_print

pytestmark = pytest.mark.gpu


def _pinned(cells):
    s = demos.soft_block_scene(cells=cells, bottom=0.3)
    for b in s.bodies[1:1 + (cells + 1)]:
        b["density"] = 0.0
    return s


def _pair(**kw):
    return demos.soft_block_scene(**kw)


def _corner(cells):
    s = demos.soft_block_scene(cells=cells, bottom=0.02)
    s.addBody((0.2, 4.0, 4.0), 0.0, 0.7, (0.61, 0.0, 1.0))
    return s


def _close(a, b):
    pa, ra, va, wa = a.bodyStates()
    pb, rb, vb, wb = b.bodyStates()
    ulp = float(np.abs(pb[1:]).max()) * 2.0 ** -23
    assert np.array_equal(ra, rb) and np.array_equal(wa, wb)
    assert np.abs(pa - pb).max() <= 8 * ulp
    assert np.abs(va - vb).max() <= 8 * ulp * 60


SCENES = {
    "block_1": lambda: _pair(cells=1, bottom=0.02), "block_3": lambda: _pair(cells=3, bottom=0.02),
    "block_4": lambda: _pair(cells=4, bottom=0.02), "block_5": lambda: _pair(cells=5, bottom=0.02, iterations=3),
    "block_9": lambda: _pair(cells=9, bottom=0.02), "block_20": lambda: _pair(cells=20, bottom=0.02),
    "pinned_6": lambda: _pinned(6), "corner_4": lambda: _corner(4),
    "self_contact_7": lambda: _pair(cells=7, bottom=0.02, radius_factor=0.7),
    "too_large_33": lambda: _pair(cells=33, bottom=0.02, iterations=3),
}


@pytest.mark.parametrize("name", list(SCENES))
def test_tiles_equal_the_color_launches(name):
    flush_print(f"[gpu case] tiles vs per-color launches: {name}")
    scene = SCENES[name]()
    with GPUSolver(scene, lanesPerBody=32) as a, GPUSolver(scene, lanesPerBody=32, sweepMode=1) as b:
        p, r, v, w = a.bodyStates()
        v[1:, 2] -= 1.5
        idx = np.arange(len(p), dtype=np.uint32)
        a.setBodyStates(idx, p, r, v, w)
        b.setBodyStates(idx, p, r, v, w)
        for _ in range(6):
            a.step()
            b.step()
        _close(a, b)
        for tol, count in ((0.5, None), (1e-9, 45)):
            (na, xa), (nb, xb) = a.stepToResidual(tol, 45, 10), b.stepToResidual(tol, 45, 10)
            # a converged residual is the rounding of element forces of about 100 m g: 100 * 2^-23 = 1.2e-5
            assert na == nb and (count is None or na == count) and abs(xa - xb) <= 0.01 * xb + 1.2e-5
        a.step(3)
        b.step(3)
        _close(a, b)
        m = a.manifolds()["header"]
        m = m[m[:, 2] > 0]  # active: bodies, contacts
        static = a.bodyMass() <= 0
        between = int((~static[m[:, 0]] & ~static[m[:, 1]]).sum())
        _, touching = np.unique(m[:, :2][~static[m[:, :2]]], return_counts=True)
        flush_print(f"  {len(m)} contacts, {between} between particles, at most {touching.max(initial=0)} of one")
        assert len(m) or name == "pinned_6"
        assert name == "too_large_33" or (between > 0) == (name == "self_contact_7")
        assert name != "corner_4" or touching.max() == 2


def test_tiles_beside_other_solvers():
    """Tile solvers of one, 2 and 256 tiles a scene, a scene swept grid-wide and
    one of islands stepped from threads of their own at once: each ends where it
    ends alone."""
    import threading

    flush_print("[gpu case] tile solvers in threads")

    def solvers():
        rigid = demos.stack_scene(height=140)
        return [GPUSolver(_pair(cells=1, bottom=0.02)), GPUSolver(_pair(cells=2, bottom=0.02)),
                GPUSolver(_pair(cells=14, bottom=0.02)), GPUSolver(rigid, lanesPerBody=4),
                GPUSolver(rigid, lanesPerBody=8, sweepMode=2), GPUSolver(demos.stack_scene(height=6))]

    alone = []
    for g in solvers():
        with g:
            g.step(24)
            alone.append(g.bodyStates())
    together = solvers()

    def run(g):
        for _ in range(4):
            g.step(6)
            g.synchronize()

    threads = [threading.Thread(target=run, args=(g,)) for g in together]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g, want in zip(together, alone):
        with g:
            assert g.runtimeFailure is None
            for x, y in zip(g.bodyStates(), want):
                assert np.array_equal(x, y)


def test_residual_frames_beside_grid_sweeps():
    """Frames of tile solvers iterated to a residual, their graphs captured anew
    for every frame (another chunk length each), and frames that change between
    the tiles and launches per color, captured while a tile frame is in flight,
    while grid-wide sweeps step in other threads: every solver ends where it ends
    alone, and none times out."""
    import threading

    flush_print("[gpu case] residual frames beside grid sweeps")
    rigid = demos.stack_scene(height=140)
    floating, middle = _floating()
    with GPUSolver(floating) as g:
        states = g.bodyStates()
    everything = np.arange(len(states[0]), dtype=np.uint32)

    def solvers():
        return [GPUSolver(_pair(cells=2, bottom=0.02)), GPUSolver(_pair(cells=9, bottom=0.02)),
                GPUSolver(rigid, lanesPerBody=8, sweepMode=2), GPUSolver(rigid, lanesPerBody=4, sweepMode=2),
                GPUSolver(floating)]

    def run(k, g):
        for i in range(5):
            if k < 2:
                g.stepToResidual(1e-9, 40, 8 + 2 * (i % 2))
            elif k == 4:
                p, r, v, w = states
                q = p.copy()
                q[middle] += np.float32([0.04, 0, 0])
                g.settings = g.settings  # drops the graphs
                g.setBodyStates(everything, q, r, v, w)
                g.step(8)
                g.synchronize()
            else:
                g.step(8)
                g.synchronize()

    alone = []
    for k, g in enumerate(solvers()):
        with g:
            run(k, g)
            alone.append(g.bodyStates())
    together = solvers()
    threads = [threading.Thread(target=run, args=(k, g)) for k, g in enumerate(together)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g, want in zip(together, alone):
        with g:
            assert g.runtimeFailure is None
            for x, y in zip(g.bodyStates(), want):
                assert np.array_equal(x, y)


def _floating():
    """A block next to weightless whose inner particles stand 4 % apart, and its middle one."""
    s = demos.soft_block_scene(cells=4, bottom=0.5, radius_factor=0.48, vel_sigma=0.0, iterations=10)
    s.settings.gravity = -0.01
    return s, np.array([1 + (2 * 5 + 2) * 5 + 2], np.uint32)


@pytest.mark.parametrize("graph", [True, False])
def test_inner_contacts_come_and_go(graph):
    """A particle pushed into its neighbour, then apart for longer than the 120
    frames that the tile path stays off, twice: each path's frames continue the
    other's.  A frame may add the bound of _close to the displacements."""
    flush_print(f"[gpu case] contacts inside a block come and go, graphs {graph}")
    scene, middle = _floating()
    with GPUSolver(scene, lanesPerBody=32, useGraph=graph) as a, \
            GPUSolver(scene, lanesPerBody=32, sweepMode=1, useGraph=graph) as b:
        frames = 0

        def step(contacts, modes):
            nonlocal frames
            for want, mode in zip(contacts, modes, strict=True):
                a.step()
                b.step()
                sa = a.stats()
                assert sa.num_active_manifolds == b.stats().num_active_manifolds == want
                assert sa.sweep_mode == mode
            frames += len(contacts)
            pa, ra, va, wa = a.bodyStates()
            pb, rb, vb, wb = b.bodyStates()
            bound = 8 * (1 + frames) * float(np.abs(pb[1:]).max()) * 2.0 ** -23
            assert np.abs(pa - pb).max() <= bound and np.abs(va - vb).max() <= 60 * bound

        def push():
            p, r, v, w = (x[middle] for x in b.bodyStates())
            for g in (a, b):
                g.setBodyStates(middle, p + np.float32([0.04, 0, 0]), r, v, w)

        step([0] * 3, [2] * 3)
        for _ in range(2):
            push()
            step([1, 1] + [0] * 126, [2, 2] + [1] * 121 + [2] * 5)
        for tol in (1e-9, 0.5):
            push()
            for g in (a, b):
                g.stepToResidual(tol, 20, 10)
            frames += 1
            step([1] + [0] * 2, [2, 1, 1] if tol == 1e-9 else [1, 1, 1])


@pytest.mark.parametrize("write", ["all", "shuffled", "noalloc"])
def test_states_written_again_take_the_same_path(write):
    """The same start state three times in one solver, and in a new one: frames on
    the ground, where the two paths round differently, then frames with contacts
    between inner particles, after which the path stays changed for 120 frames:
    the same bits each time."""
    flush_print(f"[gpu case] the same states again, {write}")
    scene = demos.soft_block_scene(cells=4, bottom=0.13, radius_factor=0.48, vel_sigma=0.0, iterations=10)
    runs = []
    rng = np.random.default_rng(5)

    def interval(g):
        order = np.arange(len(p), dtype=np.uint32)
        if write == "shuffled":
            order = rng.permutation(len(p)).astype(np.uint32)
        if write == "noalloc":
            arrays = [np.ascontiguousarray(x[order]) for x in (p, r, v, w)]
            assert g._lib.avbd_set_body_states_noalloc(
                g._h, order.ctypes.data_as(C.POINTER(C.c_uint32)), len(order),
                *[x.ctypes.data_as(C.POINTER(C.c_float)) for x in arrays]) == _capi.OK
        else:
            g.setBodyStates(order, p[order], r[order], v[order], w[order])
        contacts = []
        for _ in range(12):
            g.step()
            contacts.append(g.stats().num_active_manifolds)
        assert contacts[:2] == [25, 25] and max(contacts) > 25  # 25 particles on the ground
        runs.append(g.bodyStates())

    with GPUSolver(scene) as g:
        p, r, v, w = g.bodyStates()
        v[1:, 2] -= 2.0
        for _ in range(3):
            interval(g)
    with GPUSolver(scene) as g:
        interval(g)
    for x in runs[1:]:
        for i, j in zip(x, runs[0]):
            assert np.array_equal(i, j)


def test_touching_as_uploaded_keeps_color_launches():
    """A block whose inner particles overlap at rest ends where one launch per
    color ends, bit for bit (the same lanes), from its first frame."""
    flush_print("[gpu case] inner particles touching as uploaded")
    scene = _pair(cells=7, bottom=0.02, radius_factor=0.7)
    with GPUSolver(scene, lanesPerBody=32) as a, GPUSolver(scene, lanesPerBody=32, sweepMode=1) as b:
        a.step(5)
        b.step(5)
        assert a.stats().sweep_mode == 1
        for x, y in zip(a.bodyStates(), b.bodyStates()):
            assert np.array_equal(x, y)


@pytest.mark.parametrize("kind", ["LOCK_EX", "LOCK_SH"])
def test_another_process_holds_the_device(kind):
    """While another process has the device's lock, a tetrahedral scene runs one
    launch per color at the tiles' lanes, and while it has it alone a rigid scene
    too large for island workgroups does so too, with the same bits; afterwards
    both are as before."""
    import gc
    import glob
    import subprocess
    import sys

    flush_print(f"[gpu case] tile and grid-wide scenes beside another process, {kind}")
    soft, rigid = _pair(cells=4, bottom=0.02), demos.stack_scene(height=520)
    hold = ("import fcntl, sys\n"
            "files = [open(p, 'r+') for p in sys.argv[2:]]\n"
            "for f in files: fcntl.lockf(f, getattr(fcntl, sys.argv[1]) | fcntl.LOCK_NB)\n"
            "print('held', flush=True)\n"
            "sys.stdin.read()\n")

    def ends(scene, mode, lanes, **kw):
        with GPUSolver(scene, lanesPerBody=lanes, **kw) as g:
            g.step(6)
            assert g.stats().sweep_mode == mode
            return g.bodyStates()

    def same(a, b):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)

    gc.collect()  # solvers that earlier tests left open hold the lock for this process
    tiles, grid = ends(soft, 2, 32), ends(rigid, 2, 4, sweepMode=2)
    other = subprocess.Popen([sys.executable, "-c", hold, kind, *glob.glob("/dev/shm/avbd_device_*")],
                             stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True)
    try:
        assert other.stdout.readline().strip() == "held"
        same(ends(soft, 1, 0), ends(soft, 1, 32, sweepMode=1))
        same(ends(rigid, 1 if kind == "LOCK_EX" else 2, 4, sweepMode=2), grid)
    finally:
        other.stdin.close()
        other.wait(timeout=30)
        other.stdout.close()
    same(ends(soft, 2, 0), tiles)
    same(ends(rigid, 2, 4, sweepMode=2), grid)
