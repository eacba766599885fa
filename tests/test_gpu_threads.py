"""Solvers and networks in threads of their own while others capture their
graphs: a synchronous copy, fill, allocation or free anywhere in the process
ends a capture under way, so the library keeps the two apart.  Every thread's
results are those it gets alone."""
import threading

import numpy as np
import pytest

from avbd_amd import GPUSolver, WarmStartMLP, demos
from conftest import flush_print

pytestmark = pytest.mark.gpu


def test_captures_beside_copies_and_creates():
    flush_print("[gpu case] graph captures beside copies, creates and training in threads")
    block, stack = demos.soft_block_scene(cells=4, bottom=0.02), demos.stack_scene(height=12)
    rng = np.random.default_rng(3)
    x, t = (rng.standard_normal((500, k)).astype(np.float32) for k in (24, 3))

    def residual(scene):  # new graphs every frame
        with GPUSolver(scene) as g:
            for i in range(10):
                g.stepToResidual(1e-9, 20, 8 + 2 * (i % 2))
            return g.bodyStates()

    def intervals(scene):  # states written and read between frames
        with GPUSolver(scene) as g:
            start = g.bodyStates()
            every = np.arange(len(start[0]), dtype=np.uint32)
            for _ in range(12):
                g.setBodyStates(every, *start)
                g.settings = g.settings  # drops the graphs
                g.step(2)
                ends = g.bodyStates()
            return ends

    def creates(scene):
        for _ in range(6):
            with GPUSolver(scene) as g:
                g.step(2)
                ends = g.bodyStates()
        return ends

    def trains(_):
        net = WarmStartMLP(seed=2)
        for k in range(8):
            net.train(x, t, epochs=1, batch=100, lr=1e-3, seed=k)
        return [net.params, net.forward(x)]

    work = [(residual, block), (residual, stack), (intervals, block), (intervals, stack), (creates, block),
            (creates, stack), (trains, None)]
    alone = [f(scene) for f, scene in work]
    got, failed = [None] * len(work), []

    def run(k):
        try:
            got[k] = work[k][0](work[k][1])
        except Exception as e:  # shown below, from the main thread
            failed.append((work[k][0].__name__, repr(e)))

    threads = [threading.Thread(target=run, args=(k,)) for k in range(len(work))]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not failed, failed
    for a, b in zip(got, alone):
        for p, q in zip(a, b):
            assert np.array_equal(p, q)
