"""GPU training steps against the loss gradient and a float64 Adam: the batch
rows read through the shuffle, tiles shared by the waves of a workgroup and
the fused update, at batches below, at and above a 16-row tile, with rows that
the last partial batch drops, over two calls (moments carry over, gradient
sums start at zero).

Bound: Adam divides by its own root, so a step's error is lr times the
relative error of the gradient entry.  Both gradients are bf16 products summed
in f32 in different orders: an entry differs by up to about 1e-5 of the largest
one, so entries above 1e-2 of it by 1e-3 relative (the bound below is 1e-2 lr
per step).  The operand layouts must be those of the final parameters: the
forward pass is bitwise the one after uploading them again."""
import numpy as np
import pytest

from avbd_amd import WarmStartMLP
from conftest import flush_print

pytestmark = pytest.mark.gpu

M64 = (1 << 64) - 1


def _shuffled(n, seed):
    o, s = list(range(n)), seed
    for i in range(n - 1, 0, -1):
        s = (s + 0x9E3779B97F4A7C15) & M64
        z = s
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M64
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
        z ^= z >> 31
        j = z % (i + 1)
        o[i], o[j] = o[j], o[i]
    return np.array(o)


@pytest.mark.parametrize("outputs,n,batch", [(3, 1, 1), (6, 15, 15), (3, 33, 16), (6, 70, 32), (3, 300, 300),
                                             (3, 9000, 4500)])
def test_training_steps(outputs, n, batch):
    flush_print(f"[gpu case] MLP training steps, {outputs} outputs, {n} rows, batches of {batch}")
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, 24)).astype(np.float32)
    t = rng.standard_normal((n, outputs)).astype(np.float32)
    lr = 1e-3
    net, ref = WarmStartMLP(seed=4, outputs=outputs), WarmStartMLP(seed=4, outputs=outputs)
    p = ref.params.astype(np.float64)
    m, v, step = np.zeros_like(p), np.zeros_like(p), 0
    sure = np.ones(len(p), bool)
    for call in range(2):
        loss = net.train(x, t, epochs=1, batch=batch, lr=lr, seed=call)
        order, means = _shuffled(n, call), []
        for k in range(n // batch):
            rows = order[k * batch:(k + 1) * batch]
            ref.params = p.astype(np.float32)
            l, g = ref.lossGrad(x[rows], t[rows])
            means.append(l)
            step += 1
            g = g.astype(np.float64)
            sure &= np.abs(g) > 1e-2 * np.abs(g).max()
            m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
            p -= lr * (m / (1 - 0.9 ** step)) / (np.sqrt(v / (1 - 0.999 ** step)) + 1e-8)
        # the loss of a batch moves by less than its gradient's bound
        assert abs(loss[0] - np.mean(means)) <= 1e-2 * np.mean(means)
        err = np.abs(net.params - p)
        flush_print(f"  call {call}: {int(sure.sum())} entries, max error {err[sure].max() / lr:.1e} lr")
        assert sure.any() and err[sure].max() <= 1e-2 * lr * step
        assert err.max() <= 2.2 * lr * step  # an entry of no certain sign moves by at most a step either way
    y = net.forward(x[:100])
    net.params = net.params
    assert np.array_equal(y, net.forward(x[:100]))


@pytest.mark.parametrize("outputs,n,batch", [(3, 50, 97), (6, 20000, 97), (3, 9000, 512), (3, 12000, 4096),
                                             (3, 20000, 17000)])
def test_training_repeats_bit_for_bit(outputs, n, batch):
    """Sums over workgroups in a fixed order: one and several parts of the
    weight and of the bias sums, more row tiles than parts."""
    flush_print(f"[gpu case] repeated MLP training, {outputs} outputs, {n} rows, batches of {batch}")
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, 24)).astype(np.float32)
    t = rng.standard_normal((n, outputs)).astype(np.float32)
    runs = []
    for _ in range(3):
        net = WarmStartMLP(seed=4, outputs=outputs)
        loss = net.train(x, t, epochs=2, batch=batch, lr=1e-3, seed=9)
        l, g = net.lossGrad(x[:5000], t[:5000])
        runs.append((net.params, loss, l, g))
    for r in runs[1:]:
        for a, b in zip(r, runs[0]):
            assert np.array_equal(a, b)
