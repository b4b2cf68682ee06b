"""Every copy of the weights after training: the row-major one and the forward and
backward fragment orders are refreshed by each Adam step, so a trained network
and a new one with its parameters give the same loss, gradients and logits bit
for bit.  Batches of one slice and of several; the learning rate moves every
weight by several bf16 units per step."""
import numpy as np
import pytest

from oracle import mlp_ref as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,steps", [(48, 3), (1040, 2)])
def test_trained_equals_set(fd2lib, B, steps):
    rng = np.random.default_rng(B)
    x = rng.random((B, 5)).astype(np.float32)
    y = np.zeros((B, 65), np.float32)
    y[:, 0] = rng.uniform(0.05, 0.95, B)
    y[:, 1:] = rng.dirichlet(np.ones(64) * 0.5, B)
    p = M.init_params(B)
    print(f"[trained] B={B}", flush=True)
    with fd2lib.Mlp() as net, fd2lib.Mlp() as new:
        net.set_params(p)
        net.gradients(x, y)  # the fragment orders exist before the first step
        net.set_data(x, y)
        net.train(steps, batch=B, lr=2e-2, seed=1)
        w = net.params()
        moved = np.abs(w - p)[[M.W_OFF[l] + 7 for l in range(4)]]
        assert moved.min() > 1e-3
        new.set_params(w)
        loss, g = net.gradients(x, y)
        loss_n, g_n = new.gradients(x, y)
        assert loss == loss_n and np.array_equal(g, g_n)
        assert np.array_equal(net.logits(x), new.logits(x))
        assert np.array_equal(net.logits(x, layered=True), new.logits(x, layered=True))


@pytest.mark.parametrize("B", [48, 1040])
def test_gradients_leave_training_alone(fd2lib, B):
    """A call for gradients changes nothing of the training that follows."""
    rng = np.random.default_rng(B + 1)
    x = rng.random((B, 5)).astype(np.float32)
    y = np.zeros((B, 65), np.float32)
    y[:, 0] = rng.uniform(0.05, 0.95, B)
    y[:, 1:] = rng.dirichlet(np.ones(64) * 0.5, B)
    runs = []
    for ask in (False, True):
        with fd2lib.Mlp(seed=B) as net:
            net.set_data(x, y)
            if ask:
                net.gradients(x, y)
            losses, _ = net.train(2, batch=B, lr=1e-3, seed=1)
            runs.append((losses, net.params()))
    assert np.array_equal(runs[0][0], runs[1][0]) and np.array_equal(runs[0][1], runs[1][1])
