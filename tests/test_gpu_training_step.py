"""The fused training step at the edges of its batch split: one group of 16
rows, an odd number of groups, a wave without rows, several slices.  Gradients
against the float64 reference with the kernels' bf16 rounding points: FP32
accumulation moves a value by about 1e-6 of itself, which turns a bf16
rounding (2^-8) in one value of 10^3, each one of 256 terms of a sum: below
5e-3 of a layer's norm.  Two calls give the same bits; an Adam step from
those gradients gives the trained weights."""
import numpy as np
import pytest

from oracle import mlp_ref as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [16, 32, 48, 144, 1040, 8208])
def test_step(fd2lib, B):
    rng = np.random.default_rng(B)
    p = M.init_params(B)
    for l in range(4):
        p[M.B_OFF[l]:M.B_OFF[l] + (65 if l == 3 else 256)] = rng.normal(0, 0.1, 65 if l == 3 else 256)
    x = rng.random((B, 5)).astype(np.float32)
    y = np.zeros((B, 65), np.float32)
    y[:, 0] = rng.uniform(0.05, 0.95, B)
    y[:, 1:] = rng.dirichlet(np.ones(64) * 0.5, B)
    y[::5, 1:] = 0.0
    print(f"[training-step] B={B}", flush=True)
    with fd2lib.Mlp() as net:
        net.set_params(p)
        loss, g = net.gradients(x, y)
        loss2, g2 = net.gradients(x, y)
        assert loss == loss2 and np.array_equal(g, g2)
        rl, rg = M.loss_and_grads(p, x, y, rnd=True)
        assert abs(loss - rl) < 1e-4 * max(1.0, abs(rl))
        for l in range(4):
            for off, size in ((M.W_OFF[l], M.SHAPES[l][0] * M.SHAPES[l][1]),
                              (M.B_OFF[l], M.SHAPES[l][1])):
                a, b = g[off:off + size].astype(np.float64), rg[off:off + size]
                assert np.linalg.norm(a - b) < 5e-3 * np.linalg.norm(b), (l, off)
        # one training step draws its rows from a data set of one repeated row
        net.set_data(np.repeat(x[:1], 7, 0), np.repeat(y[1:2], 7, 0))
        losses, _ = net.train(1, batch=B, lr=1e-3, seed=3)
        w = net.params()
    with fd2lib.Mlp() as net:
        net.set_params(p)
        loss, g = net.gradients(np.repeat(x[:1], B, 0), np.repeat(y[1:2], B, 0))
    assert losses[0] == np.float32(loss)
    g = g.astype(np.float64)
    step = 1e-3 * g / (np.abs(g) + 1e-8 * 1.0)
    # first step: m/c1 = g and sqrt(v/c2) = |g| up to FP32 roundings (1e-6 of lr)
    assert np.abs(w - (p - step)).max() < 1e-5
