"""The sampler's training step at the edges of its tiles, workgroups and batches.

Gradients of row counts around a tile (16), a workgroup (64) and a pass of all
of them (4,096) against the FP64 oracle with the same rounding points, with
the bounds of test_gpu_mlp; steps against Adam in float32 on the gradients of
the same rows (equal rows, so that the shuffled order does not matter); and the
mean loss of many batches, which are read back in groups.
"""
import ctypes

import numpy as np
import pytest

import oracle
from compound_ray_amd import eyerenderer as er
from test_gpu_mlp import IN, P, loss_grad, params_of, set_params

pytestmark = pytest.mark.gpu


def train(lib, x, t, epochs, batch, lr, seed=3):
    losses = np.zeros(epochs, np.float32)
    rc = lib.mlpTrain(x.ctypes.data_as(ctypes.c_void_p), t.ctypes.data_as(ctypes.c_void_p), x.shape[0], epochs, batch,
                      ctypes.c_float(lr), seed, losses.ctypes.data_as(ctypes.c_void_p))
    assert rc == 0, er.last_error(lib)
    return losses


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1025, 4095, 4096, 4097, 12289])
def test_gradient_sizes(lib, n):
    rng = np.random.default_rng(n)
    x = rng.normal(size=(n, IN)).astype(np.float32)
    t = rng.normal(size=n).astype(np.float32)
    assert lib.mlpInit(11) == 0
    loss, g = loss_grad(lib, x, t)
    _, want, wloss = oracle.mlp_loss_grad(params_of(lib), x, t, mode=1)
    assert abs(loss - wloss) <= 1e-3 * max(1.0, wloss)
    at = 0
    for size in (IN * 64, 64, 4096, 64, 4096, 64, 64, 1):
        d = np.linalg.norm(g[at:at + size] - want[at:at + size])
        assert d <= 1e-2 * np.linalg.norm(want[at:at + size]) + 1e-7, (at, d)
        at += size


@pytest.mark.parametrize("n,batch", [(16, 16), (48, 16), (70, 32), (5, 100)])
def test_steps_are_adam(lib, n, batch):
    rng = np.random.default_rng(n)
    x = np.repeat(rng.normal(size=(1, IN)), n, 0).astype(np.float32)
    t = np.full(n, 0.7, np.float32)
    f = np.float32
    assert lib.mlpInit(5) == 0
    start = w = params_of(lib)
    m = np.zeros(P, f)
    v = np.zeros(P, f)
    lr = f(1e-2)
    for k, b0 in enumerate(range(0, n, batch), 1):
        rows = min(batch, n - b0)
        set_params(lib, w)
        _, g = loss_grad(lib, x[:rows], t[:rows])
        m = f(0.9) * m + f(0.1) * g
        v = f(0.999) * v + f(0.001) * g * g
        w = w - lr * (m / f(1 - 0.9 ** k)) / (np.sqrt(v / f(1 - 0.999 ** k)) + f(1e-8))
    set_params(lib, start)
    train(lib, x, t, 1, batch, float(lr))
    # the corrections' powers are float32 on one side: 1 - 0.999^k to 1e-4
    # relative, so a step of at most lr to half of that
    assert np.max(np.abs(params_of(lib) - w)) <= 1e-4 * float(lr) * -(-n // batch)


@pytest.mark.parametrize("n,batch", [(1030, 1), (2050, 2), (1000, 64), (4100, 4096)])
def test_epoch_loss(lib, n, batch):
    """Without a learning rate the epochs' mean losses are that of all rows."""
    rng = np.random.default_rng(n)
    x = rng.normal(size=(n, IN)).astype(np.float32)
    t = rng.normal(size=n).astype(np.float32)
    assert lib.mlpInit(6) == 0
    before = params_of(lib)
    loss, _ = loss_grad(lib, x, t)
    assert np.allclose(train(lib, x, t, 2, batch, 0.0), loss, rtol=1e-5)
    assert np.array_equal(params_of(lib), before)
