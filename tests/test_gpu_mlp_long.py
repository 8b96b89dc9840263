"""Long training loops on the two-launch path: losses and parameters at the
edges of the loss partials' buffer (4096 steps), and device memory that does
not grow with the number of steps."""
import ctypes as C

import numpy as np
import pytest

from sp_hip import device
from sp_hip.surrogate import Mlp

pytestmark = pytest.mark.gpu

SHAPE = (6, 128, 1, 32)


def data():
    rng = np.random.default_rng(4)
    x = rng.uniform(-1.0, 1.0, (500, SHAPE[0])).astype(np.float32)
    return x, np.sin(x @ rng.standard_normal((SHAPE[0], SHAPE[3]))).astype(np.float32)


@pytest.mark.parametrize("nsteps", [4095, 4096, 4097])
def test_losses_over_the_partials_edge(monkeypatch, nsteps):
    got = []
    for eager in ("0", "1"):
        monkeypatch.setenv("SP_MLP_EAGER", eager)
        with Mlp(*SHAPE, batch_max=64, seed=2) as net:
            net.set_data(*data())
            print("long", nsteps, eager, flush=True)
            got.append((net.train(nsteps, 32, 1e-3, 1e-5, seed=5), net.get_params()))
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


def test_memory_does_not_grow_with_steps():
    free, total = C.c_size_t(), C.c_size_t()

    def left():
        assert device._rt().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    with Mlp(*SHAPE, batch_max=64, seed=2) as net:
        net.set_data(*data())
        net.train(10, 32, 1e-3, 1e-5, seed=5)
        before = left()
        losses = net.train(30000, 32, 1e-3, 1e-5, seed=6)
        # 4 MiB of partials, 120 kB of losses; 1 KiB a step would be 30 MB
        assert before - left() <= 12 << 20
    assert np.isfinite(losses).all()
