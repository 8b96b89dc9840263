"""Training where device memory has no room for the two-launch step's own
buffers takes the layer kernels instead, with the same losses and parameters;
once there is room it takes the two launches."""
import ctypes as C

import numpy as np
import pytest

from sp_hip import device
from sp_hip.surrogate import Mlp

pytestmark = pytest.mark.gpu

SHAPE = (6, 256, 4, 64)
BATCH = 2_000_000       # activations and gradients as fragments: 4.2 GB each


def test_training_without_memory_for_fragments():
    rng = np.random.default_rng(4)
    x = rng.uniform(-1.0, 1.0, (5000, SHAPE[0])).astype(np.float32)
    t = np.sin(x @ rng.standard_normal((SHAPE[0], SHAPE[3]))).astype(np.float32)
    got = []
    for tight in (False, True):
        with Mlp(*SHAPE, batch_max=BATCH, seed=2) as net:
            net.set_data(x, t)
            ballast = None
            if tight:
                # room for the activations' fragments, not for the gradients'
                free, total = C.c_size_t(), C.c_size_t()
                assert device._rt().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
                ballast = device.DeviceArray(free.value - 6_500_000_000, np.uint8)
            print("memory", tight, flush=True)
            losses = [net.train(2, BATCH, 1e-3, 1e-5, seed=5)]
            if tight:
                ballast.free()
            losses.append(net.train(2, BATCH, 1e-3, 1e-5, seed=6))
            got.append((np.concatenate(losses), net.get_params()))
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)
