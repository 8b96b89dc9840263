"""The two-launch training step against the layer-by-layer kernels
(SP_MLP_EAGER=1): the same accumulation orders and rounding points, so the
same losses and parameters bit for bit, over batch sizes around the 32-row
blocks, the 128-row splits and the 16-row bias chunks, and over the network
shapes it serves."""
import numpy as np
import pytest

from sp_hip.surrogate import Mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,batch", [
    ((6, 256, 4, 64), 1), ((6, 256, 4, 64), 33), ((6, 256, 4, 64), 257), ((6, 256, 4, 64), 4096),
    ((6, 256, 4, 64), 8192), ((6, 256, 2, 64), 8191), ((16, 256, 1, 128), 512), ((5, 256, 5, 32), 1000),
    ((6, 128, 2, 32), 200), ((1, 128, 5, 128), 2049), ((6, 128, 1, 64), 96)])
def test_training_steps_equal_layer_kernels(monkeypatch, shape, batch):
    rng = np.random.default_rng(batch)
    x = rng.uniform(-1.0, 1.0, (3000, shape[0])).astype(np.float32)
    t = np.sin(x @ rng.standard_normal((shape[0], shape[3]))).astype(np.float32)
    got = []
    for eager in ("0", "1"):
        monkeypatch.setenv("SP_MLP_EAGER", eager)
        with Mlp(*shape, batch_max=max(batch, 64), seed=21) as net:
            net.set_data(x, t)
            print("train", shape, batch, eager, flush=True)
            # two runs: the second starts from the fragments the first left
            losses = [net.train(6, batch, 3e-3, 1e-4, seed=5), net.train(3, batch, 1e-3, 1e-4, seed=6)]
            y = net.forward(x[:77])
            net.train_step(x[:50], t[:50], 1e-3)
            losses.append(net.train(1, batch, 1e-3, 1e-4, seed=7))
            got.append((np.concatenate(losses), net.get_params(), y))
    for a, b in zip(*got):
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, b)
