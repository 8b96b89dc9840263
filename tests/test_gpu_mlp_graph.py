"""Training loops that the two-launch step does not take (other widths, more
than five hidden layers, SP_MLP_UNFUSED=1) record one step as a HIP graph and
replay it: every chunk of replays, with other work on the stream between
chunks, equals the same steps launched one by one."""
import numpy as np
import pytest

from sp_hip.surrogate import Mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,unfused", [
    ((6, 64, 3, 64), False), ((6, 256, 6, 64), False), ((20, 128, 2, 32), False), ((6, 256, 4, 64), True)])
def test_graph_replays_equal_single_launches(monkeypatch, shape, unfused):
    rng = np.random.default_rng(shape[1])
    x = rng.uniform(-1.0, 1.0, (4000, shape[0])).astype(np.float32)
    t = np.sin(x @ rng.standard_normal((shape[0], shape[3]))).astype(np.float32)
    if unfused:
        monkeypatch.setenv("SP_MLP_UNFUSED", "1")
    with Mlp(*shape, seed=9, batch_max=1024) as g, Mlp(*shape, seed=9, batch_max=1024) as e:
        g.set_data(x, t)
        e.set_data(x, t)
        first = None
        for k in range(3):
            print("graph", shape, unfused, k, flush=True)
            lg = g.train(40, batch=1000, lr0=1e-3, lr_min=1e-4, seed=3)
            monkeypatch.setenv("SP_MLP_EAGER", "1")
            le = e.train(40, batch=1000, lr0=1e-3, lr_min=1e-4, seed=3)
            monkeypatch.delenv("SP_MLP_EAGER")
            np.testing.assert_array_equal(g.forward(x[:300]), e.forward(x[:300]))
            np.testing.assert_array_equal(lg, le)
            np.testing.assert_array_equal(g.get_params(), e.get_params())
            first = lg[0] if first is None else first
        assert lg[-1] < first
