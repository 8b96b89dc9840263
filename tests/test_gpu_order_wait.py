"""Batches of many particles per lane, whose lanes wait for the wave's other
work: the same particles as the same batch with a step budget that is never
reached, which runs in index order and does that work at once.  Sizes: just
over five and over sixteen particles per resident lane, with remainders."""
import numpy as np
import pytest

from helpers import cfg2d
from sp_hip import ParkerPusher, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1000003, 3300001])
def test_waiting_lanes_change_no_particle(n):
    c = cfg2d(64, dt_max_rel=5e-2, pmin=0.5, pmax=2.0, precision="f32")
    nodes = workloads.fields_2d(64, 64)
    k = [n // 2, n // 3, n - n // 2 - n // 3]
    variants = [(1e-4, 0.01, 1.5), (2e-2, 0.3, 1.7), (3e-3, 1e-3, 1.2)]
    out = []
    for budget in (0, 1 << 30):
        print("wait", n, budget, flush=True)
        with ParkerPusher(**dict(c, nptl_max=n, sort_steps=budget)) as pz:
            pz.upload_fields(nodes)
            pz.calc_fields_gradients()
            pz.set_variants(variants)
            pz.inject_variants(k, 1e-7, 1, 5.0, 0.0, 0.0, [(0, 0, 0, 1, 1, 1)] * 3)
            st = [pz.particle_mover(0.02 * i, 0.02, 2, 10) for i in range(2)]
            a = pz.get_particles()
            o = np.argsort(a["tag_injected"], kind="stable")
            out.append(([s["steps"] for s in st], [s["leak"] for s in st], {q: v[o] for q, v in a.items()}))
    assert out[0][:2] == out[1][:2]
    for q in out[0][2]:
        np.testing.assert_array_equal(out[0][2][q], out[1][2][q], err_msg=q)
