"""The 3D FP16 mover's default grid with an acceleration region, for populations
that fill one block per CU but not two: as one block per CU (two took 1.24
times as long), and the same particles."""
import numpy as np
import pytest

from sp_hip import ParkerPusher, workloads

pytestmark = pytest.mark.gpu


def test_half_filled_second_block(monkeypatch):
    n, g = 100_000, 64
    c = dict(workloads.config_3d(g), precision="f32h", nptl_max=n + 8, kpara0=1e-3, dt_max_rel=1e-2,
             dt_min_rel=1e-4, acc_region_flag=1, acc_region=(0.1, 0.8, 0.2, 0.9, 0.0, 0.7))
    nodes = workloads.fields_3d(g, seed=5)
    dtf = workloads.interval_2d(g, 300, 1e-3)
    ms, last = [], []
    for blocks in (None, "1"):
        if blocks:
            monkeypatch.setenv("SP_MOVER_BLOCKS_PER_CU", blocks)
        with ParkerPusher(**c) as pz:
            pz.upload_fields(nodes)
            pz.calc_fields_gradients()
            got = []
            for _ in range(5):
                pz.set_particles({k: v[:0] for k, v in pz.get_particles().items()})
                pz.inject_particles_spatial_uniform(n, 1e-7, 1, 5.0, 0.0, 0.0, (0, 0, 0, 1, 1, 1))
                got.append(pz.particle_mover(0.0, dtf, 1, 10)["kernel_ms"])
            ms.append(np.median(got[1:]))
            a = pz.get_particles()
            last.append({k: v[np.argsort(a["tag_injected"], kind="stable")] for k, v in a.items()})
    print("half filled", ms, flush=True)
    for k in last[0]:
        np.testing.assert_array_equal(last[0][k], last[1][k], err_msg=k)
    assert ms[0] <= 1.1 * ms[1]
