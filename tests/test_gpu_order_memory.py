"""A batch without sorting whose context leaves no device memory for the work
order's scratch runs in index order, with the same particles; the sort itself
says that it has no memory; both work once there is some."""
import ctypes as C

import numpy as np
import pytest

from helpers import cfg2d
from sp_hip import ParkerPusher, SpError, device, workloads

pytestmark = pytest.mark.gpu

NMAX = 400_000_000     # scratch: four arrays of 1.6 GB


def test_batch_without_scratch_memory():
    n = 300_007
    c = cfg2d(64, dt_max_rel=5e-2, pmin=0.5, pmax=2.0, precision="f32", sort_every=0)
    nodes = workloads.fields_2d(64, 64)
    k = [n // 2, n // 3, n - n // 2 - n // 3]
    out = []
    for tight in (False, True):
        print("scratch", tight, flush=True)
        with ParkerPusher(**dict(c, nptl_max=NMAX if tight else n)) as pz:
            pz.upload_fields(nodes)
            pz.calc_fields_gradients()
            pz.set_variants([(1e-4, 0.01, 1.5), (2e-2, 0.3, 1.7), (3e-3, 1e-3, 1.2)])
            pz.inject_variants(k, 1e-7, 1, 5.0, 0.0, 0.0, [(0, 0, 0, 1, 1, 1)] * 3)
            ballast = None
            if tight:
                # room for the first of the four arrays, not for the second
                free, total = C.c_size_t(), C.c_size_t()
                assert device._rt().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
                ballast = device.DeviceArray(free.value - 2_500_000_000, np.uint8)
            st = [pz.particle_mover(0.0, 0.05, 1, 10)]
            if tight:
                with pytest.raises(SpError, match="no memory"):
                    pz.sort_particles()
                ballast.free()
            st.append(pz.particle_mover(0.05, 0.05, 1, 10))
            pz.sort_particles()
            a = pz.get_particles()
            o = np.argsort(a["tag_injected"], kind="stable")
            out.append(([s["steps"] for s in st], {q: v[o] for q, v in a.items()}))
    assert out[0][0] == out[1][0]
    for q in out[0][1]:
        np.testing.assert_array_equal(out[0][1][q], out[1][1][q], err_msg=q)
