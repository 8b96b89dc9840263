"""The FP64 step's divisions by constants round as IEEE divisions do.

Without kappa's momentum and |B| dependence a step calls no pow, so the
single-step kernel must give the oracle's bits (signs of zeros aside) on
grids, momenta and intervals whose reciprocals are inexact."""
import numpy as np
import pytest

import oracle
from helpers import cfg2d, cfg3d, nodes_for, random_states
from sp_hip import ParkerPusher

pytestmark = pytest.mark.gpu

COLS = ("x", "y", "z", "p", "t", "dt")


@pytest.mark.parametrize("ndim,n,ti", [(2, 47, 0), (2, 33, 1), (3, 11, 0), (3, 13, 1)])
def test_step_without_powers_is_bit_exact(ndim, n, ti):
    c = (cfg2d if ndim == 2 else cfg3d)(n, momentum_dependency=0, mag_dependency=0, p0=1.3,
                                        time_interp=ti)
    if ndim == 2:   # cells that are not square: the dt rule's smallest half cell is dy's
        c.update(ny=n + 6, dy=1.0 / (n + 6))
    nodes = [nodes_for(c, seed=s) for s in (7, 8)[:1 + ti]]
    prm = oracle.params(c)
    fa = [oracle.gradients(prm, f) for f in nodes]
    a = random_states(c, 1500, seed=5)
    r = np.random.default_rng(6).uniform(-1.7, 1.7, size=(len(a), 4))
    fixed = (np.arange(len(a)) % 5 == 0).astype(np.int8)
    t0, dtf = 0.0, 0.037
    with ParkerPusher(**dict(c, precision="f64", nptl_max=16)) as pz:
        for k, f in enumerate(nodes):
            pz.upload_fields(f, k)
            pz.calc_fields_gradients(k)
        st, d = pz.step_once(np.stack([a[k] for k in COLS], 1), r, fixed, t0, dtf)
    for i in range(len(a)):
        row, dr = oracle.step_once(prm, fa[0], a[i], t0, dtf, fixed[i], r[i], *fa[1:])
        np.testing.assert_array_equal(st[i], [row[k] for k in COLS], err_msg=str(i))
        np.testing.assert_array_equal(d[i], dr, err_msg=str(i))


@pytest.mark.parametrize("acc,mag", [(0, 0), (1, 1)])
def test_3d_record_cache_changes_no_bit(acc, mag):
    """A budget of one step per launch starts nearly every step with an empty
    cache; without a budget a lane's records serve until the cell changes."""
    c = cfg3d(13, pbcx=1, dt_max_rel=1e-3, acc_region_flag=acc, mag_dependency=mag,
              acc_region=(0.1, 0.8, 0.2, 0.9, 0.0, 0.7))
    out = []
    for budget in (0, 1):
        with ParkerPusher(**dict(c, precision="f64", nptl_max=4000, sort_steps=budget)) as pz:
            pz.upload_fields(nodes_for(c), 0)
            pz.calc_fields_gradients(0)
            pz.inject_particles_spatial_uniform(3000, 1e-7, 1, 5.0, 0.0, 0.05, (0, 0, 0, 1, 1, 1))
            st = pz.particle_mover(0.0, 0.05, 2, 10)
            a = pz.get_particles()
            o = np.argsort(a["tag_injected"])
            out.append((st["steps"], {k: v[o] for k, v in a.items()}))
    assert out[0][0] == out[1][0]
    for k in out[0][1]:
        np.testing.assert_array_equal(out[0][1][k], out[1][1][k], err_msg=k)
