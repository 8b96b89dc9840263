"""FP64 steps with operands that are not finite or too large, against the
oracle bit for bit (signs of zeros aside): infinite and huge momenta,
infinite times, gradients that overflow; increments and given time steps that
are infinite, NaN or negative."""
import numpy as np
import pytest

import oracle
from helpers import cfg2d, cfg3d, grid_shape, nodes_for, random_states
from sp_hip import ParkerPusher

pytestmark = pytest.mark.gpu

COLS = ("x", "y", "z", "p", "t", "dt")


def compare(c, nodes, a, r, fixed):
    prm = oracle.params(c)
    fa = [oracle.gradients(prm, f) for f in nodes]
    with ParkerPusher(**dict(c, precision="f64", nptl_max=16)) as pz:
        for k, f in enumerate(nodes):
            pz.upload_fields(f, k)
            pz.calc_fields_gradients(k)
        st, d = pz.step_once(np.stack([a[k] for k in COLS], 1), r, fixed, 0.0, 0.037)
    for i in range(len(a)):
        row, dr = oracle.step_once(prm, fa[0], a[i], 0.0, 0.037, fixed[i], r[i], *fa[1:])
        np.testing.assert_array_equal(st[i], [row[k] for k in COLS], err_msg=str(i))
        np.testing.assert_array_equal(d[i], dr, err_msg=str(i))
    return st


@pytest.mark.parametrize("acc", [0, 1])
@pytest.mark.parametrize("ndim,n,ti", [(2, 33, 0), (2, 33, 1), (3, 11, 0), (3, 11, 1)])
def test_steps_with_special_operands(ndim, n, ti, acc):
    c = (cfg2d if ndim == 2 else cfg3d)(n, momentum_dependency=0, mag_dependency=0, p0=1.3, time_interp=ti,
                                        acc_region_flag=acc, acc_region=(0.0, 0.5, 0.0, 1.0, 0.0, 1.0))
    rng = np.random.default_rng(ndim)
    nodes = [nodes_for(c, seed=s) for s in (7, 8)[:1 + ti]]
    for f in nodes:    # some cells with velocities whose gradients overflow
        far = rng.random(grid_shape(c)) < 0.02
        f[..., 0][far] = rng.choice([-1e38, 1e38], far.sum())
    a = random_states(c, 1600, seed=5)
    k = np.arange(len(a)) % 8
    a["p"][k == 1] = np.inf
    a["p"][k == 2] = 1.7e308
    a["p"][k == 3] = 1e-290
    a["p"][k == 4] = 0.0
    a["t"][k == 5] = np.inf
    r = rng.uniform(-1.7, 1.7, (len(a), 4))
    fixed = (rng.random(len(a)) < 0.2).astype(np.int8)
    st = compare(c, nodes, a, r, fixed)
    assert np.isfinite(st[:, 3]).any() and not np.isfinite(st[:, 3]).all()


@pytest.mark.parametrize("ndim", [2, 3])
def test_infinite_momentum_with_kappas_momentum_dependence(ndim):
    c = (cfg2d if ndim == 2 else cfg3d)(24 if ndim == 2 else 11, momentum_dependency=1, mag_dependency=0, p0=1.3,
                                        acc_region_flag=1, acc_region=(0.0, 0.5, 0.0, 1.0, 0.0, 1.0))
    a = random_states(c, 200, seed=6)
    a["p"] = np.inf
    r = np.random.default_rng(1).uniform(-1.7, 1.7, (len(a), 4))
    compare(c, [nodes_for(c)], a, r, np.zeros(len(a), np.int8))


@pytest.mark.parametrize("acc", [0, 1])
@pytest.mark.parametrize("ndim,n", [(2, 33), (3, 11)])
def test_steps_with_special_increments(ndim, n, acc):
    c = (cfg2d if ndim == 2 else cfg3d)(n, momentum_dependency=0, mag_dependency=0, p0=1.3, acc_region_flag=acc,
                                        acc_region=(0.0, 0.5, 0.0, 1.0, 0.0, 1.0))
    a = random_states(c, 800, seed=8)
    rng = np.random.default_rng(ndim)
    k = np.arange(len(a)) % 8
    r = rng.uniform(-1.7, 1.7, (len(a), 4))
    r[k == 1, 3] = np.inf
    r[k == 2, 3] = np.nan
    r[k == 3, 0] = np.inf
    fixed = (rng.random(len(a)) < 0.2).astype(np.int8)
    fixed[k >= 4] = 1
    a["dt"][k == 4] = -1e-5
    a["dt"][k == 5] = np.inf
    a["dt"][k == 6] = np.nan
    compare(c, [nodes_for(c)], a, r, fixed)
