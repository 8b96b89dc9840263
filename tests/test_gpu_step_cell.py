"""The cell of a particle far outside the grid is the outermost one, on either
side of every axis: a position of +-2^40 (2^45 cells, beyond a 32-bit
cell number, exact in FP64) has the offset 0 inside its cell, so its
increments are those of a particle on that cell's first node."""
import numpy as np
import pytest

from helpers import cfg2d, cfg3d, nodes_for
from sp_hip import ParkerPusher

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ndim,precision", [(2, "f64"), (2, "f32"), (2, "f32h"), (3, "f64"), (3, "f32"), (3, "f32h")])
def test_positions_far_outside_take_the_outermost_cell(ndim, precision):
    n = 32 if ndim == 2 else 16      # powers of two: the node positions are exact
    c = cfg2d(n) if ndim == 2 else cfg3d(n)
    lo, hi = [], []
    for k in "xyz"[:ndim]:
        d = (c[k + "max"] - c[k + "min"]) / n
        lo.append(c[k + "min"] - 2 * d)
        hi.append(c[k + "max"])
    mid = [c[k + "min"] + 0.37 * (c[k + "max"] - c[k + "min"]) for k in "xyz"]
    near, far = [], []
    for axis in range(ndim):
        for at, out in ((lo[axis], -2.0**40), (hi[axis], 2.0**40)):
            p = list(mid) + [1.3, 0.0, 1e-4]
            near.append(p[:axis] + [at] + p[axis + 1:])
            far.append(p[:axis] + [out] + p[axis + 1:])
    r = np.random.default_rng(3).uniform(-1.7, 1.7, size=(len(near), 4))
    fixed = np.zeros(len(near), np.int8)
    with ParkerPusher(**dict(c, precision=precision, nptl_max=100)) as pz:
        pz.upload_fields(nodes_for(c))
        pz.calc_fields_gradients()
        s1, d1 = pz.step_once(np.array(near), r, fixed, 0.0, 0.05)
        s2, d2 = pz.step_once(np.array(far), r, fixed, 0.0, 0.05)
    assert np.all(np.isfinite(d1)) and np.any(d1 != 0.0)
    np.testing.assert_array_equal(d2, d1)
    np.testing.assert_array_equal(s2[:, 3:], s1[:, 3:])
