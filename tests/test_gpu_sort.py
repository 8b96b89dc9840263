"""The spatial sort against numpy's stable sort by the same Morton keys, at
particle counts around a wave's 64, a wave's 512 and a tile's 2048 particles,
with one, two, three and four digit passes; every member of every particle
moves with it."""
import numpy as np
import pytest

from helpers import cfg2d, cfg3d
from sp_hip import ParkerPusher

pytestmark = pytest.mark.gpu


def morton(c, a):
    nd = c["ndim"]
    bits = max(1, int(np.ceil(np.log2(max(c["nx"], c["ny"], c["nz"] if nd == 3 else 1)))))
    shift = max(0, bits - 6)
    key = np.zeros(len(a["x"]), np.int64)
    for k, (q, n, d) in enumerate(zip("xyz"[:nd], ("nx", "ny", "nz"), ("dx", "dy", "dz"))):
        cell = np.clip(np.floor((a[q] - c[q + "min"]) * (1.0 / c[d])), 0, c[n] - 1).astype(np.int64) >> shift
        for b in range(10):
            key |= ((cell >> b) & 1) << (nd * b + k)
    return key


@pytest.mark.parametrize("make,grid", [(cfg2d, 2), (cfg2d, 50), (cfg3d, 16), (cfg3d, 33), (cfg2d, 300)])
@pytest.mark.parametrize("n", [2, 63, 64, 65, 511, 513, 2047, 2048, 2049, 9001])
def test_sort_is_numpys_stable_sort(make, grid, n):
    c = make(grid)
    r = np.random.default_rng(n + grid)
    a = dict(x=r.random(n), y=r.random(n), z=r.random(n), p=r.random(n) + 0.5, v=r.random(n),
             mu=r.random(n), weight=0.5 ** r.integers(0, 5, n), t=r.random(n), dt=r.random(n),
             split_times=r.integers(0, 30, n).astype(np.int8),
             count_flag=r.integers(-6, 2, n).astype(np.int8))
    for k in ("origin", "nsteps_tracked", "nsteps_pushed", "tag_injected", "tag_splitted"):
        a[k] = r.integers(-2**31, 2**31 - 2, n).astype(np.int32)
    a["rng_step"] = r.integers(0, 2**32, n).astype(np.uint32)
    with ParkerPusher(**dict(c, nptl_max=n + 3)) as pz:
        pz.set_particles(a)
        pz.sort_particles()
        g = pz.get_particles()
    o = np.argsort(morton(c, a), kind="stable")
    for k in a:
        np.testing.assert_array_equal(g[k], a[k][o], err_msg=k)
