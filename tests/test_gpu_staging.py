"""Rows and histograms that cross the pinned host staging in pieces: sizes at
the edges of a 64-row block, a 2304-row piece and a group of four pieces, and
local maps at the edges of a piece (32768 bins) and over two groups."""
import numpy as np
import pytest

import oracle
from helpers import cfg2d, nodes_for, random_states
from sp_hip import ParkerPusher

pytestmark = pytest.mark.gpu

SQ3 = np.sqrt(3.0)
STATE_COLS = ("x", "y", "z", "p", "t", "dt")


@pytest.mark.parametrize("nlgc", [0, 1])
def test_rows_in_pieces(nlgc):
    c = cfg2d(32, nlgc=nlgc, **(dict(kperp_kpara=0.05) if nlgc else {}))
    big = 8 * 2304 + 65
    a = random_states(c, big, seed=5)
    a["mu"] = np.random.default_rng(6).uniform(-0.99, 0.99, big)
    st = np.stack([a[k] for k in STATE_COLS], 1)
    rng = np.random.default_rng(7)
    r = rng.uniform(-SQ3, SQ3, size=(big, 4))
    fixed = rng.integers(0, 2, big).astype(np.int8)
    with ParkerPusher(**dict(c, precision="f64", nptl_max=big)) as pz:
        pz.upload_fields(nodes_for(c))
        pz.calc_fields_gradients()
        pz.set_particles(oracle.soa_from_particles(a))   # NLGC: row i takes mu of particle i
        for n in (1, 63, 64, 65, 2303, 2304, 2305, 9216, 9217, 18432, big):
            print("rows", nlgc, n, flush=True)
            s1, d1 = pz.step_once(st[:n], r[:n], fixed[:n], 0.0, 0.05)
            s2, d2 = pz.step_once(st[:n], r[:n], fixed[:n], 0.0, 0.05, noalloc=True)
            np.testing.assert_array_equal(s1, s2)
            np.testing.assert_array_equal(d1, d2)
            assert np.any(s1[-1] != st[n - 1])


@pytest.mark.parametrize("npbins", [7, 8, 9, 32, 33, 97])
def test_histograms_in_pieces(npbins):
    c = cfg2d(64)
    a = random_states(c, 30000, seed=8, slack=False)
    a["p"] = np.exp(np.random.default_rng(9).uniform(np.log(0.02), np.log(80.0), len(a)))
    dcfg = dict(npp_global=128, nmu_global=1, local_dist=1,
                local=[dict(enabled=1, npbins=npbins, nmu=1, rx=1, ry=1, rz=1, pmin=1e-2, pmax=1e2),
                       None, dict(enabled=1, npbins=3, nmu=2, rx=4, ry=2, rz=1, pmin=0.1, pmax=10.0), None])
    with ParkerPusher(**dict(c, precision="f64", nptl_max=len(a))) as pz:
        pz.upload_fields(nodes_for(c))
        pz.calc_fields_gradients()
        pz.set_particles(oracle.soa_from_particles(a))
        pz.init_particle_distributions(**dcfg)
        fg, locs = pz.calc_particle_distributions()
    fg_ref, locs_ref = oracle.distributions(oracle.params(c), dcfg, a)
    np.testing.assert_array_equal(fg, fg_ref)
    for k in (0, 2):
        np.testing.assert_array_equal(locs[k].ravel(), locs_ref[k])
    assert locs[0].size > 64 * 64 * npbins - 1
