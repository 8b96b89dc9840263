"""Contexts and networks of one process share their pinned staging: four host
threads, each with a context and a network of its own, give the results that
each gives alone."""
import threading

import numpy as np
import pytest

import oracle
from helpers import cfg2d, nodes_for, random_states
from sp_hip import ParkerPusher
from sp_hip.surrogate import Surrogate

pytestmark = pytest.mark.gpu


def calls(k, rounds):
    c = cfg2d(32)
    a = random_states(c, 6000 + 5000 * k, seed=k)
    st = np.stack([a[q] for q in ("x", "y", "z", "p", "t", "dt")], 1)
    rng = np.random.default_rng(k)
    r = rng.uniform(-1.7, 1.7, (len(a), 4))
    fixed = rng.integers(0, 2, len(a)).astype(np.int8)
    x = rng.uniform(-1.0, 1.0, (40 + 300 * k, 6)).astype(np.float32)
    out = []
    with ParkerPusher(**dict(c, precision="f64", nptl_max=len(a))) as pz, Surrogate(seed=k, batch_max=2048) as s:
        pz.upload_fields(nodes_for(c))
        pz.calc_fields_gradients()
        pz.set_particles(oracle.soa_from_particles(a))
        pz.init_particle_distributions(64, 1, 1, [dict(enabled=1, npbins=40 + k, nmu=1, rx=1, ry=1, rz=1,
                                                       pmin=1e-2, pmax=1e2)])
        for _ in range(rounds):
            fg, loc = pz.calc_particle_distributions()
            out.append(pz.step_once(st, r, fixed, 0.0, 0.05) + (fg, loc[0]) + s.predict(x) +
                       (np.array(list(pz.quick_check().values())),))
    return out


def test_threads_share_staging():
    alone = [calls(k, 1)[0] for k in range(4)]
    got = [None] * 4

    def work(k):
        got[k] = calls(k, 6)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for k in range(4):
        assert got[k] is not None
        for one in got[k]:
            for p, q in zip(one, alone[k]):
                np.testing.assert_array_equal(p, q, err_msg=str(k))
