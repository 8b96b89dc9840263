"""Bins and counts of variants arrive together: odd and even numbers of bins
and variants, and more variants than one piece of the staging holds."""
import numpy as np
import pytest

import oracle
from helpers import cfg2d, nodes_for, random_states
from sp_hip import ParkerPusher

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npp,nvar", [(1, 1), (5, 3), (64, 7), (7, 40000), (128, 64)])
def test_counts_follow_bins(npp, nvar):
    c = cfg2d(16)
    a = random_states(c, 5000, seed=npp)
    a["origin"] = np.random.default_rng(nvar).integers(0, nvar, len(a))
    a["weight"] = 0.5 ** np.random.default_rng(1).integers(0, 4, len(a))
    with ParkerPusher(**dict(c, precision="f64", nptl_max=len(a))) as pz:
        pz.upload_fields(nodes_for(c))
        pz.calc_fields_gradients()
        pz.set_particles(oracle.soa_from_particles(a))
        pz.init_particle_distributions(npp_global=npp)
        pz.set_variants([(1e-3, 0.1, 1.6)] * nvar)
        f, cnt = pz.variant_distributions()
        fg, _ = pz.calc_particle_distributions()
    np.testing.assert_array_equal(cnt, np.bincount(a["origin"], minlength=nvar))
    np.testing.assert_array_equal(f.sum(0), fg)
