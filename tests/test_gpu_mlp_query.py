"""Ensemble spectra of few rows (one launch, pinned or device memory) against
the layer-by-layer kernels (SP_MLP_UNFUSED=1), bit for bit: row counts around
the 32-row blocks, the pinned staging's size and the largest count the kernel
takes, over the shapes and members of a block."""
import numpy as np
import pytest

from sp_hip.device import DeviceArray
from sp_hip.surrogate import Surrogate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nhidden,nlayers,nout,members", [
    (256, 4, 64, 2), (256, 1, 128, 1), (128, 2, 32, 4), (128, 5, 128, 3), (256, 3, 32, 3)])
def test_query_rows_equal_layer_kernels(monkeypatch, nhidden, nlayers, nout, members):
    rng = np.random.default_rng(nlayers)
    with Surrogate(members=members, nhidden=nhidden, nlayers=nlayers, nbins=nout, seed=5,
                   batch_max=9000) as s:
        for rows in (1, 8, 31, 33, 100, 940, 2048, 8192, 8193):
            x = rng.uniform(-1.0, 1.0, (rows, 6)).astype(np.float32)
            spec, est = s.predict(x)
            assert s.nets[0].last_forward_ms() > 0
            with DeviceArray.from_host(x) as xd, DeviceArray((rows, nout)) as sd, DeviceArray(rows) as rd:
                s.predict_device(xd, sd, rd)
                spec_d, spread_d = sd.to_host(), rd.to_host()
            monkeypatch.setenv("SP_MLP_UNFUSED", "1")
            spec_g, est_g = s.predict(x)
            monkeypatch.delenv("SP_MLP_UNFUSED")
            np.testing.assert_array_equal(spec, spec_g, err_msg=str(rows))
            np.testing.assert_array_equal(est, est_g, err_msg=str(rows))
            np.testing.assert_array_equal(spec_d, spec_g, err_msg=str(rows))
            np.testing.assert_array_equal(s.estimate(spread_d), est_g, err_msg=str(rows))
