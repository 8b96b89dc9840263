"""Ensemble spectra of host rows whose results lie in several pinned slots of
256 KiB: row counts at a slot's edges, against the same rows in device memory."""
import numpy as np
import pytest

from sp_hip.device import DeviceArray
from sp_hip.surrogate import Surrogate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nhidden,nout,members", [(256, 64, 2), (128, 128, 3), (128, 32, 1)])
def test_rows_over_several_slots(nhidden, nout, members):
    per = (256 << 10) // (4 * (6 + nout + 1)) // 32 * 32   # rows of a slot
    rng = np.random.default_rng(nout)
    with Surrogate(members=members, nhidden=nhidden, nlayers=2, nbins=nout, seed=3, batch_max=8192) as s:
        for rows in (per - 1, per, per + 1, 2 * per, min(8192, 3 * per + 33), 8192):
            x = rng.uniform(-1.0, 1.0, (rows, 6)).astype(np.float32)
            spec, est = s.predict(x)
            with DeviceArray.from_host(x) as xd, DeviceArray((rows, nout)) as sd, DeviceArray(rows) as rd:
                s.predict_device(xd, sd, rd)
                np.testing.assert_array_equal(spec, sd.to_host(), err_msg=str(rows))
                np.testing.assert_array_equal(est, s.estimate(rd.to_host()), err_msg=str(rows))
