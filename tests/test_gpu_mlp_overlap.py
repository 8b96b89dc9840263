"""Device queries whose rows lie in the memory that receives the spectra or the
spreads give the results of rows elsewhere."""
from types import SimpleNamespace

import numpy as np
import pytest

from sp_hip.device import DeviceArray
from sp_hip.surrogate import Surrogate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,at", [(64, 0), (3000, 0), (8192, 0), (3000, 100), (3000, 3000 * 58)])
def test_rows_inside_the_spectra(rows, at):
    rng = np.random.default_rng(rows)
    x = rng.uniform(-1.0, 1.0, (rows, 6)).astype(np.float32)
    with Surrogate(members=2, seed=3, batch_max=1024) as s, DeviceArray.from_host(x) as xd, \
            DeviceArray((rows, 64)) as sd, DeviceArray(rows) as rd:
        s.predict_device(xd, sd, rd)
        want = sd.to_host(), rd.to_host()
        for _ in range(3):
            host = np.zeros(rows * 64, np.float32)
            host[at:at + x.size] = x.ravel()
            with DeviceArray.from_host(host) as both:
                xv = SimpleNamespace(ptr=both.ptr + 4 * at, shape=x.shape, dtype=np.float32)
                sv = SimpleNamespace(ptr=both.ptr, shape=(rows, 64), dtype=np.float32)
                s.predict_device(xv, sv, rd)
                np.testing.assert_array_equal(both.to_host().reshape(rows, 64), want[0])
                np.testing.assert_array_equal(rd.to_host(), want[1])


def test_rows_inside_the_spreads():
    rows = 8000
    x = np.random.default_rng(1).uniform(-1.0, 1.0, (rows, 6)).astype(np.float32)
    with Surrogate(members=2, seed=3, batch_max=1024) as s, DeviceArray.from_host(x) as xd, \
            DeviceArray((rows, 64)) as sd, DeviceArray(rows) as rd:
        s.predict_device(xd, sd, rd)
        want = sd.to_host(), rd.to_host()
        s.predict_device(xd, sd, SimpleNamespace(ptr=xd.ptr, shape=(rows,), dtype=np.float32))
        np.testing.assert_array_equal(sd.to_host(), want[0])
        np.testing.assert_array_equal(xd.to_host().ravel()[:rows], want[1])
