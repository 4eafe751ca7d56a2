"""scalar_lambert with float32 layer optics refuses what it refuses with double
ones, also in the arguments that the driver does not read."""
import os

import numpy as np
import pytest

from aeroapps_amd import vlidort as V
from aeroapps_amd._lib import LIB_PATH

pytestmark = pytest.mark.skipif(not os.path.exists(LIB_PATH), reason="library not built")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("name,bad", [("channels", "blue"), ("channels", [[354.0], [354.0, 388.0]]), ("g", "none"),
                                      ("pe", [[1.0], [2.0, 3.0]]), ("te", np.array(["x"]))])
def test_unread_arguments_are_checked(dtype, name, bad):
    o = lambda *s: np.asfortranarray(np.full(s, 0.1, dtype=dtype))
    d = lambda *s: np.full(s, 1.0)
    a = dict(channels=d(1), ROT=d(3, 2, 1), depol=d(1), tau=o(3, 1, 2), ssa=o(3, 1, 2), g=o(3, 1, 2),
             pmom=o(3, 1, 2, 4, 1), pe=d(4, 2), he=d(4, 2), te=d(4, 2), albedo=d(2, 1), solar_zenith=d(2),
             relat_azymuth=d(2), sensor_zenith=d(2))
    a[name] = bad
    with pytest.raises((TypeError, ValueError)):
        V.scalar_lambert(nstreams=2, plane_parallel=False, MISSING=1.0e15, **a)
