"""The Chem_Mie optics kernel's lane layouts (four moments per lane where the
moments come in whole groups of four, one otherwise; one wavefront per layer
chunk or per column) at their edges: bit for bit the oracle's float32 sums."""
import numpy as np
import pytest

from aeroapps_amd import chem_mie as AM
from aeroapps_amd import synthetic as S
from oracle import chem_mie as CM

pytestmark = pytest.mark.gpu
CH = (354.0, 550.0)


@pytest.mark.parametrize("nmom", [1, 4, 30, 32, 36, 64, 68, 128, 132, 256, 260])
@pytest.mark.parametrize("km,ncol,npol", [(11, 3, 1), (8, 2, 6), (72, 1, 4)])
def test_moment_groups_bit_exact(gpu, nmom, km, ncol, npol):
    print(f"case mie groups nmom={nmom} km={km} npol={npol}", flush=True)
    cols = S.make_columns(ncol, km, CH, seed=41)
    tabs = S.make_mie_tables(CH, nmom=nmom, npol=npol)
    mie = AM.MieTables.from_synthetic(tabs)
    out = AM.get_aop_vector(mie, np.asarray(CH), S.TRACERS, 0, cols.qm.T, cols.rh.T, nmom, npol)
    ref = CM.get_aop_vector(tabs, CH, tabs[0].lambda_m, S.TRACERS, cols.qm, cols.rh, nmom, npol)
    for a, b in zip(out[:4], ref[:4]):
        assert np.array_equal(a, b.T)
    assert out[4] == ref[4]
