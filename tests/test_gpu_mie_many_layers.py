"""Chem_Mie optics of a call with more layer chunks than a grid's second
dimension holds (65,536): a flat list of points given as one column."""
import numpy as np
import pytest

from aeroapps_amd import chem_mie as AM
from aeroapps_amd import synthetic as S
from oracle import chem_mie as CM

pytestmark = pytest.mark.gpu
CH = (550.0,)


@pytest.mark.parametrize("nmom", [4, 3])   # four moments per lane, and one
def test_more_layer_chunks_than_a_grid_dimension(gpu, nmom):
    km = 8 * 65536 + 13
    print(f"case {km} layers nmom={nmom}", flush=True)
    cols = S.make_columns(8, 72, CH, seed=43)
    qm = np.resize(np.moveaxis(cols.qm, 1, 0).reshape(len(S.TRACERS), -1), (len(S.TRACERS), km))[None]
    rh = np.resize(cols.rh.reshape(-1), km)[None]
    # (an own value in the last, partial chunk)
    qm = np.ascontiguousarray(qm, dtype=np.float32)
    qm[:, :, -7:] *= np.float32(1.5)
    tabs = S.make_mie_tables(CH, nmom=nmom, npol=1)
    mie = AM.MieTables.from_synthetic(tabs)
    out = AM.get_aop_vector(mie, np.asarray(CH), S.TRACERS, 0, qm.T, rh.T, nmom, 1)
    ref = CM.get_aop_vector(tabs, CH, tabs[0].lambda_m, S.TRACERS, qm, rh, nmom, 1)
    for a, b in zip(out[:4], ref[:4]):
        assert np.array_equal(a, b.T)
    assert out[4] == ref[4]


@pytest.mark.parametrize("nmom,pairs", [(4, 24576), (4, 24577), (3, 49152), (3, 49153)])
def test_chunks_apart_and_walked_are_the_same(gpu, nmom, pairs):
    """Around the batch size from which a wavefront walks the layer chunks of its
    column: the bits of a few columns by themselves."""
    print(f"case chunks nmom={nmom} pairs={pairs}", flush=True)
    km = 11
    one = S.make_columns(97, km, CH, seed=47)
    qm = np.resize(one.qm, (pairs,) + one.qm.shape[1:])
    rh = np.resize(one.rh, (pairs, km))
    mie = AM.MieTables.from_synthetic(S.make_mie_tables(CH, nmom=nmom, npol=1))
    many = AM.get_aop_vector(mie, np.asarray(CH), S.TRACERS, 0, qm.T, rh.T, nmom, 1)
    few = AM.get_aop_vector(mie, np.asarray(CH), S.TRACERS, 0, one.qm.T, one.rh.T, nmom, 1)
    for a, b in zip(many[:4], few[:4]):
        for lo in (0, 97 * (pairs // 97 - 1)):
            assert np.array_equal(a[:, :, lo:lo + 97], b)
        rest = pairs % 97
        assert rest == 0 or np.array_equal(a[:, :, pairs - rest:], b[:, :, :rest])
