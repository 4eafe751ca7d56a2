"""The column set-up kernels (k_geom, k_item) at the ends of their input
ranges, against the oracle."""
import numpy as np
import pytest

import oracle
from aeroapps_amd import synthetic as S
from aeroapps_amd import vlidort as V
from oracle import chem_mie as CM
from _fixtures import RTOL_FP64, max_rel

pytestmark = pytest.mark.gpu
CH = (354.0,)


def inputs(ncol, km, seed):
    cols = S.make_columns(ncol, km, CH, seed=seed)
    tabs = S.make_mie_tables(CH, nmom=32, npol=1)
    tau, ssa, g, pm, _ = CM.get_aop_vector(tabs, CH, tabs[0].lambda_m, S.TRACERS, cols.qm, cols.rh, 32, 1)
    return (cols,) + tuple(np.asarray(a, dtype=np.float64) for a in (tau, ssa, g, pm))


def both(cols, tau, ssa, g, pm, N, plane_parallel):
    I, R, rc, nf = V.scalar_lambert(cols.channels, N, plane_parallel, cols.rot.T, cols.depol, tau.T, ssa.T, g.T, pm.T,
                                    cols.pe.T, cols.he.T, cols.te.T, cols.albedo.T, cols.sza, cols.raa, cols.vza,
                                    S.MISSING, return_nfourier=True)
    I0, R0, nf0, rc0 = oracle.port().scalar_lambert(cols.km, cols.channels, N, 32, cols.rot, cols.depol, tau, ssa, g,
                                                    pm, cols.pe, cols.he, cols.te, cols.albedo, cols.sza, cols.raa,
                                                    cols.vza, plane_parallel=plane_parallel)
    assert rc == rc0 == 0
    return I, R, nf, I0.T, R0.T, nf0.T


@pytest.mark.parametrize("sza", [89.9999, 89.999999, 89.9999999, 89.99999999])
def test_sun_at_the_horizon(gpu, sza):
    """cos(sza) below 7.5e-9 rounds the sine to 1: the Chapman ray then starts
    at its own tangent point.  The oracle's arcsines are NaN there for the
    columns whose sine rounds above 1; elsewhere they are off by up to the
    square root of one rounding, 1.5e-8 rad or 1e-4 km of a lowest layer's path
    of at least 30 km, which an optical path of up to 88 turns into 3e-4."""
    print(f"case horizon sza={sza}", flush=True)
    cols, *opt = inputs(12, 72, seed=7)
    cols.sza[:] = sza
    I, R, nf, I0, R0, nf0 = both(cols, *opt, 3, False)
    assert np.isfinite(I).all() and np.isfinite(R).all()
    ok = np.isfinite(I0)
    assert ok.sum() >= 2
    assert np.max(np.abs(I[ok] / I0[ok] - 1.0)) < 3.0e-4
    assert np.max(np.abs(R[ok] / R0[ok] - 1.0)) < 3.0e-4
    assert (nf[ok] == nf0[ok]).all()


@pytest.mark.parametrize("thick", [0, 20, 62, 63, 64, 71])
def test_plane_parallel_depth_above_a_thick_layer(gpu, thick):
    """The beam at the top of a layer is that of the layers above it, however
    thick the layer itself is: a difference of inclusive sums would leave
    1e10 x 1.1e-16 = 1e-6 in the slant depth."""
    print(f"case plane-parallel thick layer {thick}", flush=True)
    cols, tau, ssa, g, pm = inputs(7, 72, seed=11)
    tau[:, :, thick] = 1.0e10
    I, R, nf, I0, R0, nf0 = both(cols, tau, ssa, g, pm, 4, True)
    assert max_rel(I, I0) < RTOL_FP64 and max_rel(R, R0) < RTOL_FP64
    assert (nf == nf0).all()
