"""The symmetric radiance path (k_modes, k_adding) at the edges of what it takes:
stream counts from 1 to its largest n, item counts around the four items of a
wavefront, conservative and reflective limits, and the items that it hands over
to the general path (k_rescue), alone and among ordinary ones.  FP64 within
1e-9 of the oracle (Q, U of |I|) with identical Fourier counts; the mixed path
within its 1e-5."""
import numpy as np
import pytest

import oracle
from aeroapps_amd import synthetic as S
from aeroapps_amd import vlidort as V
from oracle import chem_mie as CM
from _fixtures import RTOL_FP64, max_rel

pytestmark = pytest.mark.gpu
CH = (354.0, 550.0)


def inputs(ncol, km, nch, nmom, npol, seed):
    cols = S.make_columns(ncol, km, CH[:nch], seed=seed)
    tabs = S.make_mie_tables(CH[:nch], nmom=nmom, npol=npol)
    tau, ssa, g, pm, _ = CM.get_aop_vector(tabs, CH[:nch], tabs[0].lambda_m, S.TRACERS, cols.qm, cols.rh, nmom, npol)
    f = lambda a: np.asarray(a, dtype=np.float64)
    return cols, f(tau), f(ssa), f(g), f(pm)


def scalar(cols, tau, ssa, g, pm, N, albedo, precision=0):
    return V.scalar_lambert(cols.channels, N, False, cols.rot.T, cols.depol, tau.T, ssa.T, g.T, pm.T, cols.pe.T,
                            cols.he.T, cols.te.T, albedo.T, cols.sza, cols.raa, cols.vza, S.MISSING,
                            precision=precision, return_nfourier=True)


def check_scalar(cols, tau, ssa, g, pm, N, albedo, precision=0):
    I, R, rc, nf = scalar(cols, tau, ssa, g, pm, N, albedo, precision)
    I0, R0, nf0, rc0 = oracle.port().scalar_lambert(cols.km, cols.channels, N, pm.shape[1], cols.rot, cols.depol, tau,
                                                    ssa, g, pm, cols.pe, cols.he, cols.te, albedo, cols.sza,
                                                    cols.raa, cols.vza)
    assert rc == rc0
    if precision == 0:
        assert (nf == nf0.T).all()
    tol = RTOL_FP64 if precision == 0 else 1.0e-5
    ok = (nf == nf0.T)
    assert max_rel(I[ok], I0.T[ok]) < tol
    assert max_rel(R[ok], R0.T[ok]) < tol


@pytest.mark.parametrize("N,ncol,km,nch,precision", [
    (1, 1, 1, 1, 0), (1, 5, 72, 1, 0), (2, 3, 2, 2, 0), (2, 4, 9, 1, 1), (3, 17, 30, 1, 0), (5, 2, 72, 2, 1),
    (7, 9, 11, 1, 1), (7, 1, 72, 1, 0), (8, 5, 40, 1, 0), (8, 3, 40, 1, 1), (10, 3, 20, 1, 0), (12, 6, 72, 1, 0),
    (12, 2, 5, 1, 1), (13, 2, 6, 1, 0), (9, 7, 3, 1, 0), (14, 35, 1, 1, 0), (15, 3, 24, 1, 0)])
def test_scalar_edges(gpu, N, ncol, km, nch, precision):
    print(f"case scalar N={N} ncol={ncol} km={km} precision={precision}", flush=True)
    cols, *opt = inputs(ncol, km, nch, 32, 1, seed=71 + N)
    check_scalar(cols, *opt, N, cols.albedo, precision)


@pytest.mark.parametrize("N,ncol,km,precision", [(2, 1, 72, 0), (2, 6, 3, 1), (3, 5, 20, 0), (4, 7, 12, 0), (5, 2, 4, 0),
                                                 (3, 3, 20, 1)])
def test_vector_edges(gpu, N, ncol, km, precision):
    print(f"case vector N={N} ncol={ncol} km={km} precision={precision}", flush=True)
    cols, tau, ssa, g, pm = inputs(ncol, km, 1, 24, 6, seed=91 + N)
    alpha = np.zeros_like(cols.rot)
    I, R, Q, U, rc, nf = V.vector_lambert(cols.channels, N, False, cols.rot.T, cols.depol, alpha.T, tau.T, ssa.T,
                                          pm.T, cols.pe.T, cols.he.T, cols.te.T, cols.albedo.T, cols.sza, cols.raa,
                                          cols.vza, cols.flux_factor.T, S.MISSING, precision=precision,
                                          return_nfourier=True)
    I0, R0, Q0, U0, nf0, rc0 = oracle.port().vector_lambert(km, cols.channels, N, 24, cols.rot, cols.depol, alpha,
                                                            tau, ssa, pm, cols.pe, cols.he, cols.te, cols.albedo,
                                                            cols.sza, cols.raa, cols.vza, cols.flux_factor)
    tol = RTOL_FP64 if precision == 0 else 1.0e-5
    assert rc == rc0 and (nf == nf0.T).all()
    assert max_rel(I, I0.T) < tol
    for a, b in ((Q, Q0), (U, U0)):
        assert np.max(np.abs(a - b.T) / np.abs(I0.T)) < tol


@pytest.mark.parametrize("N", [2, 6, 8, 12])
def test_surface_and_scattering_limits(gpu, N):
    """Albedo 0 and 1, conservative layers (single-scattering albedo capped at
    0.99999 by the driver), almost empty and very thick layers, against the
    independent 64-bit solution of perf/cases.py: the oracle's eigensolver, like
    the reference's, loses (k_max / k)^2 eps on conservative layers (up to 1.1e-8
    here, where this path and the independent solution agree to 6e-11)."""
    import torch
    from perf import cases
    print(f"case limits N={N}", flush=True)
    cols, tau, ssa, g, pm = inputs(9, 24, 1, 32, 1, seed=17)
    albedo = cols.albedo.copy()
    albedo[0, :3] = (0.0, 1.0, 0.6)
    ssa[3], ssa[4] = 1.0, 1.0
    tau[4] *= 300.0
    tau[5] *= 1.0e-9
    tau[6, 0, 7:] *= 500.0
    I, R, rc, nf = scalar(cols, tau, ssa, g, pm, N, albedo)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a))
    geo = dict(rot=t(cols.rot), sza=t(cols.sza), vza=t(cols.vza), raa=t(cols.raa), he=t(cols.he), depol=t(cols.depol))
    I0, R0 = cases._exact_radiance(dict(nstreams=N, nch=1), geo, t(albedo), t(tau), t(ssa),
                                   t(np.moveaxis(pm[0], 0, -1)))
    assert rc == 0
    assert max_rel(I, I0.numpy()) < RTOL_FP64
    assert max_rel(R, R0.numpy()) < RTOL_FP64


@pytest.mark.parametrize("N", [4, 6, 12])
@pytest.mark.parametrize("precision", [0, 1])
def test_handed_over_items(gpu, N, precision):
    """Surfaces that reflect more than they receive (albedo above 1 or far below
    0) leave the symmetric path; the ordinary items beside them do not change."""
    print(f"case rescue N={N} precision={precision}", flush=True)
    cols, *opt = inputs(11, 16, 2, 32, 1, seed=23)
    albedo = cols.albedo.copy()
    plain = scalar(cols, *opt, N, albedo, precision)
    albedo[0, 2], albedo[1, 2], albedo[0, 9] = 1.7, -3.0, 1.2
    check_scalar(cols, *opt, N, albedo, precision)
    I, R, rc, nf = scalar(cols, *opt, N, albedo, precision)
    same = (albedo == cols.albedo).T
    assert np.array_equal(I[same], plain[0][same]) and np.array_equal(nf[same], plain[3][same])


def test_partial_isolation_is_missing(gpu):
    """Three Stokes components with scattering in I only (no Rayleigh, no delta-M
    truncation): the Q and U rows have no off-diagonal element while the I rows
    do, which the general eigensolver reports."""
    print("case partial isolation", flush=True)
    cols, tau, ssa, g, pm = inputs(3, 5, 1, 24, 6, seed=5)
    alpha, rot = np.zeros_like(cols.rot), np.zeros_like(cols.rot)
    pm[1:] = 0.0
    pm[:, 4:] = 0.0
    I, R, Q, U, rc, nf = V.vector_lambert(cols.channels, 2, False, rot.T, cols.depol, alpha.T, tau.T, ssa.T,
                                          pm.T, cols.pe.T, cols.he.T, cols.te.T, cols.albedo.T, cols.sza, cols.raa,
                                          cols.vza, cols.flux_factor.T, S.MISSING, return_nfourier=True)
    assert (I == S.MISSING).all() and (Q == S.MISSING).all() and (U == S.MISSING).all() and (nf == 0).all()


@pytest.mark.parametrize("ncol,km,nch,nmom", [(3, 7, 1, 9), (1, 1, 1, 1), (5, 6, 2, 32)])
@pytest.mark.parametrize("precision", [0, 1])
def test_float32_optics_give_the_same_bits(gpu, ncol, km, nch, nmom, precision):
    """Fortran-ordered float32 optics take their own entry point; the results
    are those of the widened arrays, bit for bit."""
    print(f"case float32 optics ncol={ncol} km={km} nmom={nmom}", flush=True)
    cols = S.make_columns(ncol, km, CH[:nch], seed=29)
    tabs = S.make_mie_tables(CH[:nch], nmom=nmom, npol=1)
    tau, ssa, g, pm, _ = CM.get_aop_vector(tabs, CH[:nch], tabs[0].lambda_m, S.TRACERS, cols.qm, cols.rh, nmom, 1)
    f = lambda a: np.asarray(a, dtype=np.float64)
    wide = scalar(cols, f(tau), f(ssa), f(g), f(pm), 3, cols.albedo, precision)
    half = scalar(cols, tau, ssa, g, pm, 3, cols.albedo, precision)
    assert tau.dtype == np.float32
    for a, b in zip(wide, half):
        assert np.array_equal(a, b)
