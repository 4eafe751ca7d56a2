// Layer modes of the discrete-ordinate radiance path, symmetric form.
//
//   k_pi:    one thread per (item, Fourier term): the PI functions at the user
//            angle and the solar cosine, which every layer of the item shares.
//   k_modes: one thread per (item, layer) of a Fourier term: the homogeneous
//            modes, their beam amplitudes and the layer's upwelling source
//            coefficients (the quantities of VLIDORT_QHOM_SOLUTION,
//            UHOM_SOLUTION, HMULT and GBEAM_SOLUTION,
//            REG/vlidort_solutions.f90:150-2932).
//
// The eigenproblem.  With streams scaled by g_i = sqrt(w_i mu_i), the two
// halves S = diag(1/mu) - sum_{l+} phi_l B_l phi_l^T and D (the other parity)
// of the reference's SAB and DAB are symmetric, because the PI matrices and the
// Greek matrices B_l are (Nakajima and Tanaka 1986 use the same property).
// Where both are positive definite, S = L L^T and D = G G^T (Cholesky), and the
// singular values of G^T L are the separation constants k themselves (not
// k^2), with left singular vectors v.  The modes' sum and difference vectors
//   E = X+ + X- = G v / sqrt(k),   F = X+ - X- = sqrt(k) G^-T v
// satisfy S E = F k, D F = E k and F^T E = 1, so no inverse of E or F is ever
// formed.  (S is the half that is nearly singular, at Fourier 0 of a
// conservative layer: the columns of G^T L are graded, so one-sided Jacobi
// keeps each v accurate relative to its own k, and both vectors come from G
// alone.  With the columns of L^T G instead, E lost (k_max / k)^2 eps: 1e-8 at
// N = 12 and omega 0.99999.)  The SVD is one-sided Jacobi: every rotation is a
// dot product and a 2-column update with compile-time indices in registers,
// the quadrature's order (ascending mu) leaves the columns graded, and 3-4
// sweeps converge for N <= 6 (45 rotations at N = 6, 90 at N = 8, 235 at
// N = 12), where ASYMTX's nonsymmetric double-shift QR walks data-dependent
// deflation states.
// Rotation angles are formed in float: an angle that is off by 1e-7 leaves
// 1e-7 of an off-diagonal element that the next sweep removes; the rotation
// itself (c, s) is orthonormal in double.
//
// An item with a layer whose S or D is not positive definite, whose Jacobi
// iteration does not converge, or whose eigenmatrix is partially isolated
// (some rows without off-diagonal elements) is marked in W.tflag and continues
// on the reference's general eigensolver and banded solve (k_rescue).
//
// Mixed precision: SAB/DAB come from the FP32 contraction and are symmetric
// only to FP32 rounding.  The symmetric parts go through the same steps; the
// antisymmetric parts enter by first-order perturbation of E and F, whose
// error is the square of 1e-7.
//
// Measured against k_layer + k_sabdab (per call): N = 6 FP64, 400,000 items
// 201 -> 58 ms (127 with the records stored straight from the lanes), mixed,
// 240,004 items 110 -> 63 ms (168); three Stokes components N = 4, 16,000 items
// 361 -> 17.2 ms (k_modes_pair; a lane per layer, its matrix partly in scratch,
// took 33 and 12 for the triangles from k_sabdab).  At N = 6 FP64 an item and
// term write 65.4 KB (its records are 59.9), 2.3 TB/s at 400,000 items, and read
// 27.6; a wavefront issues 6.8k VALU instructions, which keep the VALU busy half
// of the time.
#pragma once
#include <type_traits>
#include "rt_work.h"
#include "rt_device.h"

namespace aa {

namespace {

// compile-time loop: f(integral_constant<int, B>) .. f(integral_constant<int, E - 1>)
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>());
    static_for<B + 1, E>(f);
  }
}

// x of the other lane of the lane pair (2 i, 2 i + 1)
__device__ __forceinline__ double dpp_pair(double x) {
  const int lo = __double2loint(x), hi = __double2hiint(x);
  return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, 0xB1, 0xF, 0xF, false),
                          __builtin_amdgcn_update_dpp(lo, lo, 0xB1, 0xF, 0xF, false));
}
// x of the even lane of the lane pair
__device__ __forceinline__ double dpp_even(double x) {
  const int lo = __double2loint(x), hi = __double2hiint(x);
  return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, 0xA0, 0xF, 0xF, false),
                          __builtin_amdgcn_update_dpp(lo, lo, 0xA0, 0xF, 0xF, false));
}
// Orders the LDS accesses of a workgroup that is one wavefront (they complete
// in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// PI functions of every Fourier term: one thread per (item, M).
template <int N, int S>
__global__ __launch_bounds__(64) void k_pi(RTWork W, int nitems) {
  constexpr int LM = 2 * N;
  constexpr PiOff PO(N, S);
  const long t = (long)blockIdx.x * 64 + threadIdx.x;
  const int it = (int)(t / LM), M = (int)(t - (long)it * LM);
  if (it >= nitems || M > W.nmoments || W.status[it] != 0) return;
  const int obs = global_item(W, it) / W.nch;
  const double ustream = cos(DEG_TO_RAD * W.vza[obs]);
  double* out = W.pis + (size_t)it * PO.size();
#pragma unroll 1
  for (int w = 0; w < 2; ++w) {
    double x[LM][S][S];
    pimatrix_x<S, LM>(M, W.nmoments, w == 0 ? ustream : W.csza[it], x);
#pragma unroll
    for (int l = 0; l < LM; ++l) {
      out[PO.at(M, l, w, 0)] = x[l][0][0];
      if constexpr (S == 3) {
        out[PO.at(M, l, w, 1)] = x[l][1][1];
        out[PO.at(M, l, w, 2)] = x[l][1][2];
      }
    }
  }
}

// Element (a, b) of a PI matrix from its three functions (P, R, T): rows
// [P 0 0; 0 R T; 0 T R].
template <int S>
__device__ __forceinline__ double pi_el(const double (&f)[S == 1 ? 1 : 3], int a, int b) {
  if (S == 1) return f[0];
  if (a == 0 || b == 0) return a == b ? f[0] : 0.0;
  return a == b ? f[1] : f[2];
}

// Cholesky factor of the lower triangle a (in place).  Returns false where a
// pivot is not positive.
template <int n>
__device__ __forceinline__ bool cholesky(double (&a)[n * (n + 1) / 2]) {
  auto ix = [](int r, int c) constexpr { return r * (r + 1) / 2 + c; };
  bool ok = true;
#pragma unroll
  for (int c = 0; c < n; ++c) {
    double p = a[ix(c, c)];
#pragma unroll
    for (int q = 0; q < c; ++q) p = fma(-a[ix(c, q)], a[ix(c, q)], p);
    ok = ok && p > 0.0;
    const double rs = rsqrt_nr(p);
    a[ix(c, c)] = p * rs;
#pragma unroll
    for (int r = c + 1; r < n; ++r) {
      double v = a[ix(r, c)];
#pragma unroll
      for (int q = 0; q < c; ++q) v = fma(-a[ix(r, q)], a[ix(c, q)], v);
      a[ix(r, c)] = v * rs;
    }
  }
  return ok;
}

// Triangle of one parity class of the eigenproblem, diag(1/mu) minus the sum of
// PI_i B PI_j over the (degree l, Stokes row o') of the class: cls 0 the even
// degrees for I, Q and the odd ones for U, cls 1 the others.
template <int N, int S, int CLS>
__device__ __forceinline__ void build_triangle(const RTWork& W, int M, const double* __restrict__ ogp,
                                               double (&a)[N * S * (N * S + 1) / 2]) {
  constexpr int n = N * S;
  constexpr QOff QO(N, S);
  const double* __restrict__ Qt = W.quad;
  const double* __restrict__ ph = W.phi;
  auto ix = [](int r, int c) constexpr { return r * (r + 1) / 2 + c; };
#pragma unroll
  for (int r = 0; r < n; ++r)
#pragma unroll
    for (int c = 0; c <= r; ++c) a[ix(r, c)] = r == c ? Qt[QO.rmu(r / S)] : 0.0;
  // (rolled: unrolled over the degrees the kernels outgrow the instruction cache)
  if constexpr (S == 1) {
    const int l0 = M + ((M & 1) != CLS ? 1 : 0);
#pragma unroll 1
    for (int l = l0; l <= W.nmoments; l += 2) {
      const double o = ogp[l];
      double f[N];
#pragma unroll
      for (int i = 0; i < N; ++i) f[i] = ph[QO.xq(M, l, i, 0, 0)];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const double w = -o * f[i];
#pragma unroll
        for (int j = 0; j <= i; ++j) a[ix(i, j)] = fma(w, f[j], a[ix(i, j)]);
      }
    }
  } else {
#pragma unroll 1
    for (int l = M; l <= W.nmoments; ++l) {
      const double* g = ogp + l * S * S;
      double P[N], R[N], T[N];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        P[i] = ph[QO.xq(M, l, i, 0, 0)]; R[i] = ph[QO.xq(M, l, i, 1 % S, 1 % S)];
        T[i] = ph[QO.xq(M, l, i, 1 % S, 2 % S)];
      }
      if ((l & 1) == CLS) {   // the class holds I, Q of this degree
        const double g00 = g[0], g01 = g[1], g10 = g[S], g11 = g[S + 1];
#pragma unroll
        for (int i = 0; i < N; ++i) {
          // minus PI_i B, columns I and Q
          const double u[3][2] = {{-P[i] * g00, -P[i] * g01}, {-R[i] * g10, -R[i] * g11}, {-T[i] * g10, -T[i] * g11}};
#pragma unroll
          for (int j = 0; j <= i; ++j)
#pragma unroll
            for (int o1 = 0; o1 < S; ++o1)
#pragma unroll
              for (int o2 = 0; o2 < S; ++o2) {
                const int r = i * S + o1, c = j * S + o2;
                if (c > r) continue;
                a[ix(r, c)] = fma(u[o1][o2 == 0 ? 0 : 1], o2 == 0 ? P[j] : (o2 == 1 ? R[j] : T[j]), a[ix(r, c)]);
              }
        }
      } else {   // U
        const double g22 = g[2 * S + 2];
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const double u[3] = {0.0, -T[i] * g22, -R[i] * g22};
#pragma unroll
          for (int j = 0; j <= i; ++j)
#pragma unroll
            for (int o1 = 1; o1 < S; ++o1)
#pragma unroll
              for (int o2 = 1; o2 < S; ++o2) {
                const int r = i * S + o1, c = j * S + o2;
                if (c > r) continue;
                a[ix(r, c)] = fma(u[o1], o2 == 1 ? T[j] : R[j], a[ix(r, c)]);
              }
        }
      }
    }
  }
}

// Rows of a symmetric matrix (lower triangle) without off-diagonal elements, as
// a bit mask.
template <int n>
__device__ __forceinline__ unsigned isolated_rows(const double (&a)[n * (n + 1) / 2]) {
  auto ix = [](int r, int c) constexpr { return r * (r + 1) / 2 + c; };
  unsigned m = 0u;
#pragma unroll
  for (int i = 0; i < n; ++i) {
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < n; ++j)
      if (j != i) s += fabs(a[i > j ? ix(i, j) : ix(j, i)]);
    if (s == 0.0) m |= 1u << i;
  }
  return m;
}

// Jacobi rotation of two columns with squared norms ni, nj and product g:
// tangent (0 where the pair is orthogonal to rounding); `act` whether it rotates.
template <int n>
__device__ __forceinline__ double jacobi_tan(double g, double ni, double nj, bool& act) {
  // cosine of the columns' angle, about twice the rounding of an n-term dot
  // product
  constexpr double TOL2 = (6.0e-16 * n) * (6.0e-16 * n);
  act = g * g > TOL2 * (ni * nj);
  // t = sign(z) / (|z| + sqrt(1 + z^2)), z = (|cj|^2 - |ci|^2) / (2 g)
  const float gf = (float)(2.0 * g), df = (float)(nj - ni);
  const float z = df * __builtin_amdgcn_rcpf(gf);
  // (the square root saturates before z^2 overflows; it is |z| there)
  const float az = fabsf(z), zm = fminf(az, 1.0e18f);
  const float ta = __builtin_amdgcn_rcpf(az + fmaxf(az, __builtin_amdgcn_sqrtf(fmaf(zm, zm, 1.0f))));
  return act ? (double)copysignf(ta, z) : 0.0;
}

// One-sided Jacobi iteration on the n columns c[j]; each lane holds R of their
// rows (PAIR: the lane pair holds them together).  Pairs of one antidiagonal
// (i + j constant) are disjoint: up to three are rotated side by side, so that
// their dependent chains (product, angle, reciprocal roots: about 450 cycles)
// overlap; rows' order, where each waits for the one before, needs a tenth fewer
// (a whole call: N = 12, 1,200 items 4.2 -> 4.1 ms, N = 6, 400,000 items
// 132.8 -> 132.0).  Returns whether the lane's columns converged.
template <int n, int R, bool PAIR>
__device__ __forceinline__ bool jacobi_columns(double (&c)[n][R]) {
  double nrm[n];
  bool conv = false;
#pragma unroll 1
  for (int sweep = 0; sweep < 16; ++sweep) {
    bool rot = false;
#pragma unroll
    for (int j = 0; j < n; ++j) {
      double v = 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r) v = fma(c[j][r], c[j][r], v);
      nrm[j] = PAIR ? v + dpp_pair(v) : v;
    }
    static_for<1, 2 * n - 2>([&](auto sc) __attribute__((always_inline)) {
      constexpr int s = decltype(sc)::value, lo = s - n + 1 > 0 ? s - n + 1 : 0, hi = (s + 1) / 2;
      static_for<0, (hi - lo + 2) / 3>([&](auto qc) __attribute__((always_inline)) {
        constexpr int i0 = lo + 3 * decltype(qc)::value, P = hi - i0 < 3 ? hi - i0 : 3;
        double g[P], tt[P];
        bool any = false;
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const int i = i0 + p, j = s - i;
          double v = 0.0;
#pragma unroll
          for (int r = 0; r < R; ++r) v = fma(c[i][r], c[j][r], v);
          g[p] = PAIR ? v + dpp_pair(v) : v;   // (the same sum in both lanes)
        }
#pragma unroll
        for (int p = 0; p < P; ++p) {
          bool act;
          tt[p] = jacobi_tan<n>(g[p], nrm[i0 + p], nrm[s - i0 - p], act);
          any = any || act;
        }
        if (__ballot(any) == 0ull) return;   // no lane rotates: skip the update
        rot = rot || any;
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const int i = i0 + p, j = s - i;
          const double cs = rsqrt_nr(fma(tt[p], tt[p], 1.0)), sn = cs * tt[p];
          nrm[i] = fma(-tt[p], g[p], nrm[i]);
          nrm[j] = fma(tt[p], g[p], nrm[j]);
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const double x = c[i][r], y = c[j][r];
            c[i][r] = fma(-sn, y, cs * x);
            c[j][r] = fma(sn, x, cs * y);
          }
        }
      });
    });
    conv = !rot;
    if (__ballot(rot) == 0ull) break;
  }
  return conv;
}

// User-angle (v) and beam (q) vectors of one (item, layer), by parity of the
// degree: the sums over the degrees are taken before those over the streams
// (per layer 2N rows of n, then n products per mode, where the reference forms
// n Legendre sums per mode).
template <int N, int S>
__device__ __forceinline__ void source_vectors(const RTWork& W, int it, int M, const double* __restrict__ ogp,
                                               double (&va)[S][N * S], double (&vb)[S][N * S], double (&qa)[N * S],
                                               double (&qb)[N * S]) {
  constexpr int n = N * S;
  constexpr QOff QO(N, S);
  constexpr PiOff PO(N, S);
  const int NMOM = W.nmoments;
  const double* __restrict__ ph = W.phi;
#pragma unroll
  for (int r = 0; r < n; ++r) {
    qa[r] = 0.0; qb[r] = 0.0;
#pragma unroll
    for (int o = 0; o < S; ++o) { va[o][r] = 0.0; vb[o][r] = 0.0; }
  }
  {
    const double* __restrict__ pis = W.pis + (size_t)it * PO.size();
    // one degree into the vectors of its parity (x: user angle, y: beam) and,
    // with three Stokes components, of the other parity (z: the U row)
    auto degree = [&](int l, double (&x)[S][n], double (&y)[n], double (&z)[S][n]) __attribute__((always_inline)) {
      if constexpr (S == 1) {
        const double o = ogp[l];
        const double cu = 0.5 * o * pis[PO.at(M, l, 0, 0)], cq = o * pis[PO.at(M, l, 1, 0)];
#pragma unroll
        for (int i = 0; i < n; ++i) {
          const double f = ph[QO.xq(M, l, i, 0, 0)];
          x[0][i] = fma(cu, f, x[0][i]);
          y[i] = fma(cq, f, y[i]);
        }
      } else {
        const double* g = ogp + l * S * S;
        const double g00 = g[0], g01 = g[1], g10 = g[S], g11 = g[S + 1], g22 = g[2 * S + 2];
        const double p = 0.5 * pis[PO.at(M, l, 0, 0)], r = 0.5 * pis[PO.at(M, l, 0, 1)], t = 0.5 * pis[PO.at(M, l, 0, 2)];
        const double p0 = pis[PO.at(M, l, 1, 0)];
        // 1/2 DMAT(o1) PI_user(o1, o) B(o, o'): rows o1, columns I, Q and U
        const double cu[3][3] = {{p * g00, p * g01, 0.0}, {r * g10, r * g11, t * g22}, {-t * g10, -t * g11, -r * g22}};
        const double q0 = g00 * p0, q1 = g10 * p0;
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const double P = ph[QO.xq(M, l, i, 0, 0)], R = ph[QO.xq(M, l, i, 1 % S, 1 % S)],
                       T = ph[QO.xq(M, l, i, 1 % S, 2 % S)];
#pragma unroll
          for (int o1 = 0; o1 < S; ++o1) {
            x[o1][i * S] = fma(cu[o1][0], P, x[o1][i * S]);
            x[o1][i * S + 1] = fma(cu[o1][1], R, x[o1][i * S + 1]);
            x[o1][i * S + 2] = fma(cu[o1][1], T, x[o1][i * S + 2]);
            if (o1 > 0) {
              z[o1][i * S + 1] = fma(cu[o1][2], T, z[o1][i * S + 1]);
              z[o1][i * S + 2] = fma(cu[o1][2], R, z[o1][i * S + 2]);
            }
          }
          y[i * S] = fma(q0, P, y[i * S]);
          y[i * S + 1] = fma(q1, R, y[i * S + 1]);
          y[i * S + 2] = fma(q1, T, y[i * S + 2]);
        }
      }
    };
#pragma unroll 1
    for (int l = M + (M & 1); l <= NMOM; l += 2) degree(l, va, qa, vb);
#pragma unroll 1
    for (int l = M + 1 - (M & 1); l <= NMOM; l += 2) degree(l, vb, qb, va);
    const int g = global_item(W, it);
    const int obs = g / W.nch, ch = g - obs * W.nch;
    const double F1 = (W.flux ? W.flux[(size_t)obs * W.nch + ch] : 1.0) / PI4;
#pragma unroll
    for (int r = 0; r < n; ++r) { qa[r] *= F1; qb[r] *= F1; }
  }
}

// What a mode's multipliers depend on besides its separation constant.
struct LayerBeam {
  double dtau, tduser, avsec, itrans, tdmubar, itransu, emultup, sigp, usec, sg;
  bool lsc, beam;
};
template <int N>
__device__ __forceinline__ LayerBeam layer_beam(const RTWork& W, int it, int layer, int M) {
  const size_t il = (size_t)it * W.km + layer;
  const double* trr = W.tr + il * TR_NFIELDS;
  LayerBeam b;
  b.dtau = trr[TR_DTAU]; b.tduser = trr[TR_TDUSER]; b.avsec = trr[TR_AVSEC]; b.itrans = trr[TR_ITRANS];
  b.tdmubar = trr[TR_TDMUBAR]; b.itransu = trr[TR_ITRANSU]; b.emultup = trr[TR_EMULTUP]; b.sigp = trr[TR_SIGP];
  b.lsc = (M < 3) ? true : (((W.lsc[il] >> M) & 1u) != 0u);
  b.beam = (layer + 1 <= W.beam_cutoff[it]) && b.lsc;
  b.usec = W.usec[it];
  b.sg = (M & 1) ? -1.0 : 1.0;
  return b;
}

// One mode (separation constant kv; products of its vectors with the source
// vectors, ua = va . E', ub = vb . F', qe = qa . E', qf = qb . F'):
// transmittance and beam amplitudes x = {t, gup, gdn}, source coefficients cl,
// cm; adds the mode's beam source to spar.
template <int S>
__device__ __forceinline__ void mode_terms(const LayerBeam& B, double kv, const double (&ua)[S], const double (&ub)[S],
                                           double qe, double qf, double (&x)[3], double (&cl)[S], double (&cm)[S],
                                           double (&spar)[S]) {
  const double help = kv * B.dtau;
  const double zdel = (help > MAX_TAU_PATH) ? 0.0 : exp(-help);
  // HMULT (REG/vlidort_solutions.f90:1651-1790)
  const double rho_m = B.usec - kv;
  double h1 = B.usec * (zdel - B.tduser) * rcp_nr(rho_m);
  if (fabs(rho_m) < TAYLOR_SMALL) h1 = taylor1(rho_m, B.dtau, B.tduser, B.usec);
  const double h2 = B.usec * (1.0 - zdel * B.tduser) * rcp_nr(B.usec + kv);
  double gup = 0.0, gdn = 0.0, dn[S], up[S];
#pragma unroll
  for (int o = 0; o < S; ++o) {
    up[o] = ua[o] + ub[o];
    dn[o] = B.sg * (ua[o] - ub[o]);
    cl[o] = B.lsc ? dn[o] * h2 : 0.0;
    cm[o] = B.lsc ? up[o] * h1 : 0.0;
  }
  if (B.beam) {
    // Green's-function amplitudes (:2649-2932)
    const double gamp = B.avsec + kv, gamm = B.avsec - kv;
    const double rgp = rcp_nr(gamp), rgm = rcp_nr(gamm);
    const double aterm = qe + qf, bterm = B.sg * (qe - qf);
    double cf = B.itrans * (zdel - B.tdmubar) * rgm;
    double sd = (B.itrans * h2 - B.emultup) * rgm;
    if (fabs(gamm) < TAYLOR_SMALL) {
      cf = taylor1(gamm, B.dtau, B.tdmubar, B.itrans);
      sd = B.itransu * taylor2(gamm, B.sigp, B.dtau, 1.0, B.tdmubar * B.tduser, 1.0);
    }
    const double df = B.itrans * (1.0 - zdel * B.tdmubar) * rgp;
    const double su = fma(-B.itrans * B.tdmubar, h1, B.emultup) * rgp;
    gdn = cf * aterm;
    gup = df * bterm;
#pragma unroll
    for (int o = 0; o < S; ++o) spar[o] += dn[o] * sd * aterm + up[o] * su * bterm - cm[o] * gdn;
  }
  x[0] = zdel; x[1] = gup; x[2] = gdn;
}

// A wavefront's records go to memory through LDS: every lane puts the fields of
// its record in order, and each 64-byte piece is written whole, eight records
// per store.  Stored from the lanes directly (8 bytes of 64 records per store,
// 13 MB of records open at once against 4 MB of L2) the pieces were evicted
// partially written: 53 GB for 12 GB of records (N = 6, 40,022 items), which
// bounded the kernel.
struct RecordOut {
  double* base;       // the wavefront's first record
  int left, lane;     // records of the wavefront, this lane
  double (*lds)[9];   // [64][8 + 1]
  template <int f, int AS>
  __device__ __forceinline__ void put(double v) {
    lds[lane][f & 7] = v;
    if constexpr ((f & 7) == 7) flush<f & ~7, AS>();
  }
  // records 8 q + lane / 8, field f0 + lane % 8
  template <int f0, int AS>
  __device__ __forceinline__ void flush() {
    wave_lds_fence();
    const int j = lane >> 3, i = lane & 7;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const double v = lds[8 * q + j][i];
      if (8 * q + j < left) base[(size_t)(8 * q + j) * AS + f0 + i] = v;
    }
    wave_lds_fence();
  }
};

// One thread per (item, layer).  VGPR budget: the n x n matrix of the Jacobi
// iteration (2 n^2 registers) and the factor G; two wavefronts
// per SIMD up to n = 6, one above.
template <int N, int S, bool MIX>
__global__ __launch_bounds__(64, (N * S <= (MIX ? 4 : 6)) ? 2 : 1) void k_modes(RTWork W, int M0, int group) {
  constexpr int n = N * S, LM = 2 * N, NT = n * (n + 1) / 2;
  static_assert(n <= 8, "k_modes_pair above");
  constexpr AOff O(N, S);
  constexpr QOff QO(N, S);
  constexpr PiOff PO(N, S);
  constexpr int AS = O.size();
  __shared__ double lds[64][9];
  // dense (item, layer) slots of this term; lanes beyond the last repeat it
  const int t0 = blockIdx.x * 64, nslot = W.lcnt[group], km = W.km;
  if (t0 >= nslot) return;
  const int t = min(t0 + (int)threadIdx.x, nslot - 1);
  const int it = W.lown[t];
  const int layer = t - W.loff[it];
  const int tg = blockIdx.y, M = M0 + tg;   // this term of the group
  const size_t sb = (size_t)tg * W.cap * km;
  RecordOut out{W.abuf + (sb + t0) * AS, nslot - t0, (int)threadIdx.x, lds};
  const int NMOM = W.nmoments;
  const double* __restrict__ Qt = W.quad;
  const double* __restrict__ ph = W.phi;   // sqrt(w/mu) x the quadrature PI matrices, the table's layout
  const size_t il = (size_t)it * km + layer;
  const double* __restrict__ ogp = W.og + il * (size_t)(LM * S * S);
  auto ix = [](int r, int c) constexpr { return r * (r + 1) / 2 + c; };
  // Degrees l of even and odd parity are summed apart ("a" and "b"): the even
  // ones belong to S for even M and to D for odd M, so for odd M the two
  // matrices, and with them E and F, change names.
  const bool odd = (M & 1) != 0;

  double a[NT], b[NT];
  double xa[MIX ? NT : 1], xb[MIX ? NT : 1];   // antisymmetric parts (mixed)
  bool ok = true;
  if constexpr (!MIX) {
    build_triangle<N, S, 0>(W, M, ogp, a);
    build_triangle<N, S, 1>(W, M, ogp, b);
  } else {
    const float* rec = W.sab32 + (sb + il) * (size_t)(2 * n * n);
    const float* ra = rec + (odd ? n * n : 0);
    const float* rb = rec + (odd ? 0 : n * n);
#pragma unroll
    for (int i = 0; i < n; ++i)
#pragma unroll
      for (int j = 0; j <= i; ++j) {
        const double sc = Qt[QO.g(i / S)] * Qt[QO.rg(j / S)];
        double va = (double)ra[i * n + j] * sc, vb = (double)rb[i * n + j] * sc;
        const double st = Qt[QO.g(j / S)] * Qt[QO.rg(i / S)];
        const double ta = (double)ra[j * n + i] * st, tb = (double)rb[j * n + i] * st;
        xa[ix(i, j)] = 0.5 * (va - ta);
        xb[ix(i, j)] = 0.5 * (vb - tb);
        va = 0.5 * (va + ta);
        vb = 0.5 * (vb + tb);
        a[ix(i, j)] = i == j ? va + Qt[QO.rmu(i / S)] : va;
        b[ix(i, j)] = i == j ? vb + Qt[QO.rmu(i / S)] : vb;
      }
  }
  if constexpr (n > 2) {   // partial isolation (the reference's prepass, n > 2 only as there)
    const unsigned iso = isolated_rows<n>(a) & isolated_rows<n>(b);
    ok = iso == 0u || iso == (1u << n) - 1u;
  }
  ok = cholesky<n>(a) && ok;
  ok = cholesky<n>(b) && ok;

  // c[j][r] = (G^T L)(r, j): column j, held as the vector the rotations mix
  double c[n][n];
#pragma unroll
  for (int j = 0; j < n; ++j)
#pragma unroll
    for (int r = 0; r < n; ++r) {
      double v = 0.0;
#pragma unroll
      for (int q = 0; q < n; ++q)
        if (q >= r && q >= j) v = fma(b[ix(q, r)], a[ix(q, j)], v);
      c[j][r] = v;
    }
  ok = jacobi_columns<n, n, false>(c) && ok;
  if (!ok) W.tflag[(size_t)it * W.terms + tg] = 1;

  // c = k v: E' = G v / sqrt(k), then F' = sqrt(k) G^-T v in place of c
  double keig[n], rsk[n];   // k, 1 / sqrt(k)
#pragma unroll
  for (int k = 0; k < n; ++k) {
    double v = 0.0;
#pragma unroll
    for (int r = 0; r < n; ++r) v = fma(c[k][r], c[k][r], v);
    keig[k] = v * rsqrt_nr(v);
    rsk[k] = rsqrt_nr(keig[k]);
  }
  double rdg[n];   // 1 / G(r, r)
#pragma unroll
  for (int r = 0; r < n; ++r) rdg[r] = rcp_nr(b[ix(r, r)]);
  auto efcol = [&](int k, double (&e)[n]) __attribute__((always_inline)) {
    const double sf = rsk[k], se = sf * sf * sf;
#pragma unroll
    for (int r = 0; r < n; ++r) {
      double v = 0.0;
#pragma unroll
      for (int q = 0; q <= r; ++q) v = fma(b[ix(r, q)], c[k][q], v);
      e[r] = v * se;
    }
#pragma unroll
    for (int r = n - 1; r >= 0; --r) {
      double v = c[k][r] * sf;
#pragma unroll
      for (int q = r + 1; q < n; ++q) v = fma(-b[ix(q, r)], c[k][q], v);
      c[k][r] = v * rdg[r];
    }
  };
  double em[n][n];   // E'
#pragma unroll
  for (int k = 0; k < n; ++k) efcol(k, em[k]);
  if constexpr (MIX) {
    // S' = E^T S E = K + s, D' = F^T D F = K + d with antisymmetric s, d; to
    // first order E -> E (1 + C), F -> F (1 + B) with
    //   C_jk = (k_j s_jk + k_k d_jk) / (k_k^2 - k_j^2), B_jk = (k_j d_jk + k_k s_jk) / (k_k^2 - k_j^2)
    float ya[n][n], yb[n][n];   // (S_a E)(., k), (D_a F)(., k)
#pragma unroll
    for (int k = 0; k < n; ++k)
#pragma unroll
      for (int r = 0; r < n; ++r) {
        float va = 0.0f, vb = 0.0f;
#pragma unroll
        for (int q = 0; q < n; ++q) {
          if (q == r) continue;
          const float sa = q < r ? (float)xa[ix(r, q)] : -(float)xa[ix(q, r)];
          const float sb = q < r ? (float)xb[ix(r, q)] : -(float)xb[ix(q, r)];
          va = fmaf(sa, (float)em[k][q], va);
          vb = fmaf(sb, (float)c[k][q], vb);
        }
        ya[k][r] = va;
        yb[k][r] = vb;
      }
    float cc[n][n], cb[n][n];
#pragma unroll
    for (int j = 0; j < n; ++j)
#pragma unroll
      for (int k = j; k < n; ++k) {
        if (j == k) { cc[j][k] = 0.0f; cb[j][k] = 0.0f; continue; }
        float sj = 0.0f, dj = 0.0f;
#pragma unroll
        for (int r = 0; r < n; ++r) {
          sj = fmaf((float)em[j][r], ya[k][r], sj);
          dj = fmaf((float)c[j][r], yb[k][r], dj);
        }
        const double kj = keig[j], kk = keig[k];
        const double gap = (kk - kj) * (kk + kj);
        const float kjf = (float)kj, kkf = (float)kk;
        const float rg = gap != 0.0 ? __builtin_amdgcn_rcpf((float)gap) : 0.0f;
        // (s and d change sign under j <-> k, the gap too)
        float v1 = (kjf * sj + kkf * dj) * rg, v2 = (kjf * dj + kkf * sj) * rg;
        float v3 = (kkf * sj + kjf * dj) * rg, v4 = (kkf * dj + kjf * sj) * rg;
        // (a pair closer than its perturbation stays as the symmetric parts have it)
        if (!(fabsf(v1) + fabsf(v2) + fabsf(v3) + fabsf(v4) < 1.0e-2f)) { v1 = v2 = v3 = v4 = 0.0f; }
        cc[j][k] = v1; cb[j][k] = v2; cc[k][j] = v3; cb[k][j] = v4;
      }
    // the increments of all columns from the unperturbed ones, then the update
    float de[n][n], df[n][n];
#pragma unroll
    for (int k = 0; k < n; ++k)
#pragma unroll
      for (int r = 0; r < n; ++r) {
        float v = 0.0f, w = 0.0f;
#pragma unroll
        for (int j = 0; j < n; ++j) {
          if (j == k) continue;
          v = fmaf((float)em[j][r], cc[j][k], v);
          w = fmaf((float)c[j][r], cb[j][k], w);
        }
        de[k][r] = v; df[k][r] = w;
      }
#pragma unroll
    for (int k = 0; k < n; ++k)
#pragma unroll
      for (int r = 0; r < n; ++r) { em[k][r] += (double)de[k][r]; c[k][r] += (double)df[k][r]; }
  }
  {
    auto rows = [&](auto first, const double (&x)[n][n]) __attribute__((always_inline)) {
      constexpr int f0 = decltype(first)::value;
      static_for<0, n * n>([&](auto fc) __attribute__((always_inline)) {
        constexpr int f = decltype(fc)::value;
        out.put<f0 + f, AS>(x[f % n][f / n]);
      });
    };
    if (odd) {
      rows(std::integral_constant<int, 0>(), c);
      rows(std::integral_constant<int, n * n>(), em);
    } else {
      rows(std::integral_constant<int, 0>(), em);
      rows(std::integral_constant<int, n * n>(), c);
    }
  }

  // ---- sources and multipliers
  const LayerBeam B = layer_beam<N>(W, it, layer, M);
  double va[S][n], vb[S][n], qa[n], qb[n];
  source_vectors<N, S>(W, it, M, ogp, va, vb, qa, qb);
  double ox[n][3], ocl[n][S], ocm[n][S], spar[S];
#pragma unroll
  for (int o = 0; o < S; ++o) spar[o] = 0.0;
#pragma unroll
  for (int k = 0; k < n; ++k) {
    double ua[S], ub[S], qe = 0.0, qf = 0.0;
#pragma unroll
    for (int o = 0; o < S; ++o) {
      double s1 = 0.0, s2 = 0.0;
#pragma unroll
      for (int r = 0; r < n; ++r) { s1 = fma(va[o][r], em[k][r], s1); s2 = fma(vb[o][r], c[k][r], s2); }
      ua[o] = s1; ub[o] = s2;
    }
#pragma unroll
    for (int r = 0; r < n; ++r) { qe = fma(qa[r], em[k][r], qe); qf = fma(qb[r], c[k][r], qf); }
    mode_terms<S>(B, keig[k], ua, ub, qe, qf, ox[k], ocl[k], ocm[k], spar);
  }
  // the rest of the record in field order, padded to whole pieces
  static_for<O.t(0), AS>([&](auto fc) __attribute__((always_inline)) {
    constexpr int f = decltype(fc)::value, q = f - O.t(0), w = q / n, k = q % n;
    double v = 0.0;
    if constexpr (w < 3) v = ox[k][w];
    else if constexpr (w < 3 + S) v = ocl[k][w - 3];
    else if constexpr (w < 3 + 2 * S) v = ocm[k][w - 3 - S];
    else if constexpr (f - O.csrc(0) < S) v = spar[f - O.csrc(0)];
    out.put<f, AS>(v);
  });
}

// The same for 8 < n <= 15: two lanes per (item, layer), 32 of them per
// wavefront.  A lane alone would hold the n x n matrix of the Jacobi iteration
// in more than the 256 registers that arithmetic addresses (n = 12: 288), and
// every rotation then moved columns through the accumulation registers and
// scratch.  Here lane h of a pair sums the source vectors and the triangle of
// parity class h and factors it (S in lane 0, D in lane 1), holds half of the
// rows of the columns in the iteration (n = 12: 144 registers; a column product
// is two partial sums and one lane exchange, the rotation's angle is computed
// in both), and forms and writes E, F and the source terms of half of the
// modes.  G, the PI functions of the streams and the Greek coefficients of the
// wavefront's layers, in whose place the source vectors come later, are in LDS:
// n = 12 takes 38 KB, four wavefronts on a compute unit, one on each SIMD,
// because a lane uses its 512 registers (at two per SIMD 1.3 KB of a lane spill:
// three Stokes components N = 4 took 57 ms a call where one took 37).  What it
// spends at N = 4 with three components, 16,000 items, of 17.2 ms: about 9 in
// the iteration (issue-bound), 4 to store 19 GB, 3 to 4 in E, F and the
// multipliers, 2 in the triangles and factors.  Both lanes summing both classes
// from coefficients read degree by degree, and E and F read back for the
// source terms, took 28.5.
template <int N, int S>
__global__ __launch_bounds__(64, 1) void k_modes_pair(RTWork W, int M0, int group) {
  constexpr int n = N * S, NT = n * (n + 1) / 2, H = (n + 1) / 2, LM = 2 * N, P = S == 1 ? 1 : 3;
  constexpr AOff O(N, S);
  constexpr QOff QO(N, S);
  constexpr PiOff PO(N, S);
  constexpr int AS = O.size(), BS = O.block();
  __shared__ double gl[NT][32];            // G
  __shared__ double xl[2 * S * n][32];     // Greek coefficients [l][S][S], then the source vectors [class][o][n]
  __shared__ double tab[LM][N][P];         // PI functions at the streams
  const int lane = threadIdx.x, pr = lane >> 1, h = lane & 1;
  const int t0 = blockIdx.x * 32, nslot = W.lcnt[group], km = W.km;
  if (t0 >= nslot) return;
  const int tg = blockIdx.y, M = M0 + tg;   // this term of the group
  const bool live = t0 + pr < nslot;
  const int t = live ? t0 + pr : nslot - 1;
  const int it = W.lown[t];
  const int layer = t - W.loff[it];
  const int NMOM = W.nmoments;
  auto ix = [](int r, int c) constexpr { return r * (r + 1) / 2 + c; };
  const bool odd = (M & 1) != 0;
  double* lrec = W.abuf + ((size_t)tg * W.cap * km + t) * AS;
  auto swap = [](double x) { return dpp_pair(x); };

  // ---- the degrees' coefficients and tables, zero outside M .. NMOM, so that a
  // class may run over whole pairs of degrees
  {
    static_assert(LM * S * S == 2 * S * n && (LM * S * S) % 2 == 0, "coefficients and source vectors share xl");
    constexpr int NQ = LM * S * S / 2;
    const double2* __restrict__ og2 =
        reinterpret_cast<const double2*>(W.og + ((size_t)it * km + layer) * (size_t)(LM * S * S));
    double2 v[(NQ + 1) / 2];
#pragma unroll
    for (int j = 0; j < (NQ + 1) / 2; ++j) {
      const int q = 2 * j + h;
      v[j] = (q < NQ && 2 * q + 1 >= M * S * S) ? og2[q] : make_double2(0.0, 0.0);
    }
    for (int e = lane; e < LM * N * P; e += 64) {
      const int l = e / (N * P), i = (e / P) % N, p = e % P;
      // (P, R, T: elements (0,0), (1,1), (1,2) of the PI matrix)
      tab[l][i][p] = (l >= M && l <= NMOM) ? W.phi[QO.xq(M, l, i, p == 0 ? 0 : 1, p)] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < (NQ + 1) / 2; ++j) {
      const int q = 2 * j + h;
      if (q < NQ) {
        xl[2 * q][pr] = 2 * q / (S * S) <= NMOM ? v[j].x : 0.0;
        xl[2 * q + 1][pr] = (2 * q + 1) / (S * S) <= NMOM ? v[j].y : 0.0;
      }
    }
  }
  wave_lds_fence();

  // ---- the triangle of class h and its factor; G^T L row by row of L
  bool ok;
  double c[n][H];   // c[j][rl] = (G^T L)(h H + rl, j)
  {
    double a[NT];
#pragma unroll
    for (int r = 0; r < n; ++r)
#pragma unroll
      for (int q = 0; q <= r; ++q) a[ix(r, q)] = r == q ? W.quad[QO.rmu(r / S)] : 0.0;
#pragma unroll 1
    for (int d = M & ~1; d <= NMOM; d += 2) {
      const int l1 = d + h, l2 = d + 1 - h;
      if constexpr (S == 1) {
        const double o = xl[l1][pr];
        double f[N];
#pragma unroll
        for (int i = 0; i < N; ++i) f[i] = tab[l1][i][0];
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const double w = -o * f[i];
#pragma unroll
          for (int j = 0; j <= i; ++j) a[ix(i, j)] = fma(w, f[j], a[ix(i, j)]);
        }
      } else {
        const double g00 = xl[l1 * S * S][pr], g01 = xl[l1 * S * S + 1][pr], g10 = xl[l1 * S * S + S][pr],
                     g11 = xl[l1 * S * S + S + 1][pr], g22 = xl[l2 * S * S + 2 * S + 2][pr];
        double f[N][P], f2[N][2];
#pragma unroll
        for (int i = 0; i < N; ++i) {
#pragma unroll
          for (int p = 0; p < P; ++p) f[i][p] = tab[l1][i][p];
          f2[i][0] = tab[l2][i][2 % P]; f2[i][1] = tab[l2][i][1 % P];
        }
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
          for (int o1 = 0; o1 < S; ++o1) {
            // minus PI_i B: columns I, Q of degree l1, U of degree l2
            const double u0 = -f[i][o1 % P] * (o1 == 0 ? g00 : g10), u1 = -f[i][o1 % P] * (o1 == 0 ? g01 : g11);
            const double u2 = o1 > 0 ? -f2[i][(o1 + 1) % 2] * g22 : 0.0;
#pragma unroll
            for (int j = 0; j <= i; ++j)
#pragma unroll
              for (int o2 = 0; o2 < S; ++o2) {
                const int r = i * S + o1, q = j * S + o2;
                if (q > r) continue;
                a[ix(r, q)] = fma(o2 == 0 ? u0 : u1, f[j][o2 % P], a[ix(r, q)]);
                if (o1 > 0 && o2 > 0) a[ix(r, q)] = fma(u2, f2[j][(o2 + 1) % 2], a[ix(r, q)]);
              }
          }
      }
    }
    unsigned iso = isolated_rows<n>(a);
    iso &= (unsigned)__builtin_amdgcn_update_dpp((int)iso, (int)iso, 0xB1, 0xF, 0xF, false);
    ok = cholesky<n>(a) && (iso == 0u || iso == (1u << n) - 1u);
    if (h == 1) {
#pragma unroll
      for (int q = 0; q < NT; ++q) gl[q][pr] = a[q];
    }
    wave_lds_fence();
#pragma unroll
    for (int j = 0; j < n; ++j)
#pragma unroll
      for (int r = 0; r < H; ++r) c[j][r] = 0.0;
#pragma unroll
    for (int q = 0; q < n; ++q) {
      double lq[n];   // row q of L, from lane 0
#pragma unroll
      for (int j = 0; j <= q; ++j) lq[j] = dpp_even(a[ix(q, j)]);
#pragma unroll
      for (int r = 0; r < H; ++r) {
        if (r > q) continue;
        const int row = h * H + r;
        const double g = row <= q ? gl[ix(q, 0) + (row <= q ? row : 0)][pr] : 0.0;
#pragma unroll
        for (int j = 0; j <= q; ++j) c[j][r] = fma(g, lq[j], c[j][r]);
      }
    }
  }

  ok = jacobi_columns<n, H, true>(c) && ok;
  if (!ok) W.tflag[(size_t)it * W.terms + tg] = 1;

  // ---- source vectors of class h: user angle (sv) and beam (sq)
  double sv[S][n], sq[n];
#pragma unroll
  for (int r = 0; r < n; ++r) {
    sq[r] = 0.0;
#pragma unroll
    for (int o = 0; o < S; ++o) sv[o][r] = 0.0;
  }
  {
    const double* __restrict__ pis = W.pis + (size_t)it * PO.size() + PO.at(M, 0, 0, 0);
#pragma unroll 2
    for (int d = M & ~1; d <= NMOM; d += 2) {
      const int l1 = d + h, l2 = d + 1 - h;   // the degrees of I, Q and of U
      const double* p1 = pis + l1 * 2 * P;
      if constexpr (S == 1) {
        const double o = xl[l1][pr], cu = 0.5 * o * p1[0], cq = o * p1[1];
#pragma unroll
        for (int i = 0; i < n; ++i) {
          const double f = tab[l1][i][0];
          sv[0][i] = fma(cu, f, sv[0][i]);
          sq[i] = fma(cq, f, sq[i]);
        }
      } else {
        const double* p2 = pis + l2 * 2 * P;
        const double g00 = xl[l1 * S * S][pr], g01 = xl[l1 * S * S + 1][pr], g10 = xl[l1 * S * S + S][pr],
                     g11 = xl[l1 * S * S + S + 1][pr], g22 = xl[l2 * S * S + 2 * S + 2][pr];
        const double p = 0.5 * p1[0], r = 0.5 * p1[1 % P], t_ = 0.5 * p1[2 % P], p0 = p1[P];
        const double r2 = 0.5 * p2[1 % P] * g22, t2 = 0.5 * p2[2 % P] * g22;
        // 1/2 DMAT(o1) PI_user(o1, o) B(o, o'): rows o1, columns I and Q
        const double cu[3][2] = {{p * g00, p * g01}, {r * g10, r * g11}, {-t_ * g10, -t_ * g11}};
        const double q0 = g00 * p0, q1 = g10 * p0;
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const double Pf = tab[l1][i][0], R = tab[l1][i][1 % P], T = tab[l1][i][2 % P];
          const double R2 = tab[l2][i][1 % P], T2 = tab[l2][i][2 % P];
#pragma unroll
          for (int o = 0; o < S; ++o) {
            sv[o][i * S] = fma(cu[o][0], Pf, sv[o][i * S]);
            sv[o][i * S + 1] = fma(cu[o][1], R, sv[o][i * S + 1]);
            sv[o][i * S + 2] = fma(cu[o][1], T, sv[o][i * S + 2]);
          }
          sv[1 % S][i * S + 1] = fma(t2, T2, sv[1 % S][i * S + 1]);
          sv[1 % S][i * S + 2] = fma(t2, R2, sv[1 % S][i * S + 2]);
          sv[2 % S][i * S + 1] = fma(-r2, T2, sv[2 % S][i * S + 1]);
          sv[2 % S][i * S + 2] = fma(-r2, R2, sv[2 % S][i * S + 2]);
          sq[i * S] = fma(q0, Pf, sq[i * S]);
          sq[i * S + 1] = fma(q1, R, sq[i * S + 1]);
          sq[i * S + 2] = fma(q1, T, sq[i * S + 2]);
        }
      }
    }
    const int g = global_item(W, it);
    const int obs = g / W.nch, ch = g - obs * W.nch;
    const double F1 = (W.flux ? W.flux[(size_t)obs * W.nch + ch] : 1.0) / PI4;
#pragma unroll
    for (int r = 0; r < n; ++r) sq[r] *= F1;
  }
  // (every lane has read the coefficients: the source vectors take their place)
  wave_lds_fence();
#pragma unroll
  for (int o = 0; o < S; ++o)
#pragma unroll
    for (int r = 0; r < n; ++r) xl[(h * S + o) * n + r][pr] = sv[o][r];

  // ---- lane h takes modes h H .. h H + H - 1 whole: rows 0 .. H - 1 are lane
  // 0's, the others lane 1's
  double v[H][2 * H], kq[H];
#pragma unroll
  for (int k = 0; k < H; ++k) {
    double s0 = 0.0, s1 = 0.0;
#pragma unroll
    for (int r = 0; r < H; ++r) {
      const double x = c[k][r], y = H + k < n ? c[H + k < n ? H + k : 0][r] : 0.0;
      s0 = fma(x, x, s0);
      s1 = fma(y, y, s1);
      const double keep = h ? y : x, got = swap(h ? x : y);
      v[k][r] = h ? got : keep;
      v[k][H + r] = h ? keep : got;
    }
    s0 += swap(s0);
    s1 += swap(s1);
    const double s = (h && H + k < n) ? s1 : s0;   // (odd n: lane 1's last mode is a pad)
    kq[k] = s * rsqrt_nr(s);
  }
  wave_lds_fence();
  const LayerBeam B = layer_beam<N>(W, it, layer, M);
  // ---- E' = G v / sqrt(k), F' = sqrt(k) G^-T v and what follows from them, mode
  // by mode (two or three at a time share the loads of G, but their vectors
  // spill: 20.3 and 23.8 ms where one at a time takes 17.2)
  double spar[S];
#pragma unroll
  for (int o = 0; o < S; ++o) spar[o] = 0.0;
  double* mrec = lrec + h * (H * BS);
  static_for<0, H>([&](auto kc) __attribute__((always_inline)) {
    constexpr int k = decltype(kc)::value;
    double e[n];
    double(&f)[2 * H] = v[k];
    // (the fences end the reuse of loaded values: kept from one mode to the
    // next, G alone takes as many registers as the vectors)
    wave_lds_fence();
    const double sf = rsqrt_nr(kq[k]), se = sf * sf * sf;
#pragma unroll
    for (int r = 0; r < n; ++r) {
      double w = 0.0;
#pragma unroll
      for (int q = 0; q <= r; ++q) w = fma(gl[ix(r, q)][pr], f[q], w);
      e[r] = w * se;
    }
    wave_lds_fence();
#pragma unroll
    for (int r = n - 1; r >= 0; --r) {
      const double rd = rcp_nr(gl[ix(r, r)][pr]);
      double w = f[r] * sf;
#pragma unroll
      for (int q = r + 1; q < n; ++q) w = fma(-gl[ix(q, r)][pr], f[q], w);
      f[r] = w * rd;
    }
    wave_lds_fence();
    double ua[S], ub[S], qe = 0.0, qf = 0.0;
#pragma unroll
    for (int o = 0; o < S; ++o) { ua[o] = 0.0; ub[o] = 0.0; }
#pragma unroll
    for (int r = 0; r < n; ++r) {
      const double own = sq[r], other = swap(own);
      qe = fma(h ? other : own, e[r], qe);
      qf = fma(h ? own : other, f[r], qf);
#pragma unroll
      for (int o = 0; o < S; ++o) {
        ua[o] = fma(xl[o * n + r][pr], e[r], ua[o]);
        ub[o] = fma(xl[(S + o) * n + r][pr], f[r], ub[o]);
      }
    }
    if (n % 2 == 1 && h * H + k >= n) return;   // (the pad of odd n)
    double x[3], cl[S], cm[S];
    mode_terms<S>(B, kq[k], ua, ub, qe, qf, x, cl, cm, spar);
    if (live) {
      double* m = mrec + k * BS;
#pragma unroll
      for (int r = 0; r < n; ++r) m[r] = odd ? f[r] : e[r];
#pragma unroll
      for (int r = 0; r < n; ++r) m[n + r] = odd ? e[r] : f[r];
#pragma unroll
      for (int q = 0; q < 3; ++q) m[2 * n + q] = x[q];
#pragma unroll
      for (int o = 0; o < S; ++o) { m[2 * n + 3 + o] = cl[o]; m[2 * n + 3 + S + o] = cm[o]; }
    }
  });
#pragma unroll
  for (int o = 0; o < S; ++o) {
    const double s = spar[o] + swap(spar[o]);
    if (live && h == 0) lrec[O.csrc(o)] = s;
  }
}

}  // namespace
}  // namespace aa
