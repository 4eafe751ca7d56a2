// Boundary-value problem and TOA radiance of one Fourier term by adding the
// layers from the surface up (k_adding).
//
// In a layer the downwelling field d and the upwelling field u (Stokes
// components 3, 4 of u negated, as the modes store them) are
//   d + u = E (p + beam),  d - u = F (q + beam),
// with p = T L + M, q = T L - M at the layer's bottom (L, M the amplitudes of
// the down- and up-decaying modes at the top and the bottom, T their
// transmittances; the integration constants of REG/vlidort_bvproblem.f90:
// 147-2311).  Everything below a level is the affine relation Q = Z P - z
// between the beam-inclusive P and Q of the layer above it.  One layer:
//   H = (1 + Z)^-1,  M = (2H - 1) T L + m                      (solve 1)
//   rho = T (2H - 1) T,  s = T m + gup                         (reflection at its top)
//   [J j] = (1 + rho)^-1 [A s],  A = F_below^T E_above         (solve 2)
//   Z' = A^T (2J - A),  z' = 2 A^T j                           (next layer's relation)
// with A = E_below^-1 E_above because F^T E = 1 (k_modes).  Z is a symmetric
// positive definite impedance for a reciprocal surface, and |rho| < 1, so
// neither solve needs pivoting; n x n systems replace the 3n x 4n panels of the
// banded factorisation, and there is no pivot search.  The TOA radiance at the
// user angle, I = g . L + h of everything below, is carried along the same
// way, so nothing is stored and there is no downward sweep.  A pivot that is
// not clearly positive (a surface record that reflects more than it receives)
// or an item marked by k_modes goes to k_rescue.
//
// Mapping: 16 lanes per item, lane c holds column c of every matrix and lane n
// the vectors; a row's or column's element reaches the other lanes by the
// row_newbcast lane move, so a product of two matrices costs n^2 move + FMA
// pairs per lane and no LDS.
//
// Bound: the dependent chain of the 2n pivots (broadcast, reciprocal, row
// update) per layer for small batches, the records' bytes (832 per layer at
// N = 6) for large ones.  Measured against the pivoted band solve (k_bvp, 8 or
// 32 lanes per item): N = 6, 400,000 items 204 -> 57 ms; one item 358 -> 51 us
// per term; N = 12, 1,200 items 15.5 -> 2.6 ms; three Stokes components N = 4,
// 16,000 items 133 -> 10 ms.
#pragma once
#include <type_traits>
#include "rt_work.h"
#include "rt_device.h"
#include "rt_modes.h"

namespace aa {

namespace {

// x of lane K of the caller's 16-lane row, in all its lanes
template <int K>
__device__ __forceinline__ double bc16(double x) {
  return __builtin_amdgcn_update_dpp(x, x, 0x150 + K, 0xF, 0xF, true);
}
// Solves K X = X in place (lane c: column c of K and of the right-hand sides),
// Gaussian elimination without row exchanges.  `low` collects the smallest
// pivot.
template <int n>
__device__ __forceinline__ void solve16(double (&K)[n], double (&X)[n], double& low) {
  static_for<0, n>([&](auto kc) __attribute__((always_inline)) {
    constexpr int k = decltype(kc)::value;
    const double p = bc16<k>(K[k]);
    low = fmin(low, p);
    if (p != p) low = -1.0;
    const double rp = rcp_nr(p);
    K[k] *= rp;
    X[k] *= rp;
#pragma unroll
    for (int i = k + 1; i < n; ++i) {
      const double f = bc16<k>(K[i]);
      X[i] = fma(-f, X[k], X[i]);
      K[i] = fma(-f, K[k], K[i]);
    }
  });
  static_for<0, n - 1>([&](auto kc) __attribute__((always_inline)) {
    constexpr int k = n - 1 - decltype(kc)::value;
#pragma unroll
    for (int i = 0; i < k; ++i) X[i] = fma(-bc16<k>(K[i]), X[k], X[i]);
  });
}

// Z = A^T Q over lanes: Z_i = sum_m A(m, i) Q_m (lane c: columns of A and Q)
template <int n>
__device__ __forceinline__ void mul_at(const double (&A)[n], const double (&Q)[n], double (&Z)[n]) {
  static_for<0, n>([&](auto ic) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value;
    double v = 0.0;
#pragma unroll
    for (int m = 0; m < n; ++m) v = fma(bc16<i>(A[m]), Q[m], v);
    Z[i] = v;
  });
}
// X += sign * A Q (A given by its columns: A(i, m) is register i of lane m)
template <int n>
__device__ __forceinline__ void sub_mul(const double (&A)[n], const double (&Q)[n], double (&X)[n]) {
  static_for<0, n>([&](auto mc) __attribute__((always_inline)) {
    constexpr int m = decltype(mc)::value;
#pragma unroll
    for (int i = 0; i < n; ++i) X[i] = fma(-bc16<m>(A[i]), Q[m], X[i]);
  });
}

template <int N, int S, bool MIX>
__global__ __launch_bounds__(64) void k_adding(RTWork W, int M, const int* __restrict__ active,
                                               const int* __restrict__ nactive, int* __restrict__ next,
                                               int* __restrict__ nnext) {
  constexpr int n = N * S, IPW = 4;
  static_assert(n <= 15, "a lane per column and one for the vectors");
  constexpr AOff O(N, S);
  constexpr QOff QO(N, S);
  constexpr BROff RO(N);
  constexpr BPOff PO(N);
  const int lane = threadIdx.x, g = lane >> 4, t = lane & 15;
  // this wavefront's items: the term's items are in LBINS lists by layer count
  int first = -1, cntb = 0;
  const int* lst = active;
  {
    int acc = 0;
#pragma unroll
    for (int b = 0; b < LBINS; ++b) {
      const int c = nactive[b], nbk = (c + IPW - 1) / IPW;
      if (first < 0 && (int)blockIdx.x < acc + nbk) {
        first = ((int)blockIdx.x - acc) * IPW;
        cntb = c;
        lst = active + (size_t)b * W.cap;
      }
      acc += nbk;
    }
  }
  if (first < 0) return;   // uniform over the wavefront
  const int ai = first + g;
  const bool valid = ai < cntb;
  const int it = valid ? lst[ai] : lst[first];
  const int km = W.km;
  const int gi = global_item(W, it), obs = gi / W.nch, ch = gi - obs * W.nch;
  const size_t oi = (size_t)ch * W.nobs + obs;
  const int L = W.L_it[it];
  int Lmax = L;
#pragma unroll
  for (int q = 0; q < IPW; ++q) Lmax = max(Lmax, __builtin_amdgcn_readlane(L, q * 16));
  const int AS = W.astride;
  const double* __restrict__ ab = W.abuf + (size_t)W.loff[it] * AS;   // the item's slots of this term
  const double* __restrict__ trr = W.tr + (size_t)it * km * TR_NFIELDS;
  const double* __restrict__ Qt = W.quad;
  const double ff = W.flux ? W.flux[(size_t)obs * W.nch + ch] : 1.0;
  const bool col = t < n, vec = t == n;
  const double dvec = vec ? 1.0 : 0.0;
  double low = 1.0;

  double E[n], F[n], Z[n], rr[S], hh[S];   // hh in every lane
  // ---- the surface: Z, z and the BOA radiance at the user angle, in the
  // bottom layer's modes
  auto load_modes = [&](int k, double (&e)[n], double (&f)[n]) __attribute__((always_inline)) {
    const double* r = ab + (size_t)k * AS;
    const int c = col ? t : 0;
#pragma unroll
    for (int m = 0; m < n; ++m) {
      const double x = r[O.e(m, 0) + c * O.estep()], y = r[O.f(m, 0) + c * O.estep()];
      e[m] = col ? x : 0.0;
      f[m] = col ? y : 0.0;
    }
  };
  load_modes(L - 1, E, F);
  {
    const bool brdf = W.brdf != nullptr;
    const bool pol = S == 3 && W.bpdf != nullptr;
    const double albedo = brdf ? 0.0 : W.albedo[oi];
    const double tsb = W.tsb[it];
    const bool surf = brdf || ((M == 0) && (albedo != 0.0));
    // reflected direct beam (DIRECTRADIANCE, REG/vlidort_miscsetups.f90:1296-1614)
    double attn = 0.0;
    if (surf && tsb != 0.0) {
      double x0 = 4.0 * W.csza[it] / ((M == 0) ? 1.0 : 2.0);
      x0 = ff * x0 / PI4;
      attn = x0 * tsb;
    }
#pragma unroll
    for (int o = 0; o < S; ++o) { rr[o] = 0.0; hh[o] = 0.0; }
    double Y[n];
    if (!brdf) {
      // Lambertian: R = 2 albedo g g^T on Stokes component 0 (Fourier 0), so
      // (1 + R)^-1 in closed form
      const double al = surf ? albedo : 0.0;
      double g2 = 0.0, y = 0.0;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const double gg = Qt[QO.g(i)];
        g2 = fma(gg, gg, g2);
        y = fma(gg, E[i * S], y);
      }
      const double den = 1.0 / (1.0 + 2.0 * al * g2);
      const double s0 = attn * al;
      // (1 + R)^-1 [E | ss]: E - 2 al den g (g^T E), ss = s0 g
      const double cy = vec ? -s0 * den : 2.0 * al * den * y;
#pragma unroll
      for (int r = 0; r < n; ++r) Y[r] = (r % S == 0) ? fma(-cy, Qt[QO.g(r / S)], E[r]) : E[r];
      rr[0] = col ? 2.0 * al * den * y : 0.0;
      hh[0] = -2.0 * al * s0 * g2 * den;
    } else {
      const double* __restrict__ rec = W.brdf + (size_t)it * W.brdf_stride;
      const double sf = (M == 0) ? 2.0 : 1.0;
      double K[n];
#pragma unroll
      for (int r = 0; r < n; ++r) {
        const int i = r / S, o1 = r - (r / S) * S;
        const double gi_ = Qt[QO.g(i)];
        double kv = (r == t) ? 1.0 : 0.0, sv = 0.0;
        if (pol || o1 == 0) {
          const int j = (col ? t : 0) / S, o2 = (col ? t : 0) - ((col ? t : 0) / S) * S;
          const double sgn = (o1 == 2) ? -1.0 : 1.0;
          if (pol) {
            kv = fma(sgn * sf * gi_ * Qt[QO.g(j)], rec[PO.f(M, i, j, o1 * 3 + o2)], kv);
            sv = sgn * attn * rec[PO.f0(M, i, o1)] * gi_;
          } else {
            if (o2 == 0) kv = fma(sf * gi_ * Qt[QO.g(j)], rec[RO.f(M, i, j)], kv);
            sv = attn * rec[RO.f0(M, i)] * gi_;
          }
        }
        K[r] = col ? kv : 0.0;
        Y[r] = vec ? sv : E[r];
      }
      solve16<n>(K, Y, low);
#pragma unroll
      for (int o = 0; o < S; ++o) {
        if (o > 0 && !pol) continue;
        double v = 0.0;
#pragma unroll
        for (int r = 0; r < n; ++r) {
          const int j = r / S, o2 = r - (r / S) * S;
          if (pol) v = fma(sf * Qt[QO.g(j)] * rec[PO.uf(M, j, o * 3 + o2)], Y[r], v);
          else if (o2 == 0) v = fma(sf * Qt[QO.g(j)] * rec[RO.uf(M, j)], Y[r], v);
        }
        rr[o] = col ? v : 0.0;
        hh[o] = -bc16<n>(v);
      }
    }
#pragma unroll
    for (int r = 0; r < n; ++r) Y[r] = fma(2.0, Y[r], -E[r]);   // (1 + R)^-1 (1 - R) E and 2 (1 + R)^-1 ss
    mul_at<n>(E, Y, Z);
    if constexpr (MIX) {
      double X[n], D[n];
      mul_at<n>(E, F, D);
#pragma unroll
      for (int r = 0; r < n; ++r) { D[r] -= (r == t) ? 1.0 : 0.0; X[r] = Z[r]; }
      sub_mul<n>(D, Z, X);
#pragma unroll
      for (int r = 0; r < n; ++r) Z[r] = X[r];
    }
  }

  for (int k = Lmax - 1; k >= 0; --k) {
    const bool here = k < L;
    if (!here) continue;   // uniform within the item's lanes
    const double* __restrict__ lr = ab + (size_t)k * AS;
    const int cl = col ? t : 0;
    const double tk = col ? lr[O.t(0) + cl] : 1.0;
    const double gup = lr[O.gup(0) + cl], gdn = lr[O.gdn(0) + cl];
    const double tdu = trr[(size_t)k * TR_NFIELDS + TR_TDUSER];
    // the layer above (the top: free space, E = F = 1)
    double E1[n], F1[n];
    if (k > 0) load_modes(k - 1, E1, F1);
    else {
#pragma unroll
      for (int m = 0; m < n; ++m) { E1[m] = (m == t) ? 1.0 : 0.0; F1[m] = E1[m]; }
    }
    double K[n], X[n];
    // ---- solve 1: H and H (2 gdn + z)
    static_for<0, n>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
      const double one = (t == i) ? 1.0 : 0.0;
      K[i] = Z[i] + one;
      X[i] = fma(bc16<i>(gdn), 2.0 * dvec, vec ? Z[i] : one);
    });
    solve16<n>(K, X, low);
    double gg[S];
#pragma unroll
    for (int o = 0; o < S; ++o) {
      const double cmv = lr[O.cm(o, 0) + cl];
      const double tv = fma(tdu, rr[o], cmv);
      double w = 0.0;
      static_for<0, n>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        w = fma(bc16<i>(tv), X[i], w);
      });
      hh[o] = fma(tdu, hh[o], bc16<n>(w) + lr[O.csrc(o)]);
      gg[o] = fma(tk, fma(2.0, w, -cmv), lr[O.cl(o, 0) + cl]);
    }
    // ---- reflection at the layer's top and solve 2
    double A[n];
    static_for<0, n>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
      const double one = (t == i) ? 1.0 : 0.0;
      double v = vec ? X[i] : fma(2.0, X[i], -one);
      v = fma(bc16<i>(gdn), -dvec, v);
      v = v * tk * bc16<i>(tk);
      v = fma(bc16<i>(gup), dvec, v);
      K[i] = v + one;
      X[i] = v;
    });
    mul_at<n>(F, E1, A);
    if constexpr (MIX) {
      double D[n], B[n];
      mul_at<n>(F, E, D);
#pragma unroll
      for (int r = 0; r < n; ++r) { D[r] -= (r == t) ? 1.0 : 0.0; B[r] = A[r]; }
      sub_mul<n>(D, A, B);
#pragma unroll
      for (int r = 0; r < n; ++r) { X[r] = vec ? X[r] : B[r]; Z[r] = B[r]; }
    } else {
#pragma unroll
      for (int r = 0; r < n; ++r) { X[r] = vec ? X[r] : A[r]; Z[r] = A[r]; }
    }
    solve16<n>(K, X, low);
#pragma unroll
    for (int o = 0; o < S; ++o) {
      double w = 0.0;
      static_for<0, n>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        w = fma(bc16<i>(gg[o]), X[i], w);
      });
      hh[o] -= bc16<n>(w);
      rr[o] = col ? w : 0.0;
    }
    double Q[n];
#pragma unroll
    for (int r = 0; r < n; ++r) Q[r] = fma(2.0, X[r], vec ? 0.0 : -Z[r]);
    mul_at<n>(A, Q, Z);
    if constexpr (MIX) {
      if (k > 0) {
        double D[n], B[n];
        mul_at<n>(E1, F1, D);
#pragma unroll
        for (int r = 0; r < n; ++r) { D[r] -= (r == t) ? 1.0 : 0.0; B[r] = Z[r]; }
        sub_mul<n>(D, Z, B);
#pragma unroll
        for (int r = 0; r < n; ++r) Z[r] = B[r];
      }
    }
#pragma unroll
    for (int r = 0; r < n; ++r) { E[r] = E1[r]; F[r] = F1[r]; }
  }
  // ---- no downwelling field at the top: (1 + Z) u = z, I = r . u + h
  double cum[S];
  {
    double K[n], X[n];
#pragma unroll
    for (int i = 0; i < n; ++i) { K[i] = Z[i] + ((t == i) ? 1.0 : 0.0); X[i] = Z[i]; }
    solve16<n>(K, X, low);
#pragma unroll
    for (int o = 0; o < S; ++o) {
      double w = 0.0;
      static_for<0, n>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        w = fma(bc16<i>(rr[o]), X[i], w);
      });
      cum[o] = bc16<n>(w) + hh[o];
    }
  }

  // ---- Fourier convergence on the item's lane 0, or hand-over to k_rescue
  bool goes_on = false;
  if (t == 0 && valid) {
    if (W.nfour[it] != 0 || !(low > 1.0e-9)) {
      W.nfour[it] = M + 1;   // (k_rescue takes the item up at this term)
      W.rlist[atomicAdd(W.rcnt, 1)] = it;
    } else {
      goes_on = converge_term<N, S>(W, it, obs, oi, ff, M, cum);
    }
  }
  const int noff = append_items(W, it, L, goes_on, nnext, next, W.lcnt + M + 1);
  const int goff = __builtin_amdgcn_ds_bpermute(4 * (lane - t), noff);
  if (goff >= 0)
    for (int l = t; l < L; l += 16) W.lown[goff + l] = it;
}

}  // namespace
}  // namespace aa
