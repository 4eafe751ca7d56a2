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
// update) per layer for small batches, the FP64 issue for large ones (N = 6: VALU
// busy four fifths of the time at three wavefronts per SIMD; an item and term
// read 66.8 KB, 832 bytes per layer and the beam's fields, 2.9 TB/s).  Measured
// against the pivoted band solve (k_bvp, 8 or 32 lanes per item): N = 6, 400,000
// items 204 -> 47 ms; one item 4.3 ms over its terms -> 0.13 ms (all terms side
// by side); N = 12, 1,200 items 15.5 -> 1.3 ms; three Stokes components N = 4,
// 16,000 items 133 -> 6.3 ms.
#pragma once
#include <type_traits>
#include "rt_work.h"
#include "rt_device.h"
#include "rt_modes.h"
#include "rt_converge.h"

namespace aa {

namespace {

// Lane broadcasts.  row_newbcast reads one lane of the caller's 16-lane row in
// all its lanes and is the one lane move that FP64 arithmetic takes as an
// operand modifier, so a broadcast multiply-add is a single v_fmac_f64 where
// the compiler emits a move and an FMA (k_adding, 400,000 items at N = 6 55 ->
// 47 ms; three Stokes components N = 4, 16,000 items 9.5 -> 6.8 ms).  A DPP operand must not be read
// within two wait states of its VALU write, and the compiler does not look
// into asm blocks: every block starts with s_nop 1, and inside a block no
// operand that was written before is read as a DPP operand.  All lanes of the
// row must be active (a broadcast under a lane's own condition reads nothing).

// x of lane K of the caller's 16-lane row, in all its lanes
template <int K>
__device__ __forceinline__ double bc16(double x) {
  double r;
  asm("s_nop 1\n\tv_mov_b64_dpp %0, %1 row_newbcast:%c2 row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(x), "n"(K));
  return r;
}
#define AA_DPP " row_newbcast:%c"
#define AA_MASK " row_mask:0xf bank_mask:0xf\n\t"
// z += a(lane I) * q and, in runs, z[j] += a(lane I + j) * q
template <int I>
__device__ __forceinline__ void fmac_bc(double& z, double a, double q) {
  asm("s_nop 1\n\tv_fmac_f64_dpp %0, %1, %2" AA_DPP "3" AA_MASK : "+&v"(z) : "v"(a), "v"(q), "n"(I));
}
template <int I>
__device__ __forceinline__ void fmac_bc2(double& z0, double& z1, double a, double q) {
  asm("s_nop 1\n\tv_fmac_f64_dpp %0, %2, %3" AA_DPP "4" AA_MASK "v_fmac_f64_dpp %1, %2, %3" AA_DPP "5" AA_MASK
      : "+&v"(z0), "+&v"(z1) : "v"(a), "v"(q), "n"(I), "n"(I + 1));
}
template <int I>
__device__ __forceinline__ void fmac_bc4(double& z0, double& z1, double& z2, double& z3, double a, double q) {
  asm("s_nop 1\n\tv_fmac_f64_dpp %0, %4, %5" AA_DPP "6" AA_MASK "v_fmac_f64_dpp %1, %4, %5" AA_DPP "7" AA_MASK
      "v_fmac_f64_dpp %2, %4, %5" AA_DPP "8" AA_MASK "v_fmac_f64_dpp %3, %4, %5" AA_DPP "9" AA_MASK
      : "+&v"(z0), "+&v"(z1), "+&v"(z2), "+&v"(z3)
      : "v"(a), "v"(q), "n"(I), "n"(I + 1), "n"(I + 2), "n"(I + 3));
}
// z[i] += a(lane i) * q for I <= i < n
template <int n, int I>
__device__ __forceinline__ void fmac_run(double (&z)[n], double a, double q) {
  if constexpr (n - I >= 4) {
    fmac_bc4<I>(z[I], z[I + 1], z[I + 2], z[I + 3], a, q);
    fmac_run<n, I + 4>(z, a, q);
  } else if constexpr (n - I >= 2) {
    fmac_bc2<I>(z[I], z[I + 1], a, q);
    fmac_run<n, I + 2>(z, a, q);
  } else if constexpr (n - I == 1) {
    fmac_bc<I>(z[I], a, q);
  }
}
// x[i] -= f[i](lane K) * xk for I <= i < E
template <int n, int K, int I, int E>
__device__ __forceinline__ void fnma_run(double (&x)[n], const double (&f)[n], double xk) {
  if constexpr (E - I >= 4) {
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, -%4, %8" AA_DPP "9" AA_MASK "v_fmac_f64_dpp %1, -%5, %8" AA_DPP "9" AA_MASK
        "v_fmac_f64_dpp %2, -%6, %8" AA_DPP "9" AA_MASK "v_fmac_f64_dpp %3, -%7, %8" AA_DPP "9" AA_MASK
        : "+&v"(x[I]), "+&v"(x[I + 1]), "+&v"(x[I + 2]), "+&v"(x[I + 3])
        : "v"(f[I]), "v"(f[I + 1]), "v"(f[I + 2]), "v"(f[I + 3]), "v"(xk), "n"(K));
    fnma_run<n, K, I + 4, E>(x, f, xk);
  } else if constexpr (E - I >= 2) {
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, -%2, %4" AA_DPP "5" AA_MASK "v_fmac_f64_dpp %1, -%3, %4" AA_DPP "5" AA_MASK
        : "+&v"(x[I]), "+&v"(x[I + 1]) : "v"(f[I]), "v"(f[I + 1]), "v"(xk), "n"(K));
    fnma_run<n, K, I + 2, E>(x, f, xk);
  } else if constexpr (E - I == 1) {
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, -%1, %2" AA_DPP "3" AA_MASK : "+&v"(x[I]) : "v"(f[I]), "v"(xk), "n"(K));
  }
}
// the same with f = x: x[i] -= x[i](lane K) * xk
template <int n, int K, int I>
__device__ __forceinline__ void fnma_self(double (&x)[n], double xk) {
  if constexpr (n - I >= 4) {
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, -%0, %4" AA_DPP "5" AA_MASK "v_fmac_f64_dpp %1, -%1, %4" AA_DPP "5" AA_MASK
        "v_fmac_f64_dpp %2, -%2, %4" AA_DPP "5" AA_MASK "v_fmac_f64_dpp %3, -%3, %4" AA_DPP "5" AA_MASK
        : "+&v"(x[I]), "+&v"(x[I + 1]), "+&v"(x[I + 2]), "+&v"(x[I + 3]) : "v"(xk), "n"(K));
    fnma_self<n, K, I + 4>(x, xk);
  } else if constexpr (n - I >= 2) {
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, -%0, %2" AA_DPP "3" AA_MASK "v_fmac_f64_dpp %1, -%1, %2" AA_DPP "3" AA_MASK
        : "+&v"(x[I]), "+&v"(x[I + 1]) : "v"(xk), "n"(K));
    fnma_self<n, K, I + 2>(x, xk);
  } else if constexpr (n - I == 1) {
    asm("s_nop 1\n\tv_fmac_f64_dpp %0, -%0, %1" AA_DPP "2" AA_MASK : "+&v"(x[I]) : "v"(xk), "n"(K));
  }
}
#undef AA_DPP
#undef AA_MASK

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
    fnma_run<n, k, k + 1, n>(X, K, X[k]);
    fnma_self<n, k, k + 1>(K, K[k]);
  });
  static_for<0, n - 1>([&](auto kc) __attribute__((always_inline)) {
    constexpr int k = n - 1 - decltype(kc)::value;
    fnma_run<n, k, 0, k>(X, K, X[k]);
  });
}

// Z = A^T Q over lanes: Z_i = sum_m A(m, i) Q_m (lane c: columns of A and Q)
template <int n>
__device__ __forceinline__ void mul_at(const double (&A)[n], const double (&Q)[n], double (&Z)[n]) {
#pragma unroll
  for (int i = 0; i < n; ++i) Z[i] = 0.0;
#pragma unroll
  for (int m = 0; m < n; ++m) fmac_run<n, 0>(Z, A[m], Q[m]);
}
// X -= A Q (A given by its columns: A(i, m) is register i of lane m)
template <int n>
__device__ __forceinline__ void sub_mul(const double (&A)[n], const double (&Q)[n], double (&X)[n]) {
  static_for<0, n>([&](auto mc) __attribute__((always_inline)) {
    constexpr int m = decltype(mc)::value;
    fnma_run<n, m, 0, n>(X, A, Q[m]);
  });
}

template <int N, int S, bool MIX>
__global__ __launch_bounds__(64) void k_adding(RTWork W, int M0, const int* __restrict__ active,
                                               const int* __restrict__ nactive) {
  constexpr int n = N * S, IPW = 4;
  const int tg = blockIdx.y, M = M0 + tg;   // this term of the group
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
  // the item's slots of this term
  const double* __restrict__ ab = W.abuf + ((size_t)tg * W.cap * km + W.loff[it]) * AS;
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
      const double x = r[O.e(m, c)], y = r[O.f(m, c)];
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

  // What a layer's step needs besides the modes, and the modes of the layers
  // above, are loaded a step ahead of their use (the modes two steps up to
  // n = 8, where the registers allow it): at the loop's top they would expose
  // the memory latency once per layer, 1.6 us per layer for a lone item.
  struct Step { double tk, gup, gdn, tdu, cm[S], cl[S], csrc[S]; };
  constexpr bool AHEAD2 = n <= 8;
  const int cl_ = col ? t : 0;
  auto load_step = [&](int k, Step& q) __attribute__((always_inline)) {
    const double* __restrict__ lr = ab + (size_t)k * AS;
    q.tk = lr[O.t(cl_)];
    q.gup = lr[O.gup(cl_)];
    q.gdn = lr[O.gdn(cl_)];
    q.tdu = trr[(size_t)k * TR_NFIELDS + TR_TDUSER];
#pragma unroll
    for (int o = 0; o < S; ++o) {
      q.cm[o] = lr[O.cm(o, cl_)];
      q.cl[o] = lr[O.cl(o, cl_)];
      q.csrc[o] = lr[O.csrc(o)];
    }
  };
  Step cur, nxt;
  load_step(L - 1, cur);
  double E1[n], F1[n];   // the layer above; the top has free space (E = F = 1) above
  double E2[AHEAD2 ? n : 1], F2[AHEAD2 ? n : 1];
  if constexpr (AHEAD2) load_modes(L > 1 ? L - 2 : 0, E1, F1);

  for (int k = Lmax - 1; k >= 0; --k) {
    if (k >= L) continue;   // uniform within the item's lanes
    if constexpr (AHEAD2) load_modes(k > 1 ? k - 2 : 0, E2, F2);
    else load_modes(k > 0 ? k - 1 : 0, E1, F1);
    load_step(k > 0 ? k - 1 : 0, nxt);
    if (k == 0) {
#pragma unroll
      for (int m = 0; m < n; ++m) { E1[m] = (m == t) ? 1.0 : 0.0; F1[m] = E1[m]; }
    }
    const double tk = col ? cur.tk : 1.0, gup = cur.gup, gdn = cur.gdn, tdu = cur.tdu;
    double K[n], X[n];
    // ---- solve 1: H and H (2 gdn + z)
    static_for<0, n>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
      const double one = (t == i) ? 1.0 : 0.0;
      K[i] = Z[i] + one;
      X[i] = vec ? Z[i] : one;
      fmac_bc<i>(X[i], gdn, 2.0 * dvec);
    });
    solve16<n>(K, X, low);
    double gg[S];
#pragma unroll
    for (int o = 0; o < S; ++o) {
      const double cmv = cur.cm[o];
      const double tv = fma(tdu, rr[o], cmv);
      double w = 0.0;
      static_for<0, n>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        fmac_bc<i>(w, tv, X[i]);
      });
      hh[o] = fma(tdu, hh[o], bc16<n>(w) + cur.csrc[o]);
      gg[o] = fma(tk, fma(2.0, w, -cmv), cur.cl[o]);
    }
    // ---- reflection at the layer's top and solve 2
    double A[n];
    static_for<0, n>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
      const double one = (t == i) ? 1.0 : 0.0;
      double v = vec ? X[i] : fma(2.0, X[i], -one);
      fmac_bc<i>(v, gdn, -dvec);
      v = v * tk;
      double w = 0.0;   // (the vector's lane adds gup; every lane of the row stays active)
      fmac_bc<i>(w, gup, dvec);
      fmac_bc<i>(w, tk, v);
      v = w;
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
        fmac_bc<i>(w, gg[o], X[i]);
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
    for (int r = 0; r < n; ++r) {
      E[r] = E1[r]; F[r] = F1[r];
      if constexpr (AHEAD2) { E1[r] = E2[r]; F1[r] = F2[r]; }
    }
    cur = nxt;
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
        fmac_bc<i>(w, rr[o], X[i]);
      });
      cum[o] = bc16<n>(w) + hh[o];
    }
  }

  if (t == 0 && valid) {
    const size_t e = (size_t)it * W.terms + tg;
#pragma unroll
    for (int o = 0; o < S; ++o) W.cums[e * S + o] = cum[o];
    if (!(low > 1.0e-9)) W.tflag[e] = 1;
  }
}

// The convergence test over a group's terms in order, one lane per item: an
// item that is done has its outputs written, one with a marked term goes to
// k_rescue at that term, the others enter the next group's lists.
template <int N, int S>
__global__ __launch_bounds__(64) void k_converge(RTWork W, int M0, int terms, const int* __restrict__ active,
                                                 const int* __restrict__ nactive, int* __restrict__ next,
                                                 int* __restrict__ nnext, int* __restrict__ lnext) {
  const int lane = threadIdx.x;
  int first = -1, cntb = 0;
  const int* lst = active;
  {
    int acc = 0;
#pragma unroll
    for (int b = 0; b < LBINS; ++b) {
      const int c = nactive[b], nbk = (c + 63) / 64;
      if (first < 0 && (int)blockIdx.x < acc + nbk) {
        first = ((int)blockIdx.x - acc) * 64;
        cntb = c;
        lst = active + (size_t)b * W.cap;
      }
      acc += nbk;
    }
  }
  if (first < 0) return;   // uniform over the wavefront
  const bool valid = first + lane < cntb;
  const int it = lst[valid ? first + lane : first];
  const int L = W.L_it[it];
  bool goes_on = false;
  if (valid) {
    const int gi = global_item(W, it), obs = gi / W.nch, ch = gi - obs * W.nch;
    const size_t oi = (size_t)ch * W.nobs + obs;
    const double ff = W.flux ? W.flux[(size_t)obs * W.nch + ch] : 1.0;
    for (int g = 0; g < terms; ++g) {
      const size_t e = (size_t)it * W.terms + g;
      if (W.tflag[e] != 0) {
        W.nfour[it] = M0 + g + 1;
        W.rlist[atomicAdd(W.rcnt, 1)] = it;
        goes_on = false;
        break;
      }
      double cum[S];
#pragma unroll
      for (int o = 0; o < S; ++o) cum[o] = W.cums[e * S + o];
      goes_on = converge_term<N, S>(W, it, obs, oi, ff, M0 + g, cum);
      if (!goes_on) break;
    }
  }
  const int off = append_items(W, it, L, goes_on, nnext, next, lnext);
  // the wavefront fills the slots of one item after the other
  for (unsigned long long todo = __ballot(off >= 0); todo != 0ull; todo &= todo - 1ull) {
    const int j = __ffsll((long long)todo) - 1;
    const int oj = __shfl(off, j, 64), Lj = __shfl(L, j, 64), ij = __shfl(it, j, 64);
    for (int l = lane; l < Lj; l += 64) W.lown[oj + l] = ij;
  }
}

}  // namespace
}  // namespace aa
