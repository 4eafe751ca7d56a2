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
// 201 -> 59 ms (127 with the records stored straight from the lanes), mixed,
// 240,004 items 110 -> 63 ms (168); N = 12, 1,200 items 32.8 -> 2.8 ms (4.9);
// three Stokes components N = 4, 16,000 items 361 -> 45 ms (71; 12 of them
// k_sabdab).  At N = 6 the records are written at 2.1 TB/s and the VALU issues
// 5.5k instructions per wavefront.
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
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int j = lane >> 3, i = lane & 7;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const double v = lds[8 * q + j][i];
      if (8 * q + j < left) base[(size_t)(8 * q + j) * AS + f0 + i] = v;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
};

// One thread per (item, layer).  VGPR budget: the n x n matrix of the Jacobi
// iteration (2 n^2 registers) and the factor G; two wavefronts
// per SIMD up to n = 6, one above.
template <int N, int S, bool MIX>
__global__ __launch_bounds__(64, (N * S <= (MIX ? 4 : 6)) ? 2 : 1) void k_modes(RTWork W, int M0, int group) {
  constexpr int n = N * S, LM = 2 * N, NT = n * (n + 1) / 2;
  constexpr bool SPLIT = n > 8;   // source terms in a second pass over the stored modes
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
  if constexpr (!MIX && S == 1) {
#pragma unroll
    for (int i = 0; i < n; ++i)
#pragma unroll
      for (int j = 0; j <= i; ++j) {
        a[ix(i, j)] = i == j ? Qt[QO.rmu(i)] : 0.0;
        b[ix(i, j)] = a[ix(i, j)];
      }
#pragma unroll
    for (int l = 0; l < LM; ++l) {
      if (l < M || l > NMOM) continue;
      const double o = ogp[l];
#pragma unroll
      for (int i = 0; i < n; ++i) {
        const double w = o * ph[QO.xq(M, l, i, 0, 0)];
#pragma unroll
        for (int j = 0; j <= i; ++j) {
          double* s = (l & 1) ? b : a;
          s[ix(i, j)] = fma(-w, ph[QO.xq(M, l, j, 0, 0)], s[ix(i, j)]);
        }
      }
    }
  } else {
    using TSD = typename std::conditional<MIX, float, double>::type;
    const TSD* rec;
    if constexpr (MIX) rec = W.sab32 + (sb + il) * (size_t)(2 * n * n);
    else rec = W.sab64 + (sb + il) * (size_t)(2 * n * n);
    const TSD* ra = rec + (odd ? n * n : 0);
    const TSD* rb = rec + (odd ? 0 : n * n);
#pragma unroll
    for (int i = 0; i < n; ++i)
#pragma unroll
      for (int j = 0; j <= i; ++j) {
        const double sc = Qt[QO.g(i / S)] * Qt[QO.rg(j / S)];
        double va = (double)ra[i * n + j] * sc, vb = (double)rb[i * n + j] * sc;
        if constexpr (MIX) {
          const double st = Qt[QO.g(j / S)] * Qt[QO.rg(i / S)];
          const double ta = (double)ra[j * n + i] * st, tb = (double)rb[j * n + i] * st;
          xa[ix(i, j)] = 0.5 * (va - ta);
          xb[ix(i, j)] = 0.5 * (vb - tb);
          va = 0.5 * (va + ta);
          vb = 0.5 * (vb + tb);
        }
        a[ix(i, j)] = i == j ? va + Qt[QO.rmu(i / S)] : va;
        b[ix(i, j)] = i == j ? vb + Qt[QO.rmu(i / S)] : vb;
      }
  }
  if constexpr (n > 2) {   // partial isolation (the reference's prepass), n > 2 only as there
    bool some = false, all = true;
#pragma unroll
    for (int i = 0; i < n; ++i) {
      double s = 0.0;
#pragma unroll
      for (int j = 0; j < n; ++j)
        if (j != i) s += fabs(a[i > j ? ix(i, j) : ix(j, i)]) + fabs(b[i > j ? ix(i, j) : ix(j, i)]);
      some = some || s == 0.0;
      all = all && s == 0.0;
    }
    ok = !some || all;
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
  double nrm[n];
  {
    // cosine of the columns' angle, about twice the rounding of an n-term dot
    // product
    constexpr double TOL2 = (6.0e-16 * n) * (6.0e-16 * n);
    bool conv = false;
#pragma unroll 1
    for (int sweep = 0; sweep < 16; ++sweep) {
      bool rot = false;
#pragma unroll
      for (int j = 0; j < n; ++j) {
        double v = 0.0;
#pragma unroll
        for (int r = 0; r < n; ++r) v = fma(c[j][r], c[j][r], v);
        nrm[j] = v;
      }
#pragma unroll
      for (int i = 0; i < n - 1; ++i)
#pragma unroll
        for (int j = i + 1; j < n; ++j) {
          double g = 0.0;
#pragma unroll
          for (int r = 0; r < n; ++r) g = fma(c[i][r], c[j][r], g);
          const bool act = g * g > TOL2 * (nrm[i] * nrm[j]);
          if (__ballot(act) == 0ull) continue;   // no lane rotates: skip the update
          rot = rot || act;
          // t = sign(z) / (|z| + sqrt(1 + z^2)), z = (|cj|^2 - |ci|^2) / (2 g)
          const float gf = (float)(2.0 * g), df = (float)(nrm[j] - nrm[i]);
          const float z = df * __builtin_amdgcn_rcpf(gf);
          // (the square root saturates before z^2 overflows; it is |z| there)
          const float az = fabsf(z), zm = fminf(az, 1.0e18f);
          const float ta = __builtin_amdgcn_rcpf(az + fmaxf(az, __builtin_amdgcn_sqrtf(fmaf(zm, zm, 1.0f))));
          const double tt = act ? (double)copysignf(ta, z) : 0.0;
          const double cs = rsqrt_nr(fma(tt, tt, 1.0)), sn = cs * tt;
          nrm[i] = fma(-tt, g, nrm[i]);
          nrm[j] = fma(tt, g, nrm[j]);
#pragma unroll
          for (int r = 0; r < n; ++r) {
            const double p = c[i][r], q = c[j][r];
            c[i][r] = fma(-sn, q, cs * p);
            c[j][r] = fma(sn, p, cs * q);
          }
        }
      conv = !rot;
      if (__ballot(rot) == 0ull) break;
    }
    ok = ok && conv;
  }
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
  double em[SPLIT ? 1 : n][n];   // E'
  if constexpr (!SPLIT) {
#pragma unroll
    for (int k = 0; k < n; ++k) efcol(k, em[k]);
  }
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
  if constexpr (SPLIT) {
    static_for<0, n>([&](auto kc) __attribute__((always_inline)) {
      constexpr int k = decltype(kc)::value;
      double e[n];
      efcol(k, e);
      static_for<0, n>([&](auto rc) __attribute__((always_inline)) {
        constexpr int r = decltype(rc)::value;
        out.put<O.e(r, k), AS>(odd ? c[k][r] : e[r]);
      });
      static_for<0, n>([&](auto rc) __attribute__((always_inline)) {
        constexpr int r = decltype(rc)::value;
        out.put<O.f(r, k), AS>(odd ? e[r] : c[k][r]);
      });
    });
    // the second pass reads the lane's own record back, which other lanes
    // wrote (a last piece that the modes leave incomplete is written again
    // when it is full)
    if constexpr (((2 * n * n) & 7) != 0) out.template flush<(2 * n * n) & ~7, AS>();
    __threadfence_block();
  } else {
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

  // ---- user-angle and beam vectors: the sums over the degrees are taken
  // before those over the streams (per layer 2N rows of n, then n products
  // per mode, where the reference forms n Legendre sums per mode)
  const double* trr = W.tr + il * TR_NFIELDS;
  const double dtau = trr[TR_DTAU], tduser = trr[TR_TDUSER], avsec = trr[TR_AVSEC], itrans = trr[TR_ITRANS];
  const double tdmubar = trr[TR_TDMUBAR], itransu = trr[TR_ITRANSU], emultup = trr[TR_EMULTUP], sigp = trr[TR_SIGP];
  const bool lsc = (M < 3) ? true : (((W.lsc[il] >> M) & 1u) != 0u);
  const bool beam = (layer + 1 <= W.beam_cutoff[it]) && lsc;
  const double usec = W.usec[it];
  double va[S][n], vb[S][n], qa[n], qb[n];
#pragma unroll
  for (int r = 0; r < n; ++r) {
    qa[r] = 0.0; qb[r] = 0.0;
#pragma unroll
    for (int o = 0; o < S; ++o) { va[o][r] = 0.0; vb[o][r] = 0.0; }
  }
  {
    const double* __restrict__ pis = W.pis + (size_t)it * PO.size();
#pragma unroll
    for (int l = 0; l < LM; ++l) {
      if (l < M || l > NMOM) continue;
      if constexpr (S == 1) {
        const double o = ogp[l];
        const double cu = 0.5 * o * pis[PO.at(M, l, 0, 0)], cq = o * pis[PO.at(M, l, 1, 0)];
#pragma unroll
        for (int i = 0; i < n; ++i) {
          const double f = ph[QO.xq(M, l, i, 0, 0)];
          if (l & 1) { vb[0][i] = fma(cu, f, vb[0][i]); qb[i] = fma(cq, f, qb[i]); }
          else { va[0][i] = fma(cu, f, va[0][i]); qa[i] = fma(cq, f, qa[i]); }
        }
      } else {
        double og[S][S], pu[S == 1 ? 1 : 3];
#pragma unroll
        for (int o1 = 0; o1 < S; ++o1)
#pragma unroll
          for (int o2 = 0; o2 < S; ++o2) og[o1][o2] = ogp[(l * S + o1) * S + o2];
#pragma unroll
        for (int p = 0; p < (S == 1 ? 1 : 3); ++p) pu[p] = pis[PO.at(M, l, 0, p)];
        const double p0 = pis[PO.at(M, l, 1, 0)];
        double cu[S][S];   // 1/2 DMAT(o1) PI_user(o1, o) B(o, o')
#pragma unroll
        for (int o1 = 0; o1 < S; ++o1)
#pragma unroll
          for (int o2 = 0; o2 < S; ++o2) {
            double v = 0.0;
#pragma unroll
            for (int o = 0; o < S; ++o)
              if ((o == 2) == (o2 == 2)) v = fma(pi_el<S>(pu, o1, o), og[o][o2], v);
            cu[o1][o2] = (o1 == 2 ? -0.5 : 0.5) * v;
          }
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
          for (int o2 = 0; o2 < S; ++o2) {
#pragma unroll
            for (int o3 = 0; o3 < S; ++o3) {
              if ((o2 == 0) != (o3 == 0)) continue;   // PI has no element between I and (Q, U)
              const double f = ph[QO.xq(M, l, i, o2, o3)];
              const bool cb_ = ((l & 1) != 0) != (o2 == 2);   // parity class of (l, o')
#pragma unroll
              for (int o1 = 0; o1 < S; ++o1) {
                if (cb_) vb[o1][i * S + o3] = fma(cu[o1][o2], f, vb[o1][i * S + o3]);
                else va[o1][i * S + o3] = fma(cu[o1][o2], f, va[o1][i * S + o3]);
              }
              if (o2 < 2) {
                const double q = og[o2][0] * p0;
                // (row o3 of PI, column o2: PI is symmetric)
                if (l & 1) qb[i * S + o3] = fma(q, f, qb[i * S + o3]);
                else qa[i * S + o3] = fma(q, f, qa[i * S + o3]);
              }
            }
          }
      }
    }
    const int g = global_item(W, it);
    const int obs = g / W.nch, ch = g - obs * W.nch;
    const double F1 = (W.flux ? W.flux[(size_t)obs * W.nch + ch] : 1.0) / PI4;
#pragma unroll
    for (int r = 0; r < n; ++r) { qa[r] *= F1; qb[r] *= F1; }
  }

  // ---- per mode: multipliers, source coefficients, beam amplitudes
  const double sg = odd ? -1.0 : 1.0;
  const double* lrec = W.abuf + (sb + t) * AS;
  double otr[n], ogu[n], ogd[n], ocl[S][n], ocm[S][n];
  double spar[S];
#pragma unroll
  for (int o = 0; o < S; ++o) spar[o] = 0.0;
  const double itw = -itrans * tdmubar;
#pragma unroll
  for (int k = 0; k < n; ++k) {
    double e[n], f[n];
#pragma unroll
    for (int r = 0; r < n; ++r) {
      if constexpr (SPLIT) {
        e[r] = lrec[(odd ? O.f(0, 0) : O.e(0, 0)) + O.e(r, k)];
        f[r] = lrec[(odd ? O.e(0, 0) : O.f(0, 0)) + O.e(r, k)];
      } else {
        e[r] = em[k][r];
        f[r] = c[k][r];
      }
    }
    double ua[S], ub[S], qe = 0.0, qf = 0.0;
#pragma unroll
    for (int o = 0; o < S; ++o) {
      double s1 = 0.0, s2 = 0.0;
#pragma unroll
      for (int r = 0; r < n; ++r) { s1 = fma(va[o][r], e[r], s1); s2 = fma(vb[o][r], f[r], s2); }
      ua[o] = s1; ub[o] = s2;
    }
#pragma unroll
    for (int r = 0; r < n; ++r) { qe = fma(qa[r], e[r], qe); qf = fma(qb[r], f[r], qf); }
    const double kv = keig[k];
    const double help = kv * dtau;
    const double zdel = (help > MAX_TAU_PATH) ? 0.0 : exp(-help);
    // HMULT (REG/vlidort_solutions.f90:1651-1790)
    const double rho_m = usec - kv;
    const bool hs = fabs(rho_m) < TAYLOR_SMALL;
    double h1 = usec * (zdel - tduser) * rcp_nr(rho_m);
    if (hs) h1 = taylor1(rho_m, dtau, tduser, usec);
    const double h2 = usec * (1.0 - zdel * tduser) * rcp_nr(usec + kv);
    double gup = 0.0, gdn = 0.0, cm[S];
#pragma unroll
    for (int o = 0; o < S; ++o) {
      const double upup = ua[o] + ub[o], updn = sg * (ua[o] - ub[o]);
      cm[o] = lsc ? upup * h1 : 0.0;
      ocl[o][k] = lsc ? updn * h2 : 0.0;
      ocm[o][k] = cm[o];
    }
    if (beam) {
      // Green's-function amplitudes (:2649-2932)
      const double gamp = avsec + kv, gamm = avsec - kv;
      const bool gs = fabs(gamm) < TAYLOR_SMALL;
      const double rgp = rcp_nr(gamp), rgm = rcp_nr(gamm);
      const double aterm = qe + qf, bterm = sg * (qe - qf);
      double cf = itrans * (zdel - tdmubar) * rgm;
      double sd = (itrans * h2 - emultup) * rgm;
      if (gs) {
        cf = taylor1(gamm, dtau, tdmubar, itrans);
        sd = itransu * taylor2(gamm, sigp, dtau, 1.0, tdmubar * tduser, 1.0);
      }
      const double df = itrans * (1.0 - zdel * tdmubar) * rgp;
      const double su = fma(itw, h1, emultup) * rgp;
      gdn = cf * aterm;
      gup = df * bterm;
#pragma unroll
      for (int o = 0; o < S; ++o) {
        const double upup = ua[o] + ub[o], updn = sg * (ua[o] - ub[o]);
        spar[o] += updn * sd * aterm + upup * su * bterm - cm[o] * gdn;
      }
    }
    otr[k] = zdel;
    ogu[k] = gup;
    ogd[k] = gdn;
  }
  // the rest of the record in field order, padded to whole pieces
  static_for<O.t(0), AS>([&](auto fc) __attribute__((always_inline)) {
    constexpr int f = decltype(fc)::value, q = f - O.t(0), w = q / n, k = q % n;
    double v = 0.0;
    if constexpr (w == 0) v = otr[k];
    else if constexpr (w == 1) v = ogu[k];
    else if constexpr (w == 2) v = ogd[k];
    else if constexpr (w < 3 + S) v = ocl[w - 3][k];
    else if constexpr (w < 3 + 2 * S) v = ocm[w - 3 - S][k];
    else if constexpr (f - O.csrc(0) < S) v = spar[f - O.csrc(0)];
    out.put<f, AS>(v);
  });
}

}  // namespace
}  // namespace aa
