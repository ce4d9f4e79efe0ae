// Plain FP64 path of the FENE-P / IBM SMAC step (the parity path).
// Compiled with -ffp-contract=off: every expression is evaluated in the
// order written, which is the order of the reference statement it restates.
#include "fp_device.h"
#include "fp_sor.h"
#include <algorithm>
#include <map>
#include <cmath>

namespace fp {

static inline int nblk(long n, int t) { return (int)((n + t - 1) / t); }

// ============================================================ FENE-P ======
// Value e of an FP64 plane of n values.  Below 2^29 cells through a raw
// buffer resource (base and size in scalar registers, one 32-bit byte offset
// per lane); BIG: through 64-bit addresses.
template <bool BIG>
__device__ __forceinline__ double ldv(const double* __restrict__ base, long n, unsigned e) {
  if constexpr (BIG) {
    return base[e];
  } else {
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)((unsigned)n * 8u), 0x00020000);
    return __builtin_bit_cast(double, (v2u)__builtin_amdgcn_raw_buffer_load_b64(r, (int)(e * 8u), 0, 0));
  }
}
// offset, in cells, of the neighbour at distance d along an axis of n cells
// whose stride is 2^ls (periodic)
__device__ __forceinline__ int wrapped(int a, int d, int n, int ls) { return (int)((unsigned)(((a + d) & (n - 1)) - a) << ls); }

// Coefficients of the candidate faces (cand_p, cand_n) as fma(cp, c, fma(cm,
// a, z b)): halves and quarters multiply exactly, (3 z)/2 rounds as 1.5 z, and a
// term that a candidate lacks adds zero, so the value is cand_p's, bit for bit,
// where that term is finite.
struct FaceCoef {
  double a, b, c;
  __device__ __forceinline__ double operator()(double cm, double z, double cp) const {
    return __builtin_fma(cp, c, __builtin_fma(cm, a, z * b));
  }
};
__device__ __forceinline__ FaceCoef face_p(int l) {
  return {l == 1 ? 0.5 : (l == 2 ? 0.25 : 0.0), l == 0 ? 1.5 : (l == 1 ? 0.5 : 1.0), l == 0 ? -0.5 : (l == 2 ? -0.25 : 0.0)};
}
__device__ __forceinline__ FaceCoef face_n(int l) {
  return {l == 1 ? -0.5 : (l == 2 ? -0.25 : 0.0), l == 0 ? 0.5 : (l == 1 ? 1.5 : 1.0), l == 0 ? 0.5 : (l == 2 ? 0.25 : 0.0)};
}

// Cstar (fenep.f90:464-507) + Lyapunov Newton (fenep.f90:518-585) + the
// Peterlin factor of the new C (f, fenep.f90:510-515, used by polymer_stress).
// The four faces of a cell and axis come from one line of five cells (30 loads an
// axis; each face with its own loads took 72).  Bound by FP64 issue: the
// Newton's 6 x 6 elimination and its central-difference Jacobian.  256x128x128
// between walls: 1420 -> 500-540 us (quotients by a shared divisor through its
// reciprocal, row swaps only where a wavefront needs one, 7 shifts a Newton
// iteration instead of 13, the shared line); 64^3: 85 -> 41 us.
template <bool WL, bool BIG>
__global__ __launch_bounds__(128) void k_cstar_newton(Grid g, CstarConst K, const double* __restrict__ C,
                                                      const uint8_t* __restrict__ sel, const double* __restrict__ U,
                                                      const double* __restrict__ V, const double* __restrict__ W,
                                                      double* __restrict__ Cn, double* __restrict__ fC, int* __restrict__ nitr) {
  const long L = xcd_cell();
  if (L >= g.n) return;
  long m;
  int i, j, k;
  band_cell(g, L, m, i, j, k);
  const double dt = g.dt;
  const unsigned mu = (unsigned)m;
  const int lz = g.lnx + g.lny;
  const int xm = wrapped(i, -1, g.nx, 0), xp = wrapped(i, 1, g.nx, 0);
  const int ym = wrapped(j, -1, g.ny, g.lnx), yp = wrapped(j, 1, g.ny, g.lnx);
  const int zm = wrapped(k, -1, g.nz, lz), zp = wrapped(k, 1, g.nz, lz);
  const bool wlo = WL && j == 0, whi = WL && j == g.ny - 1;
#define LD(F, o) ldv<BIG>(F, g.n, mu + (unsigned)(o))
  double cx[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
  for (int d = 0; d < 3; d++) {
    double v1, v2;
    if (d == 0) { v1 = LD(U, xm); v2 = LD(U, 0); }
    else if (d == 1) { v1 = wlo ? 0.0 : LD(V, ym); v2 = whi ? 0.0 : LD(V, 0); }   // V_kabe
    else { v1 = LD(W, zm); v2 = LD(W, 0); }
    const double h2 = K.h2[d], ih2 = K.ih2[d];
    const double s1 = quot_finite((-v2 + fabs(v2)) * dt, h2, ih2);
    const double s2 = 1.0 / 6.0 + quot_finite((-v2 - fabs(v2)) * dt, h2, ih2);
    const double s3 = 1.0 / 6.0 + quot_finite((v1 - fabs(v1)) * dt, h2, ih2);
    const double s4 = quot_finite((v1 + fabs(v1)) * dt, h2, ih2);
    const int a = d == 0 ? i : (d == 1 ? j : k), na = d == 0 ? g.nx : (d == 1 ? g.ny : g.nz);
    const int ls = d == 0 ? 0 : (d == 1 ? g.lnx : lz);
    const int om = wrapped(a, -1, na, ls), op = wrapped(a, 1, na, ls);
    const unsigned e[5] = {mu + (unsigned)wrapped(a, -2, na, ls), mu + (unsigned)om, mu, mu + (unsigned)op,
                           mu + (unsigned)wrapped(a, 2, na, ls)};
    const int lm = (sel[mu + (unsigned)om] >> (2 * d)) & 3, l0 = (sel[mu] >> (2 * d)) & 3,
              lp = (sel[mu + (unsigned)op] >> (2 * d)) & 3;
    const FaceCoef pl = face_p(l0), pr = face_p(lp), nl = face_n(lm), nr = face_n(l0);
    double v[6][5];
#pragma unroll
    for (int q = 0; q < 6; q++)
#pragma unroll
      for (int o = 0; o < 5; o++) v[q][o] = ldv<BIG>(C + q * g.n, g.n, e[o]);
    // the ghost rows (C_kabe): 2 C_0 - C_1; a point beyond them only feeds
    // faces whose weight is zero (a wavefront shares its row where nx >= 64)
    if (WL && d == 1 && (j < 2 || j >= g.ny - 2)) {
      const bool i0 = j == 0, i1 = j == 1, h1 = j == g.ny - 2, h0 = j == g.ny - 1;
#pragma unroll
      for (int q = 0; q < 6; q++) {
        v[q][1] = i0 ? 2.0 * v[q][2] - v[q][3] : v[q][1];
        v[q][0] = i0 ? v[q][2] : (i1 ? 2.0 * v[q][1] - v[q][2] : v[q][0]);
        v[q][3] = h0 ? 2.0 * v[q][2] - v[q][1] : v[q][3];
        v[q][4] = h0 ? v[q][2] : (h1 ? 2.0 * v[q][3] - v[q][2] : v[q][4]);
      }
    }
    double sum[6];
    bool odd = false;
#pragma unroll
    for (int q = 0; q < 6; q++) {
      double acc = cx[q] + s3 * pl(v[q][1], v[q][2], v[q][3]);   // Cp(a-1): own left face
      acc = acc + s1 * pr(v[q][2], v[q][3], v[q][4]);            // Cp(a): left face of a+1
      acc = acc + s4 * nl(v[q][0], v[q][1], v[q][2]);            // Cn(a-1): right face of a-1
      acc = acc + s2 * nr(v[q][1], v[q][2], v[q][3]);            // Cn(a): own right face
      sum[q] = acc;
      odd = odd || !(fabs(acc) < INFINITY);
    }
    // a coefficient of zero times an infinity or NaN: again, with the terms
    // that the faces have
    if (__any(odd)) {
#pragma unroll 1
      for (int q = 0; q < 6; q++) {
        double w[5];
#pragma unroll
        for (int o = 0; o < 5; o++) w[o] = v[0][o];
#pragma unroll
        for (int u = 1; u < 6; u++)
#pragma unroll
          for (int o = 0; o < 5; o++) w[o] = u == q ? v[u][o] : w[o];
        double acc = cx[0];
#pragma unroll
        for (int u = 1; u < 6; u++) acc = u == q ? cx[u] : acc;
        acc = acc + s3 * cand_p(l0, w[1], w[2], w[3]);
        acc = acc + s1 * cand_p(lp, w[2], w[3], w[4]);
        acc = acc + s4 * cand_n(lm, w[0], w[1], w[2]);
        acc = acc + s2 * cand_n(l0, w[1], w[2], w[3]);
#pragma unroll
        for (int u = 0; u < 6; u++) sum[u] = u == q ? acc : sum[u];
      }
    }
#pragma unroll
    for (int q = 0; q < 6; q++) cx[q] = sum[q];
  }
  // Lyapunov
  double b[6];
#pragma unroll
  for (int q = 0; q < 6; q++) b[q] = cx[q];
  b[0] = b[0] + K.dtwi;
  b[3] = b[3] + K.dtwi;
  b[5] = b[5] + K.dtwi;
  // the boundary rules (U_kabe, V_kabe, W_kabe) at the reads that reach a ghost
  // row or the wall face of V; B the row -1, 0, 1 of the read
#define UL(a, B, c) uw(U, a, B, c)
#define VL(a, B, c) vw(a, B, c)
#define WV(a, B, c) uw(W, a, B, c)
  auto row = [&](int B) { return B < 0 ? ym : (B > 0 ? yp : 0); };
  auto uw = [&](const double* F, int a, int B, int c) {
    const double x = LD(F, a + ((B < 0 && wlo) || (B > 0 && whi) ? 0 : row(B)) + c);
    return B < 0 && wlo ? -x : (B > 0 && whi ? 2.0 * 0.0 - x : x);
  };
  auto vw = [&](int a, int B, int c) {
    const double x = LD(V, a + row(B) + c);
    return (B < 0 && wlo) || (B == 0 && whi) ? 0.0 : x;
  };
  double a11 = -quot_finite(dt * (-UL(xm, 0, 0) + UL(0, 0, 0)), K.h[0], K.ih[0]);
  double a12 = -quot_finite(dt * (((-VL(xm, -1, 0) + VL(xp, -1, 0)) - VL(xm, 0, 0)) + VL(xp, 0, 0)), K.h4[0], K.ih4[0]);
  double a13 = -quot_finite(dt * (((-WV(xm, 0, zm) + WV(xp, 0, zm)) - WV(xm, 0, 0)) + WV(xp, 0, 0)), K.h4[0], K.ih4[0]);
  double a21 = -quot_finite(dt * (((-UL(xm, -1, 0) - UL(0, -1, 0)) + UL(xm, 1, 0)) + UL(0, 1, 0)), K.h4[1], K.ih4[1]);
  double a22 = -quot_finite(dt * (-VL(0, -1, 0) + VL(0, 0, 0)), K.h[1], K.ih[1]);
  double a23 = -quot_finite(dt * (((-WV(0, -1, zm) + WV(0, 1, zm)) - WV(0, -1, 0)) + WV(0, 1, 0)), K.h4[1], K.ih4[1]);
  double a31 = -quot_finite(dt * (((-UL(xm, 0, zm) - UL(0, 0, zm)) + UL(xm, 0, zp)) + UL(0, 0, zp)), K.h4[2], K.ih4[2]);
  double a32 = -quot_finite(dt * (((-VL(0, -1, zm) - VL(0, 0, zm)) + VL(0, -1, zp)) + VL(0, 0, zp)), K.h4[2], K.ih4[2]);
  double a33 = -quot_finite(dt * (-WV(0, 0, zm) + WV(0, 0, 0)), K.h[2], K.ih[2]);
#undef UL
#undef VL
#undef WV
  double A[9] = {a11, a12, a13, a21, a22, a23, a31, a32, a33};  // transpose(A0), column-major
  double x[6];
#pragma unroll
  for (int q = 0; q < 6; q++) x[q] = ldv<BIG>(C + q * g.n, g.n, mu);
#undef LD
  const int it = newton_d(K, A, b, x, dt);
#pragma unroll
  for (int q = 0; q < 6; q++) Cn[q * g.n + m] = x[q];
  fC[m] = peterlin_d(g.lp, x[0], x[3], x[5]);
  nitr[m] = it > K.itrmax ? -K.itrmax : it;   // negative: stopped at the cap
}

// ========================================================= predictor ======
// C0 = f(C) C - E at (i,j,k) with ghosts (polymer_stress, fenep.f90:655-659)
template <bool WL>
__device__ __forceinline__ double c0_at(const Grid& g, const double* __restrict__ C, const double* __restrict__ fC,
                                        int q, int i, int j, int k) {
  const double E = (q == 0 || q == 3 || q == 5) ? 1.0 : 0.0;
  if (g.walls && (j < 0 || j >= g.ny)) {
    double c0 = ldbw<WL>(C, g, i, j, k, BC_C), c3 = ldbw<WL>(C + 3 * g.n, g, i, j, k, BC_C), c5 = ldbw<WL>(C + 5 * g.n, g, i, j, k, BC_C);
    double f = peterlin_d(g.lp, c0, c3, c5);
    return f * ldbw<WL>(C + q * g.n, g, i, j, k, BC_C) - E;
  }
  long m = cidx(g, wrapi(i, g.nx), wrapi(j, g.ny), wrapi(k, g.nz));
  return fC[m] * C[q * g.n + m] - E;
}

// the predictor's own inputs of a cell, read where they are used
template <bool WL>
struct PredAt {
  const Grid& g;
  const double *A0, *T0, *B0, *F, *P;
  int i, j, k;
  long m;
  __device__ __forceinline__ double a0(int c) const { return A0[c * g.n + m]; }
  __device__ __forceinline__ double t0(int c) const { return T0[c * g.n + m]; }
  __device__ __forceinline__ double b0(int c) const { return B0[c * g.n + m]; }
  __device__ __forceinline__ double f(int c) const { return F ? F[c * g.n + m] : 0.0; }
  __device__ __forceinline__ double p() const { return P[m]; }
  __device__ __forceinline__ double p1(int c) const {
    return ldbw<WL>(P, g, i + (c == 0), j + (c == 1), k + (c == 2), BC_P);
  }
};
// the same, all loaded ahead
struct PredIn {
  double a[3], t[3], b[3], fv[3], pm, pp[3];
  template <bool WL>
  __device__ __forceinline__ void load(const PredAt<WL>& s, int first) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      a[c] = first ? 0.0 : s.a0(c);
      t[c] = first ? 0.0 : s.t0(c);
      b[c] = first ? 0.0 : s.b0(c);
      fv[c] = s.f(c);
      pp[c] = s.p1(c);
    }
    pm = s.p();
  }
  __device__ __forceinline__ double a0(int c) const { return a[c]; }
  __device__ __forceinline__ double t0(int c) const { return t[c]; }
  __device__ __forceinline__ double b0(int c) const { return b[c]; }
  __device__ __forceinline__ double f(int c) const { return fv[c]; }
  __device__ __forceinline__ double p() const { return pm; }
  __device__ __forceinline__ double p1(int c) const { return pp[c]; }
};

// divisors of the predictor with their correctly rounded reciprocals (quot)
struct PredConst {
  double dx, dy, dz, dxx, dyy, dzz, dx4, dy4, dz4;
  double idx, idy, idz, idxx, idyy, idzz, idx4, idy4, idz4;
};
// One cell of the predictor over a stencil accessor S (v(c, ..): velocity
// component c, c0(q, ..): C0, at an offset from the cell) and the cell's own inputs
// `in`: convection (fenep.f90:694-734), viscous (736-770), polymer_stress
// (645-691) and the predictor right-hand side of navier (803-826),
// fft_navier (1466-1511) or ibm_preliminary (1994-2013), with the history
// updates A0=A, T0=T, B0=B done in place.
template <bool WL, class Acc, class In>
__device__ __forceinline__ void pred_cell(const Grid& g, const PredConst& K, const Acc& S, const In& in, int method,
                                          int first, int polymer, int i, int j, int k, long m, double* A0, double* T0,
                                          double* B0, double* __restrict__ Rout, double bf0, double bf1, double bf2,
                                          double* __restrict__ Q) {
  const double dt = g.dt;
#define DIV(n, d) quot(n, K.d, K.i##d)
#define Ug(a, b, c) S.v(0, (a) - i, (b) - j, (c) - k)
#define Vg(a, b, c) S.v(1, (a) - i, (b) - j, (c) - k)
#define Wg(a, b, c) S.v(2, (a) - i, (b) - j, (c) - k)
  double a[3], bv[3], t[3];
  {
    double h1 = (Ug(i - 1, j, k) + Ug(i, j, k)) / 2.0, h2 = (Ug(i, j, k) + Ug(i + 1, j, k)) / 2.0;
    double ax = (DIV(-(h1 * h1) + h2 * h2, dx)
                 + DIV(-((((Vg(i, j - 1, k) + Vg(i + 1, j - 1, k)) / 2.0) * (Ug(i, j - 1, k) + Ug(i, j, k))) / 2.0)
                    + (((Vg(i, j, k) + Vg(i + 1, j, k)) / 2.0) * (Ug(i, j, k) + Ug(i, j + 1, k))) / 2.0, dy))
                + DIV(-((((Wg(i, j, k - 1) + Wg(i + 1, j, k - 1)) / 2.0) * (Ug(i, j, k - 1) + Ug(i, j, k))) / 2.0)
                   + (((Wg(i, j, k) + Wg(i + 1, j, k)) / 2.0) * (Ug(i, j, k) + Ug(i, j, k + 1))) / 2.0, dz);
    double g1 = (Vg(i, j - 1, k) + Vg(i, j, k)) / 2.0, g2 = (Vg(i, j, k) + Vg(i, j + 1, k)) / 2.0;
    double ay = (DIV(-((((Ug(i - 1, j, k) + Ug(i - 1, j + 1, k)) / 2.0) * (Vg(i - 1, j, k) + Vg(i, j, k))) / 2.0)
                  + (((Ug(i, j, k) + Ug(i, j + 1, k)) / 2.0) * (Vg(i, j, k) + Vg(i + 1, j, k))) / 2.0, dx)
                 + DIV(-(g1 * g1) + g2 * g2, dy))
                + DIV(-((((Wg(i, j, k - 1) + Wg(i, j + 1, k - 1)) / 2.0) * (Vg(i, j, k - 1) + Vg(i, j, k))) / 2.0)
                   + (((Wg(i, j, k) + Wg(i, j + 1, k)) / 2.0) * (Vg(i, j, k) + Vg(i, j, k + 1))) / 2.0, dz);
    double e1 = (Wg(i, j, k - 1) + Wg(i, j, k)) / 2.0, e2 = (Wg(i, j, k) + Wg(i, j, k + 1)) / 2.0;
    double az = (DIV(-((((Ug(i - 1, j, k) + Ug(i - 1, j, k + 1)) / 2.0) * (Wg(i - 1, j, k) + Wg(i, j, k))) / 2.0)
                  + (((Ug(i, j, k) + Ug(i, j, k + 1)) / 2.0) * (Wg(i, j, k) + Wg(i + 1, j, k))) / 2.0, dx)
                 + DIV(-((((Vg(i, j - 1, k) + Vg(i, j - 1, k + 1)) / 2.0) * (Wg(i, j - 1, k) + Wg(i, j, k))) / 2.0)
                    + (((Vg(i, j, k) + Vg(i, j, k + 1)) / 2.0) * (Wg(i, j, k) + Wg(i, j + 1, k))) / 2.0, dy))
                + DIV(-(e1 * e1) + e2 * e2, dz);
    a[0] = -ax; a[1] = -ay; a[2] = -az;
  }
  const double cb = g.beta / g.re;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    double x0 = S.v(c, (i) - i, (j) - j, (k) - k);
    double bb = (DIV((S.v(c, (i - 1) - i, (j) - j, (k) - k) - 2.0 * x0) + S.v(c, (i + 1) - i, (j) - j, (k) - k), dxx)
                 + DIV((S.v(c, (i) - i, (j - 1) - j, (k) - k) - 2.0 * x0) + S.v(c, (i) - i, (j + 1) - j, (k) - k), dyy))
                + DIV((S.v(c, (i) - i, (j) - j, (k - 1) - k) - 2.0 * x0) + S.v(c, (i) - i, (j) - j, (k + 1) - k), dzz);
    bv[c] = cb * bb;
  }
  if (polymer) {
#define C0g(q, aa, bb, cc) S.c0(q, (aa) - i, (bb) - j, (cc) - k)
    double tx = (DIV(-C0g(0, i, j, k) + C0g(0, i + 1, j, k), dx)
                 + DIV(((-C0g(1, i, j - 1, k) - C0g(1, i + 1, j - 1, k)) + C0g(1, i, j + 1, k)) + C0g(1, i + 1, j + 1, k), dy4))
                + DIV(((-C0g(2, i, j, k - 1) - C0g(2, i + 1, j, k - 1)) + C0g(2, i, j, k + 1)) + C0g(2, i + 1, j, k + 1), dz4);
    double ty = (DIV(((-C0g(1, i - 1, j, k) + C0g(1, i + 1, j, k)) - C0g(1, i - 1, j + 1, k)) + C0g(1, i + 1, j + 1, k), dx4)
                 + DIV(-C0g(3, i, j, k) + C0g(3, i, j + 1, k), dy))
                + DIV(((-C0g(4, i, j, k - 1) - C0g(4, i, j + 1, k - 1)) + C0g(4, i, j, k + 1)) + C0g(4, i, j + 1, k + 1), dz4);
    double tz = (DIV(((-C0g(2, i - 1, j, k) + C0g(2, i + 1, j, k)) - C0g(2, i - 1, j, k + 1)) + C0g(2, i + 1, j, k + 1), dx4)
                 + DIV(((-C0g(4, i, j - 1, k) + C0g(4, i, j + 1, k)) - C0g(4, i, j - 1, k + 1)) + C0g(4, i, j + 1, k + 1), dy4))
                + DIV(-C0g(5, i, j, k) + C0g(5, i, j, k + 1), dz);
#undef C0g
    const double coef = (1.0 - g.beta) / (g.re * g.wi);
    t[0] = coef * tx; t[1] = coef * ty; t[2] = coef * tz;
  } else {
    t[0] = t[1] = t[2] = 0.0;
  }
  const double bfs[3] = {bf0, bf1, bf2};
#pragma unroll
  for (int c = 0; c < 3; c++) {
    long o = c * g.n + m;
    double a0 = first ? a[c] : in.a0(c);
    double t0 = first ? t[c] : in.t0(c);
    double b0 = first ? bv[c] : in.b0(c);
    double u = S.v(c, (i) - i, (j) - j, (k) - k);
    const double dpn = dt * (-in.p() + in.p1(c));
    double dp = c == 0 ? DIV(dpn, dx) : (c == 1 ? DIV(dpn, dy) : DIV(dpn, dz));
    double fv = in.f(c) + bfs[c];
    double r;
    if (method == FP_METHOD_EXPLICIT) {
      r = (((u - dp) + (dt * (3.0 * (a[c] + bv[c]) - (a0 + b0))) / 2.0) + (dt * (t[c] + t0)) / 2.0) + dt * fv;
    } else if (method == FP_METHOD_FFT) {
      r = ((((u - dp) + (dt * (3.0 * a[c] - a0)) / 2.0) + (dt * bv[c]) / 2.0) + (dt * (t[c] + t0)) / 2.0) + dt * fv;
    } else {
      r = ((((u - dp) + (dt * (3.0 * a[c] - a0)) / 2.0) + dt * bv[c]) + (dt * (t[c] + t0)) / 2.0) + dt * fv;
    }
    Q[o] = r;
    A0[o] = a[c];
    T0[o] = t[c];
    B0[o] = bv[c];
    // ibm_predict's right-hand side where no marker reaches (f = 0): the wall
    // row of V counts as 0 there
    if (Rout) {
      const bool wall = WL && c == 1 && j == g.ny - 1;
      Rout[o] = ((wall ? 0.0 : r) + 0.0) - (dt * bv[c]) / 2.0;
    }
  }
#undef DIV
#undef Ug
#undef Vg
#undef Wg
}

// any grid: the stencil through the boundary-rule accessor
template <bool WL>
struct PredGlobal {
  const Grid& g;
  const double *U, *V, *W, *C, *fC;
  int i, j, k;
  __device__ __forceinline__ double v(int c, int a, int b, int d) const {
    return ldbw<WL>(c == 0 ? U : (c == 1 ? V : W), g, i + a, j + b, k + d, c == 0 ? BC_U : (c == 1 ? BC_V : BC_W));
  }
  __device__ __forceinline__ double c0(int q, int a, int b, int d) const {
    return c0_at<WL>(g, C, fC, q, i + a, j + b, k + d);
  }
};
template <bool WL>
__global__ __launch_bounds__(256) void k_predictor(Grid g, PredConst K, int method, int first, int polymer,
                                                   const double* __restrict__ U, const double* __restrict__ V,
                                                   const double* __restrict__ W, const double* __restrict__ P,
                                                   const double* __restrict__ C, const double* __restrict__ fC,
                                                   double* __restrict__ A0, double* __restrict__ T0, double* __restrict__ B0,
                                                   double* __restrict__ Rout, const double* __restrict__ F, double bf0,
                                                   double bf1, double bf2, double* __restrict__ Q) {
  const long L = xcd_cell();
  if (L >= g.n) return;
  long m;
  int i, j, k;
  band_cell(g, L, m, i, j, k);
  const PredAt<WL> in{g, A0, T0, B0, F, P, i, j, k, m};
  const PredGlobal<WL> S{g, U, V, W, C, fC, i, j, k};
  pred_cell<WL>(g, K, S, in, method, first, polymer, i, j, k, m, A0, T0, B0, Rout, bf0, bf1, bf2, Q);
}

// Streamed along z: a block walks kc planes of a 32 by 8 tile with U, V, W and
// C0 of three planes and a one-cell halo in the LDS, C0 = f C - E formed once a
// point instead of at each of its 22 uses, the next plane's loads in flight
// in registers.  k_predictor's wavefronts wait on some 120 loads each from
// the caches: 541 us at 256x128x128 there (with divisions; 520 without) and 289
// here, 64^3 27 and 18, 64x64x32 16 and 12.4.
#define PD_TX 32
#define PD_TY 8
#define PD_HX (PD_TX + 2)
#define PD_PTS (PD_HX * (PD_TY + 2))
struct PredLds64 {
  const double *m, *z, *p;   // planes k-1, k, k+1: nine fields of PD_PTS points
  int at;
  __device__ __forceinline__ double v(int c, int a, int b, int d) const {
    return (d < 0 ? m : (d > 0 ? p : z))[c * PD_PTS + at + a + PD_HX * b];
  }
  __device__ __forceinline__ double c0(int q, int a, int b, int d) const { return v(3 + q, a, b, d); }
};
struct PdRegs {
  double v[2][10];   // two points a thread: U, V, W, f, C
};
template <bool WL>
__device__ __forceinline__ void pd_fetch(const Grid& g, int i0, int j0, int k, int polymer, const double* __restrict__ U,
                                         const double* __restrict__ V, const double* __restrict__ W,
                                         const double* __restrict__ C, const double* __restrict__ fC, PdRegs& r) {
#pragma unroll
  for (int e = 0; e < 2; e++) {
    const int pt = threadIdx.x + 256 * e;
    if (pt >= PD_PTS) break;
    const int i = wrapi(i0 + pt % PD_HX - 1, g.nx);
    int j = j0 + pt / PD_HX - 1;
    j = WL ? min(max(j, 0), g.ny - 1) : wrapi(j, g.ny);
    const long m = cidx(g, i, j, wrapi(k, g.nz));
    r.v[e][0] = U[m];
    r.v[e][1] = V[m];
    r.v[e][2] = W[m];
    if (polymer) {
      r.v[e][3] = fC[m];
#pragma unroll
      for (int q = 0; q < 6; q++) r.v[e][4 + q] = C[q * g.n + m];
    }
  }
}
template <bool WL>
__device__ __forceinline__ void pd_put(const Grid& g, int i0, int j0, int k, int polymer, const double* __restrict__ C,
                                       const double* __restrict__ fC, const PdRegs& r, double* __restrict__ slot) {
#pragma unroll
  for (int e = 0; e < 2; e++) {
    const int pt = threadIdx.x + 256 * e;
    if (pt >= PD_PTS) break;
    const int j = j0 + pt / PD_HX - 1;
    const bool lo = WL && j < 0, hi = WL && j >= g.ny;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      double v = r.v[e][c];
      if (WL) {   // U_kabe, V_kabe, W_kabe
        if (c == 1) v = lo || j >= g.ny - 1 ? 0.0 : v;
        else v = lo ? -v : (hi ? 2.0 * 0.0 - v : v);
      }
      slot[c * PD_PTS + pt] = v;
    }
    if (!polymer) continue;
    if (lo || hi) {
      const int i = wrapi(i0 + pt % PD_HX - 1, g.nx), kz = wrapi(k, g.nz);
      for (int q = 0; q < 6; q++) slot[(3 + q) * PD_PTS + pt] = c0_at<WL>(g, C, fC, q, i, j, kz);
    } else {
#pragma unroll
      for (int q = 0; q < 6; q++) {
        const double E = (q == 0 || q == 3 || q == 5) ? 1.0 : 0.0;
        slot[(3 + q) * PD_PTS + pt] = r.v[e][3] * r.v[e][4 + q] - E;
      }
    }
  }
}
// grid: (nx / PD_TX) (ny / PD_TY) (nz / kc) blocks
template <bool WL>
__global__ __launch_bounds__(256, 2) void k_predictor_z(Grid g, PredConst K, int kc, int method, int first, int polymer,
                                                     const double* __restrict__ U, const double* __restrict__ V,
                                                     const double* __restrict__ W, const double* __restrict__ P,
                                                     const double* __restrict__ C, const double* __restrict__ fC, double* A0,
                                                     double* T0, double* B0, double* __restrict__ Rout,
                                                     const double* __restrict__ F, double bf0, double bf1, double bf2,
                                                     double* __restrict__ Q) {
  __shared__ double lds[3][9 * PD_PTS];
  const int ntx = g.nx / PD_TX, nty = g.ny / PD_TY;
  unsigned b = (unsigned)xcd_block();
  const int i0 = (int)(b % ntx) * PD_TX; b /= ntx;
  const int j0 = (int)(b % nty) * PD_TY;
  const int k0 = (int)(b / nty) * kc, k1 = k0 + kc;
  const int tx = threadIdx.x % PD_TX, ty = threadIdx.x / PD_TX;
  const int i = i0 + tx, j = j0 + ty;
  PdRegs r;
#pragma unroll 1
  for (int s = 0; s < 3; s++) {
    pd_fetch<WL>(g, i0, j0, k0 - 1 + s, polymer, U, V, W, C, fC, r);
    pd_put<WL>(g, i0, j0, k0 - 1 + s, polymer, C, fC, r, lds[s]);
  }
  int sm = 0, s0 = 1, sp = 2;
#pragma unroll 1
  for (int k = k0; k < k1; k++) {
    __syncthreads();
    const bool more = k + 1 < k1;
    if (more) pd_fetch<WL>(g, i0, j0, k + 2, polymer, U, V, W, C, fC, r);
    const long m = cidx(g, i, j, k);
    PredIn in;
    in.load(PredAt<WL>{g, A0, T0, B0, F, P, i, j, k, m}, first);
    const PredLds64 S{lds[sm], lds[s0], lds[sp], (ty + 1) * PD_HX + tx + 1};
    pred_cell<WL>(g, K, S, in, method, first, polymer, i, j, k, m, A0, T0, B0, Rout, bf0, bf1, bf2, Q);
    if (!more) break;
    __syncthreads();
    pd_put<WL>(g, i0, j0, k + 2, polymer, C, fC, r, lds[sm]);
    const int t = sm; sm = s0; s0 = sp; sp = t;
  }
}

// ======================================================= projection =======
// fft_poisson right-hand side (fenep.f90:1550-1552)
template <bool WL>
__global__ __launch_bounds__(256) void k_divergence(Grid g, const double* __restrict__ up, double* __restrict__ q) {
  const long L = xcd_cell();
  if (L >= g.n) return;
  long m;
  int i, j, k;
  band_cell(g, L, m, i, j, k);
  const double *Uu = up, *Vv = up + g.n, *Ww = up + 2 * g.n;
  q[m] = (((-ldbw<WL>(Uu, g, i - 1, j, k, BC_U) + ldbw<WL>(Uu, g, i, j, k, BC_U)) / g.dx
           + (-ldbw<WL>(Vv, g, i, j - 1, k, BC_V) + ldbw<WL>(Vv, g, i, j, k, BC_V)) / g.dy)
          + (-ldbw<WL>(Ww, g, i, j, k - 1, BC_W) + ldbw<WL>(Ww, g, i, j, k, BC_W)) / g.dz) / g.dt;
}

void f64_divergence(Ctx& c, const double* up, double* q) {
  hipLaunchKernelGGL(c.g.walls ? k_divergence<true> : k_divergence<false>, dim3(nblk(c.g.n, 256)), dim3(256), 0, c.stream, c.g, up, q);
}

// march / fft_march (fenep.f90:907-946, 1562-1604)
template <bool WL>
__global__ __launch_bounds__(256) void k_march(Grid g, int explicit_p, const double* __restrict__ up, const double* __restrict__ phi,
                                               double* __restrict__ U, double* __restrict__ V, double* __restrict__ W,
                                               double* __restrict__ P) {
  const long L = xcd_cell();
  if (L >= g.n) return;
  long m;
  int i, j, k;
  band_cell(g, L, m, i, j, k);
  const double dt = g.dt, dx = g.dx, dy = g.dy, dz = g.dz;
  const double *Uu = up, *Vv = up + g.n, *Ww = up + 2 * g.n;
#define PH(a, b, c) ldbw<WL>(phi, g, a, b, c, BC_P)
  double ph = phi[m];
  U[m] = ldbw<WL>(Uu, g, i, j, k, BC_U) - (dt * (-ph + PH(i + 1, j, k))) / dx;
  V[m] = ldbw<WL>(Vv, g, i, j, k, BC_V) - (dt * (-ph + PH(i, j + 1, k))) / dy;
  W[m] = ldbw<WL>(Ww, g, i, j, k, BC_W) - (dt * (-ph + PH(i, j, k + 1))) / dz;
  if (explicit_p) {
    P[m] = P[m] + ph;
  } else {
    const double coef = ((dt * g.beta) / g.re) / 2.0;
    double lap = ((((PH(i - 1, j, k) - 2.0 * ph) + PH(i + 1, j, k)) / (dx * dx)
                   + ((PH(i, j - 1, k) - 2.0 * ph) + PH(i, j + 1, k)) / (dy * dy))
                  + ((PH(i, j, k - 1) - 2.0 * ph) + PH(i, j, k + 1)) / (dz * dz));
    P[m] = (P[m] + ph) - coef * lap;
  }
#undef PH
}

// ============================================================ IBM ==========
// A step's IBM work is two launches: marker forces from Ua (k_ibm_forces), and
// the forced cells of the Helmholtz right-hand side (k_ibm_spread<true>), whose
// other cells the predictor has written.  Both are latency: short chains of
// dependent loads, so every thread has one sum only and its loads are issued
// ahead of the ordered additions.  256x128x128 between walls, 8 cylinders:
// 300 -> 82 us a step with the ghosted array, its folds and its pass gone.

// interpolation and marker forces of ibm_Helmholtz (fenep.f90:2076-2119,
// forces kept as in fenep_mpi.f90:1845-1853), one thread per marker and
// component: a marker per thread left 64^3 with 4 blocks (22 us).
// w: the 27 weights ibm_weight of each marker and component (k_ibm_interp_w).
template <bool WL>
__global__ __launch_bounds__(64) void k_ibm_forces(Grid g, long nmk, int nc, int nl, const double* __restrict__ mk,
                                                   const double* __restrict__ w, const double* __restrict__ ua,
                                                   double* __restrict__ mf) {
  const long id = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (id >= nmk) return;
  const int c = blockIdx.y;
  const int n = (int)(id / ((long)nc * nl)) + 1;
  const double dx3 = (g.dx * g.dx) * g.dx;
  int i0, j0; ibm_origin_d(g, c, mk[id], mk[nmk + id], i0, j0);
  const double* X = ua + c * g.n;
  const double* wm = w + (long)c * 27 * nmk + id;
  const int kind = c == 0 ? BC_U : (c == 1 ? BC_V : BC_W);
  double v[27], wv[27];
#pragma unroll
  for (int q = 0; q < 27; q++) {
    v[q] = ldbw<WL>(X, g, i0 - 1 + q % 3, j0 - 1 + q / 3 % 3, n - 2 + q / 9, kind);
    wv[q] = wm[q * nmk];
  }
  double acc = 0.0;
#pragma unroll
  for (int q = 0; q < 27; q++) acc = acc + (v[q] * wv[q]) * dx3;
  mf[c * nmk + id] = 0.0 + (mk[(3 + c) * nmk + id] - acc) / g.dt;
}

// spreading (fenep.f90:2125-2162) as a gather over the CSR of contributions
// of each ghosted target, in the reference's marker loop order
// (w: each entry's weight, k_ibm_spread_w), and the folds of ibm_PBM
// (fenep.f90:2195-2205) over each cell's ghost images.  A row that no marker
// reaches, and an image that does not exist, is the +0 of the cleared array;
// a sum begun at +0 is never -0, so adding it changes no bit.
// Three components: grid row blockIdx.y.
struct SpreadCsr {
  const int* rowp[3];
  const int* ent[3];
  const double* w[3];
  const long* cell[3];   // forced cells
  const int* row[3];     // their row; -1 - q: the 8 rows img[8q ..] (-1: none)
  const int* img[3];
  int cells[3];
};
__device__ __forceinline__ double spread_row(int r, const int* __restrict__ rowp, const int* __restrict__ ent,
                                             const double* __restrict__ w, const double* __restrict__ mf, double sw) {
  double acc = 0.0;
  if (r < 0) return acc;
  const int e1 = rowp[r + 1];
  for (int e = rowp[r]; e < e1; e += 8) {
    double f[8], x[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int p = e + q < e1 ? e + q : e1 - 1;
      f[q] = mf[ent[p]];
      x[q] = w[p];
    }
#pragma unroll
    for (int q = 0; q < 8; q++)
      if (e + q < e1) acc = acc + (f[q] * x[q]) * sw;
  }
  return acc;
}
// RHS: out = Ua + dt f - dt B/2, the right-hand side of ibm_predict
// (fenep.f90:2229), with in = Ua and B this step's viscous term.
// Otherwise out = in + f.
template <bool RHS, bool WL>
__global__ __launch_bounds__(64) void k_ibm_spread(Grid g, SpreadCsr cs, long nmk, const double* __restrict__ mf,
                                                   const double* in, const double* __restrict__ B, double* out) {
  const int c = blockIdx.y;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= cs.cells[c]) return;
  const int* rowp = cs.rowp[c];
  const int* ent = cs.ent[c];
  const double* w = cs.w[c];
  const double* mc = mf + c * nmk;
  const long m = cs.cell[c][t], o = c * g.n + m;
  const int r = cs.row[c][t];
  double f;
  if (r >= 0) {
    f = spread_row(r, rowp, ent, w, mc, g.sw);
  } else {
    const int* im = cs.img[c] + 8L * (-1 - r);   // x fastest: the folds go x, y, z
    f = 0.0;
    for (int kk = 0; kk < 2; kk++) {
      double z = 0.0;
      for (int jj = 0; jj < 2; jj++) {
        double y = 0.0;
        for (int ii = 0; ii < 2; ii++) y = y + spread_row(*im++, rowp, ent, w, mc, g.sw);
        z = z + y;
      }
      f = f + z;
    }
  }
  if (RHS) {
    double u = in[o];
    if (WL && c == 1) {
      int i, j, k;
      cell_ijk(g, m, i, j, k);
      u = ldbw<WL>(in + c * g.n, g, i, j, k, BC_V);
    }
    out[o] = (u + g.dt * f) - (g.dt * B[o]) / 2.0;
  } else {
    out[o] = in[o] + f;
  }
}

// The weights depend only on the markers and the grid: ibm_weight of every
// spreading entry (its marker at its row's target) and of every marker's 27
// interpolation points per component, evaluated once per marker set.
__global__ __launch_bounds__(256) void k_ibm_spread_w(Grid g, int comp, int rows, const int* __restrict__ rowp,
                                                      const long* __restrict__ tgt, const int* __restrict__ ent,
                                                      long nmk, const double* __restrict__ mk, double* __restrict__ w) {
  int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows) return;
  const long gx = g.nx + 2, gy = g.ny + 2;
  long t = tgt[r];
  int ii = (int)(t % gx), jj = (int)((t / gx) % gy), kk = (int)(t / (gx * gy));
  for (int e = rowp[r]; e < rowp[r + 1]; e++) {
    long id = ent[e];
    w[e] = ibm_weight(g, comp, ii, jj, kk, mk[id], mk[nmk + id], mk[2 * nmk + id]);
  }
}
__global__ __launch_bounds__(256) void k_ibm_interp_w(Grid g, long nmk, int nc, int nl, const double* __restrict__ mk,
                                                      double* __restrict__ w) {
  long id = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (id >= nmk) return;
  int n = (int)(id / ((long)nc * nl)) + 1;
  double xc = mk[id], yc = mk[nmk + id], zc = mk[2 * nmk + id];
  for (int c = 0; c < 3; c++) {
    int i0, j0; ibm_origin_d(g, c, xc, yc, i0, j0);
    double* wm = w + (long)c * 27 * nmk + id;   // point-major: the markers of a wavefront side by side
    for (int kk = n - 1; kk <= n + 1; kk++)
      for (int jj = j0; jj <= j0 + 2; jj++)
        for (int ii = i0; ii <= i0 + 2; ii++, wm += nmk) *wm = ibm_weight(g, c, ii, jj, kk, xc, yc, zc);
  }
}

static SpreadCsr spread_csr(Ctx& c, int& cmax) {
  SpreadCsr cs{};
  cmax = 0;
  for (int k = 0; k < 3; k++) {
    cs.rowp[k] = c.sp_row[k];
    cs.ent[k] = c.sp_ent[k];
    cs.w[k] = c.sp_w[k];
    cs.cell[k] = c.fc_cell[k];
    cs.row[k] = c.fc_row[k];
    cs.img[k] = c.fc_img[k];
    cs.cells[k] = c.fc_cells[k];
    cmax = std::max(cmax, c.fc_cells[k]);
  }
  return cs;
}

// out += spread of the marker values mfield (3 x nmk), over the forced cells
void f64_spread_add(Ctx& c, const double* mfield, double* out) {
  int cmax;
  const SpreadCsr cs = spread_csr(c, cmax);
  if (cmax > 0)
    hipLaunchKernelGGL((k_ibm_spread<false, false>), dim3(nblk(cmax, 64), 3), dim3(64), 0, c.stream, c.g, cs, c.nmk, mfield,
                       out, (const double*)nullptr, out);
}

// the marker forces of Ua = c.Q and the forced cells of c.Up; B0 is this
// step's B once the predictor has run
void f64_ibm(Ctx& c) {
  const Grid& g = c.g;
  hipStream_t s = c.stream;
  hipLaunchKernelGGL(g.walls ? k_ibm_forces<true> : k_ibm_forces<false>, dim3(nblk(c.nmk, 64), 3), dim3(64), 0, s, g, c.nmk,
                     c.nc, c.nl, c.mk, c.ib_w, c.Q, c.mf);
  int cmax;
  const SpreadCsr cs = spread_csr(c, cmax);
  auto k = g.walls ? k_ibm_spread<true, true> : k_ibm_spread<true, false>;
  if (cmax > 0) hipLaunchKernelGGL(k, dim3(nblk(cmax, 64), 3), dim3(64), 0, s, g, cs, c.nmk, c.mf, c.Q, c.B0, c.Up);
}

// Host-side construction of the spreading CSR: for each ghosted target the
// contributing (marker, stencil slot) pairs in the order of the reference's
// loops (markers n, m, l; then k, j, i), and the points that the ghost folds
// add to; the forced cells are the interior ones among them, each with the rows
// that it gathers (k_ibm_spread).
void f64_ibm_setup(Ctx& c) {
  const Grid& g = c.g;
  std::vector<double> mk(6 * c.nmk);
  FP_HIP_CHECK(hipMemcpy(mk.data(), c.mk, sizeof(double) * mk.size(), hipMemcpyDeviceToHost));
  const long gx = g.nx + 2, gy = g.ny + 2, gz = g.nz + 2, gn = gx * gy * gz;
  for (int comp = 0; comp < 3; comp++) {
    std::map<long, std::vector<int>> rows;
    for (long id = 0; id < c.nmk; id++) {
      int n = (int)(id / ((long)c.nc * c.nl)) + 1;
      double xc = mk[id], yc = mk[c.nmk + id];
      int i0, j0;
      if (comp == 0) { i0 = (int)(xc / g.dx - 0.5); j0 = (int)(yc / g.dy); }
      else if (comp == 1) { i0 = (int)(xc / g.dx); j0 = (int)(yc / g.dy - 0.5); }
      else { i0 = (int)(xc / g.dx); j0 = (int)(yc / g.dy); }
      int slot = 0;
      for (int kk = n - 1; kk <= n + 1; kk++)
        for (int jj = j0; jj <= j0 + 2; jj++)
          for (int ii = i0; ii <= i0 + 2; ii++, slot++) {
            if (ii < 0 || ii > g.nx + 1 || jj < 0 || jj > g.ny + 1 || kk < 0 || kk > g.nz + 1)
              throw std::string("IBM stencil outside the ghosted grid");
            rows[ii + gx * (jj + gy * (long)kk)].push_back((int)id);
          }
    }
    // fold closure
    std::vector<char> mark(gn, 0);
    for (auto& kv : rows) mark[kv.first] = 1;
    auto G = [&](long i, long j, long k) { return i + gx * (j + gy * k); };
    for (long k = 0; k < gz; k++) for (long j = 0; j < gy; j++) {
      mark[G(1, j, k)] |= mark[G(g.nx + 1, j, k)]; mark[G(g.nx, j, k)] |= mark[G(0, j, k)];
    }
    for (long k = 0; k < gz; k++) for (long i = 0; i < gx; i++) {
      mark[G(i, 1, k)] |= mark[G(i, g.ny + 1, k)]; mark[G(i, g.ny, k)] |= mark[G(i, 0, k)];
    }
    for (long j = 0; j < gy; j++) for (long i = 0; i < gx; i++) {
      mark[G(i, j, 1)] |= mark[G(i, j, g.nz + 1)]; mark[G(i, j, g.nz)] |= mark[G(i, j, 0)];
    }
    std::vector<int> rowp(1, 0), ent;
    std::vector<long> tgt;
    for (long t = 0; t < gn; t++) {
      if (!mark[t]) continue;
      auto it = rows.find(t);
      if (it != rows.end()) for (int id : it->second) ent.push_back(id);
      tgt.push_back(t);
      rowp.push_back((int)ent.size());
    }
    // the forced cells and the rows each one gathers: its own, and where it
    // borders a periodic axis those of its ghost images
    auto row_of = [&](long t) {
      const auto it = std::lower_bound(tgt.begin(), tgt.end(), t);
      return it != tgt.end() && *it == t ? (int)(it - tgt.begin()) : -1;
    };
    auto image = [](long i, int nn, int b) {   // a cell and its ghost image along an axis (-1: none)
      return !b ? i : (i == 1 ? (long)nn + 1 : (i == nn ? 0L : -1L));
    };
    std::vector<long> cell;
    std::vector<int> crow, img;
    for (size_t r = 0; r < tgt.size(); r++) {
      const long i = tgt[r] % gx, j = (tgt[r] / gx) % gy, k = tgt[r] / (gx * gy);
      if (i < 1 || i > g.nx || j < 1 || j > g.ny || k < 1 || k > g.nz) continue;
      int rr[8], ghosts = 0;
      const bool border = i == 1 || i == g.nx || j == 1 || j == g.ny || k == 1 || k == g.nz;
      for (int b = 0; border && b < 8; b++) {
        const long ii = image(i, g.nx, b & 1), jj = image(j, g.ny, b >> 1 & 1), kk = image(k, g.nz, b >> 2);
        rr[b] = b == 0 ? (int)r : (ii < 0 || jj < 0 || kk < 0 ? -1 : row_of(G(ii, jj, kk)));
        ghosts += b > 0 && rr[b] >= 0;
      }
      cell.push_back((i - 1) + g.nx * ((j - 1) + (long)g.ny * (k - 1)));
      crow.push_back(ghosts ? -1 - (int)(img.size() / 8) : (int)r);
      if (ghosts) img.insert(img.end(), rr, rr + 8);
    }
    for (void* q : {(void*)c.sp_row[comp], (void*)c.sp_tgt[comp], (void*)c.sp_ent[comp], (void*)c.sp_w[comp],
                    (void*)c.fc_cell[comp], (void*)c.fc_row[comp], (void*)c.fc_img[comp]})
      if (q) (void)hipFree(q);
    c.fc_cells[comp] = (int)cell.size();
    FP_HIP_CHECK(hipMalloc(&c.fc_cell[comp], sizeof(long) * std::max<size_t>(1, cell.size())));
    FP_HIP_CHECK(hipMalloc(&c.fc_row[comp], sizeof(int) * std::max<size_t>(1, crow.size())));
    FP_HIP_CHECK(hipMalloc(&c.fc_img[comp], sizeof(int) * std::max<size_t>(1, img.size())));
    if (!cell.empty()) {
      FP_HIP_CHECK(hipMemcpy(c.fc_cell[comp], cell.data(), sizeof(long) * cell.size(), hipMemcpyHostToDevice));
      FP_HIP_CHECK(hipMemcpy(c.fc_row[comp], crow.data(), sizeof(int) * crow.size(), hipMemcpyHostToDevice));
    }
    if (!img.empty()) FP_HIP_CHECK(hipMemcpy(c.fc_img[comp], img.data(), sizeof(int) * img.size(), hipMemcpyHostToDevice));
    c.sp_rows[comp] = (int)tgt.size();
    FP_HIP_CHECK(hipMalloc(&c.sp_row[comp], sizeof(int) * rowp.size()));
    FP_HIP_CHECK(hipMalloc(&c.sp_tgt[comp], sizeof(long) * std::max<size_t>(1, tgt.size())));
    FP_HIP_CHECK(hipMalloc(&c.sp_ent[comp], sizeof(int) * std::max<size_t>(1, ent.size())));
    FP_HIP_CHECK(hipMalloc(&c.sp_w[comp], sizeof(double) * std::max<size_t>(1, ent.size())));
    FP_HIP_CHECK(hipMemcpy(c.sp_row[comp], rowp.data(), sizeof(int) * rowp.size(), hipMemcpyHostToDevice));
    if (!tgt.empty()) FP_HIP_CHECK(hipMemcpy(c.sp_tgt[comp], tgt.data(), sizeof(long) * tgt.size(), hipMemcpyHostToDevice));
    if (!ent.empty()) FP_HIP_CHECK(hipMemcpy(c.sp_ent[comp], ent.data(), sizeof(int) * ent.size(), hipMemcpyHostToDevice));
    if (!tgt.empty())
      hipLaunchKernelGGL(k_ibm_spread_w, dim3(nblk((long)tgt.size(), 256)), dim3(256), 0, c.stream, g, comp,
                         (int)tgt.size(), c.sp_row[comp], c.sp_tgt[comp], c.sp_ent[comp], c.nmk, c.mk, c.sp_w[comp]);
  }
  if (c.ib_w) (void)hipFree(c.ib_w);
  FP_HIP_CHECK(hipMalloc(&c.ib_w, sizeof(double) * std::max<long>(1, 3 * 27 * c.nmk)));
  if (c.nmk > 0)
    hipLaunchKernelGGL(k_ibm_interp_w, dim3(nblk(c.nmk, 256)), dim3(256), 0, c.stream, g, c.nmk, c.nc, c.nl, c.mk, c.ib_w);
  FP_HIP_CHECK(hipGetLastError());
  FP_HIP_CHECK(hipStreamSynchronize(c.stream));
}

// ============================================================ SOR ==========
// Red-black SOR for the pressure-correction Poisson equation (the reference
// sweeps lexicographically with odd/even i per row, fenep.f90:885-901; the
// converged solution is the same to the solver tolerance).  Residuals are
// taken before each update, as E in the reference.
__global__ __launch_bounds__(256) void k_sor_color(Grid g, int color, double om, const double* __restrict__ q,
                                                   double* __restrict__ phi, double* __restrict__ e2,
                                                   const int* __restrict__ stop) {
  if (*stop) return;
  long h = blockIdx.x * (long)blockDim.x + threadIdx.x;
  long half = g.n / 2;
  double e = 0.0;
  if (h < half) {
    // enumerate cells of one colour: (i + j + k) % 2 == color
    long jk = h / (g.nx / 2);
    int j = (int)(jk % g.ny), k = (int)(jk / g.ny);
    int i = (int)(2 * (h % (g.nx / 2))) + ((j + k + color) & 1);
    long m = cidx(g, i, j, k);
    const double dx = g.dx, dy = g.dy, dz = g.dz;
    double BX = 1.0 / (dx * dx), BY = 1.0 / (dy * dy), BZ = 1.0 / (dz * dz);
    double B0 = ((((BX + BX) + BY) + BY) + BZ) + BZ;
    double p0 = phi[m];
    e = (((((BZ * ldb(phi, g, i, j, k - 1, BC_P) + BY * ldb(phi, g, i, j - 1, k, BC_P)) + BX * ldb(phi, g, i - 1, j, k, BC_P))
           - B0 * p0) + BX * ldb(phi, g, i + 1, j, k, BC_P)) + BY * ldb(phi, g, i, j + 1, k, BC_P)
         + BZ * ldb(phi, g, i, j, k + 1, BC_P)) - q[m];
    phi[m] = p0 + (om * e) / B0;
  }
  // block partial of e^2 (the second colour adds to the first's partial)
  __shared__ double sh[256];
  double s = block_sum256(e * e, sh);
  if (threadIdx.x == 0) e2[blockIdx.x] = color == 0 ? s : e2[blockIdx.x] + s;
}

__global__ __launch_bounds__(256) void k_sumsq(long n, const double* __restrict__ q, double* __restrict__ part) {
  long m = blockIdx.x * (long)blockDim.x + threadIdx.x;
  double v = m < n ? q[m] * q[m] : 0.0;
  __shared__ double sh[256];
  double s = block_sum256(v, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

constexpr int SOR_CHECK = 10;   // the residuals are looked at every so many sweeps

// flag[0] stop, [1] sweeps up to the first that met the test, [2] batches of
// SOR_CHECK sweeps made; host: their copy in pinned memory, once stopped.
// mode 0: er0 = sum Q^2, flags cleared (stop at once when Q = 0); mode 1: the
// residual sums of a batch of `rows` sweeps, `nb` partials each
__global__ __launch_bounds__(1024) void k_sor_decide(const double* __restrict__ part, int nb, int rows, double* __restrict__ er0,
                                                     double eps, int mode, int* __restrict__ flag, volatile int* host) {
  if (mode == 1 && flag[0]) return;
  __shared__ double res[SOR_CHECK];
  sor_row_sums(part, nb, rows, res);
  if (threadIdx.x != 0) return;
  if (mode == 0) {
    *er0 = res[0];
    flag[0] = res[0] == 0.0 ? 1 : 0;
    flag[1] = flag[2] = 0;
  } else {
    flag[2]++;
    for (int r = 0; r < rows && !flag[0]; r++) {
      flag[1]++;
      if (sqrt(res[r] / *er0) < eps) flag[0] = 1;
    }
  }
  // (a store across the bus costs microseconds: only what the host waits for)
  if (mode == 0 || flag[0]) {
    host[1] = flag[1];
    host[2] = flag[2];
    __threadfence_system();
    host[0] = flag[0];
  }
}

void f64_sor_create(Ctx& c) {
  const SorPlan<double> p = sor_plan<double>(c.g);
  const long nb = std::max(p.blocks, (long)nblk(c.g.n / 2, 256));
  FP_HIP_CHECK(hipMalloc((void**)&c.sor_part, sizeof(double) * SOR_CHECK * nb));
  FP_HIP_CHECK(hipMalloc((void**)&c.sor_flag, sizeof(int) * 4));
  FP_HIP_CHECK(hipHostMalloc((void**)&c.sor_host, 4 * sizeof(int), hipHostMallocDefault));
  for (int e = 0; e < 2; e++) FP_HIP_CHECK(hipEventCreateWithFlags(&c.sor_ev[e], hipEventDisableTiming));
}
void f64_sor_destroy(Ctx& c) {
  (void)hipFree(c.sor_part); (void)hipFree(c.sor_flag);
  if (c.sor_host) (void)hipHostFree(c.sor_host);
  for (int e = 0; e < 2; e++)
    if (c.sor_ev[e]) (void)hipEventDestroy(c.sor_ev[e]);
}

// Sweeps in batches of SOR_CHECK; every batch is enqueued before the host waits
// for the flags of the one before it (its launches end at once if that one
// stopped), so the device does not wait for the host.  The second array of the
// tiles is the previous C, which nothing reads after CStar.
int f64_sor(Ctx& c, const double* q, double* phi) {
  const Grid& g = c.g;
  hipStream_t s = c.stream;
  const double om = c.p.sor_omega > 0.0 ? c.p.sor_omega : 2.0 / (1.0 + sin(3.14159265358979323846 * g.dx));
  const SorPlan<double> plan = sor_plan<double>(g);
  const int nbh = nblk(g.n / 2, 256), nb = plan.k ? (int)plan.blocks : nbh;
  double* const buf[2] = {phi, c.C[1 - c.cur]};
  SorCoef<double> co;
  co.bx = 1.0 / (g.dx * g.dx); co.by = 1.0 / (g.dy * g.dy); co.bz = 1.0 / (g.dz * g.dz);
  co.b0 = ((((co.bx + co.bx) + co.by) + co.by) + co.bz) + co.bz;
  co.om = om; co.ib0 = 1.0 / co.b0;
  volatile int* h = c.sor_host;
  hipLaunchKernelGGL(k_sumsq, dim3(nblk(g.n, 256)), dim3(256), 0, s, g.n, q, c.part);
  hipLaunchKernelGGL(k_sor_decide, dim3(1), dim3(1024), 0, s, c.part, nblk(g.n, 256), 1, c.red, c.p.sor_eps, 0, c.sor_flag,
                     c.sor_host);
  std::vector<int> launches;   // made up to the end of each batch
  int at = 0, sweeps = 0;
  while (sweeps < c.p.sor_itrmax) {
    const int b = (int)launches.size(), batch = std::min(SOR_CHECK, c.p.sor_itrmax - sweeps);
    if (plan.k) {
      double* const from[2] = {buf[at & 1], buf[(at + 1) & 1]};
      at += sor_launch<double>(g, plan, co, q, from, c.sor_part, batch, false, c.sor_flag, s);
    } else {
      for (int r = 0; r < batch; r++)
        for (int color = 0; color < 2; color++)
          hipLaunchKernelGGL(k_sor_color, dim3(nbh), dim3(256), 0, s, g, color, om, q, phi, c.sor_part + (long)r * nbh, c.sor_flag);
    }
    sweeps += batch;
    launches.push_back(at);
    hipLaunchKernelGGL(k_sor_decide, dim3(1), dim3(1024), 0, s, c.sor_part, nb, batch, c.red, c.p.sor_eps, 1, c.sor_flag,
                       c.sor_host);
    FP_HIP_CHECK(hipEventRecord(c.sor_ev[b & 1], s));
    if (b > 0) FP_HIP_CHECK(hipEventSynchronize(c.sor_ev[(b - 1) & 1]));
    if (b > 0 && h[0]) break;
  }
  if (launches.empty()) return 0;
  FP_HIP_CHECK(hipEventSynchronize(c.sor_ev[(launches.size() - 1) & 1]));
  // the batches that ran: up to the stop, or all
  const int ran = h[0] ? h[2] : (int)launches.size();
  if (ran > 0 && (launches[ran - 1] & 1))
    FP_HIP_CHECK(hipMemcpyAsync(phi, buf[1], sizeof(double) * g.n, hipMemcpyDeviceToDevice, s));
  return h[0] ? h[1] : sweeps;
}

// ======================================================= per step =========
void f64_cstar_newton(Ctx& c) {
  const Grid& g = c.g;
  CstarConst K{};
  const double h[3] = {g.dx, g.dy, g.dz};
  for (int d = 0; d < 3; d++) {
    K.h[d] = h[d]; K.ih[d] = 1.0 / K.h[d];
    K.h2[d] = 2.0 * h[d]; K.ih2[d] = 1.0 / K.h2[d];
    K.h4[d] = 4.0 * h[d]; K.ih4[d] = 1.0 / K.h4[d];
  }
  K.wi = g.wi; K.iwi = 1.0 / g.wi; K.dtwi = g.dt / g.wi;
  K.L2 = g.lp * g.lp; K.L2m3 = K.L2 - 3.0;
  K.dc = c.p.newton_dc; K.dc2 = 2.0 * K.dc; K.idc2 = 1.0 / K.dc2;
  K.eps = c.p.newton_eps; K.itrmax = c.p.newton_itrmax;
  const bool big = g.n >= (1L << 29);
  auto kern = g.walls ? (big ? k_cstar_newton<true, true> : k_cstar_newton<true, false>)
                      : (big ? k_cstar_newton<false, true> : k_cstar_newton<false, false>);
  hipLaunchKernelGGL(kern, dim3(nblk(g.n, 128)), dim3(128), 0, c.stream, g, K, c.C[c.cur], c.sel, c.U, c.V, c.W,
                     c.C[1 - c.cur], c.fC, c.nitr);
  c.cur = 1 - c.cur;
}

void f64_predictor(Ctx& c) {
  const Grid& g = c.g;
  int polymer = c.p.beta != 1.0;
  double* Rout = c.p.method == FP_METHOD_IBM ? c.Up : nullptr;
  PredConst K{g.dx, g.dy, g.dz, g.dx * g.dx, g.dy * g.dy, g.dz * g.dz, 4.0 * g.dx, 4.0 * g.dy, 4.0 * g.dz};
  for (int q = 0; q < 9; q++) (&K.idx)[q] = 1.0 / (&K.dx)[q];
  const int first = c.has_history ? 0 : 1;
  const double* bf = c.p.body_force;
  // streamed where there are tiles for two blocks a CU: 32^3 has 128 (its step 10 us
  // a pass of 20 slower so); as many planes a block as leave 512 blocks
  const long tiles = g.nx % PD_TX || g.ny % PD_TY ? 0 : (g.nx / PD_TX) * (long)(g.ny / PD_TY);
  if (tiles * g.nz >= 512) {
    int kc = std::min(32, g.nz);
    while (tiles * (g.nz / kc) < 512) kc >>= 1;
    auto k = g.walls ? k_predictor_z<true> : k_predictor_z<false>;
    hipLaunchKernelGGL(k, dim3((unsigned)(tiles * (g.nz / kc))), dim3(256), 0, c.stream, g, K, kc, c.p.method, first, polymer,
                       c.U, c.V, c.W, c.P, c.C[c.cur], c.fC, c.A0, c.T0, c.B0, Rout, c.F, bf[0], bf[1], bf[2], c.Q);
    return;
  }
  hipLaunchKernelGGL(g.walls ? k_predictor<true> : k_predictor<false>, dim3(nblk(g.n, 256)), dim3(256), 0, c.stream, g, K,
                     c.p.method, first, polymer, c.U, c.V, c.W, c.P, c.C[c.cur], c.fC, c.A0, c.T0, c.B0, Rout, c.F, bf[0],
                     bf[1], bf[2], c.Q);
}

void f64_march(Ctx& c) {
  hipLaunchKernelGGL(c.g.walls ? k_march<true> : k_march<false>, dim3(nblk(c.g.n, 256)), dim3(256), 0, c.stream, c.g,
                     c.p.method == FP_METHOD_EXPLICIT ? 1 : 0, c.Up, c.Phi, c.U, c.V, c.W, c.P);
}

void f64_zero_c(Ctx& c) {
  zero_words(c.C[c.cur], 12 * c.g.n, c.stream);
}

}  // namespace fp
