// C+- selection of the FP64 step (CpxCnx / CpyCny / CpzCnz, fenep.f90:169-382,
// with the Vieta test of fenep.f90:425-444).  Compiled with -ffp-contract=off;
// fused multiply-adds appear only where they are written out.
//
// Per cell and axis the selection is the maxloc over {v_0, v_1, v_2, 0} of v_l =
// min(lambda_min(Cp_l), lambda_min(Cn_l)).  lambda_min is first enclosed in an
// interval about an FP64 value that needs no arc cosine and cosine; where the
// intervals leave one option, it is the reference's.  The rest of a block's
// (cell, axis) pairs are collected in LDS and decided, packed, by the reference
// formula in FP64 (vieta_d), at the levels whose intervals can hold the maximum.
//
// Bound by FP64 issue: 1449 VALU operations a cell and plane, 1174 of them FP64
// (168 of 240 us at 256x128x128; three wavefronts per SIMD).  256x128x128
// between walls, us, by what is left to the formula, against 780-806 for the
// formula at every candidate in any state: nothing (smooth, with or without
// noise) 240-260, 0.25 % (noise of 1e-3 on C = I) 264 (304 without the short
// lists' own path), a third (uniform in z) 434, all (C = I) 783.  64^3, against
// 58-66: 22, 27 (39), 38 and 63.  (Intervals from FP32 arithmetic and a second
// kernel over a list took 178-190, 250, 715 and 2740, and 40, 45, 108 and 322.)
#include "fp_device.h"
#include <algorithm>

namespace fp {

namespace {

// ------------------------------------------------------------ the intervals
// With m = tr A / 3, B = A - m I, r^2 = tr B^2 / 6, arg = det B / (2 r^3):
//   lambda_min = m + 2 r psi(s),  psi(s) = cos(acos(1 - s^2)/3 + 2 pi/3),
//   s = sqrt(1 - arg) in [0, sqrt 2].
// psi is analytic there; its Chebyshev interpolant of degree 10 at 4000 nodes, in
// powers of s, is off by at most 7.1e-11.
__device__ constexpr double PSI[11] = {-0.5000000000704921,    -0.40824827798859914,   0.05555518775970136, -0.01889610882051598,
                                       0.008204572955364291,   -0.003949059904849778,  0.0019154248291659447,
                                       -0.0008342551567161861, 0.00028350823137773714, -6.30300867806705e-05,
                                       6.634523485078444e-06};
// What the value and the reference's own, v = vieta_d(A), can differ by, with
// u = 2^-53, S = |m| + 2 r (every |a_ii| <= S, every off-diagonal entry of A
// and every entry of B at most 2 r), rho = S / r >= 2, to first order:
//  reference   a2: 5 u S, a1: 24 u S^2, a0: 32 u S^3, so p = -3 r^2 carries
//              64 u S^2 and q = -det B carries 128 u S^3: arg is off by 64 u
//              rho^3 from q, 34 u rho^2 from p and 6 u from its own operations, at
//              most 82 u rho^3; its discriminant by 165 u rho^3 r^6; its root by
//              34 u rho^2 r beside what arg's error makes
//  this value  B's diagonal 4 u S: det 48 u r^2 S and 144 u r^3 of rounding, r^2
//              8 u r S: arg 36 u rho + 90 u, and 3 times the reciprocal square
//              root's error: that of v_rsq_f64 (2^-23; 2^-24.2 is the largest of 6.7e7
//              measured) is 1.5 2^-46 after one Newton step, 4.5 2^-46 = 576 u; r is off by 4 u S + 192 u r
//  lambda'     |d lambda / d arg| <= 0.41 r / sqrt(1 - arg), and 0.58 r /
//              sqrt(1 - arg) over an interval of half-width d where 1 - arg >= 2 d
// d = 1.43e-14 rho^3 + 1e-12, 128 u rho^3 + 9000 u, is above both errors of arg together.  Where |arg| <= 1
// - 2 d the reference is inside its square root's and arc cosine's domain and
// its discriminant is negative (1 - arg^2 >= 2 d > 165 u rho^3), and
//   |lambda - v| <= r (1.42e-10 + d / sqrt(1 - arg)),
// with 0.42 of the second term left for the roundings of r, m and the root.  Elsewhere, and
// where r^2 is outside [1e-90, 1e90] (the reference's discriminant, a sixth power
// of the entries, would leave the FP64 range) or not a number, the interval is
// infinite.
constexpr double SEL_D3 = 1.43e-14, SEL_D0 = 1e-12, SEL_PSI_ERR = 1.5e-10;

struct Lam {
  double v, e;   // lambda_min, half the width of its interval
};
__device__ __forceinline__ Lam lowest(const double (&a)[6]) {
  const double m = ((a[0] + a[3]) + a[5]) * (1.0 / 3.0);
  const double b11 = a[0] - m, b22 = a[3] - m, b33 = a[5] - m;
  const double o2 = __builtin_fma(a[1], a[1], __builtin_fma(a[2], a[2], a[4] * a[4]));
  const double hp = __builtin_fma(b11, b11, __builtin_fma(b22, b22, b33 * b33));
  const double r2 = __builtin_fma(hp, 1.0 / 6.0, o2 * (1.0 / 3.0));
  const double t1 = __builtin_fma(b22, b33, -(a[4] * a[4]));
  const double t2 = __builtin_fma(a[1], b33, -(a[4] * a[2]));
  const double t3 = __builtin_fma(a[1], a[4], -(b22 * a[2]));
  const double det = __builtin_fma(b11, t1, __builtin_fma(-a[1], t2, a[2] * t3));
  const double y0 = __builtin_amdgcn_rsq(r2);
  const double ir = __builtin_fma(0.5 * y0, __builtin_fma(-(r2 * y0), y0, 1.0), y0);
  const double r = r2 * ir;
  const double arg2 = det * ((ir * ir) * ir);   // 2 arg
  const double s2 = __builtin_fma(-0.5, arg2, 1.0);
  const double rho = __builtin_fma(fabs(m), ir, 2.0);
  const double d = __builtin_fma(SEL_D3 * (rho * rho), rho, SEL_D0);
  const double w = fmax(s2, d), z0 = __builtin_amdgcn_rsq(w), s0 = w * z0;
  const double s = __builtin_fma(0.5 * s0, __builtin_fma(-s0, z0, 1.0), s0);
  double ps = 2.0 * PSI[10];
#pragma unroll
  for (int q = 9; q >= 0; q--) ps = __builtin_fma(ps, s, 2.0 * PSI[q]);
  // (written so that a NaN fails)
  const bool ok = fabs(arg2) <= __builtin_fma(-4.0, d, 2.0) && r2 >= 1e-90 && r2 <= 1e90;
  return {__builtin_fma(r, ps, m), ok ? r * __builtin_fma(d, z0, SEL_PSI_ERR) : INFINITY};
}

// the candidates' entries (cand_p, cand_n: halves and quarters are exact, (3 c)/2
// rounds as 1.5 c)
__device__ __forceinline__ Lam lowest_face(bool right, int l, const double (&v)[3][6]) {
  double a[6];
#pragma unroll
  for (int q = 0; q < 6; q++) {
    const double cm = v[0][q], c = v[1][q], cp = v[2][q];
    const double near = right ? cp : cm, far = right ? cm : cp;
    a[q] = l == (right ? 0 : 1) ? __builtin_fma(near, 0.5, 0.5 * c)
           : l == 2 ? __builtin_fma(far, -0.25, __builtin_fma(near, 0.25, c))
                    : __builtin_fma(far, -0.5, 1.5 * c);
  }
  return lowest(a);
}
__device__ __forceinline__ Lam level(const Lam& p, const Lam& n) { return {fmin(p.v, n.v), fmax(p.e, n.e)}; }

// The option that the three levels' intervals leave, or 4 + bits: the levels
// (bits 0-2) that the formula has to decide between (and the zero slope).
__device__ __forceinline__ int decide(const Lam& a, const Lam& b, const Lam& c) {
  const double lo = fmax(fmax(fmax(a.v - a.e, b.v - b.e), c.v - c.e), 0.0);
  const bool ca = !(a.v + a.e < lo), cb = !(b.v + b.e < lo), cc = !(c.v + c.e < lo), cz = !(0.0 < lo);
  const int n = (int)ca + (int)cb + (int)cc + (int)cz;
  if (n == 1) return ca ? 0 : (cb ? 1 : (cc ? 2 : 3));
  return 4 + (((int)ca | (int)cb << 1 | (int)cc << 2) << 3);
}

}  // namespace

// the first maximum of the levels taken, or the zero slope (select_d)
struct Best {
  double v = 0.0;
  int idx = -1;
  __device__ __forceinline__ void take(int l, double x) {
    if (!isnan(x) && (idx < 0 || x > v)) { idx = l; v = x; }
  }
  __device__ __forceinline__ int option() const { return idx < 0 || 0.0 > v ? 3 : idx; }
};
// The reference's selection among the levels `need` of the cells cm, c, cp.
// Where the three are the same, levels 0 and 1 have the same two faces.
__device__ __forceinline__ int formula(int need, const double (&cm)[6], const double (&c)[6], const double (&cp)[6]) {
  unsigned long long diff = 0;
#pragma unroll
  for (int q = 0; q < 6; q++) {
    const unsigned long long x = __builtin_bit_cast(unsigned long long, c[q]);
    diff |= (x ^ __builtin_bit_cast(unsigned long long, cm[q])) | (x ^ __builtin_bit_cast(unsigned long long, cp[q]));
  }
  if (diff == 0 && (need & 1)) need &= ~2;
  Best best;
#pragma unroll 1
  for (int l = 0; l < 3; l++) {
    if (!(need >> l & 1)) continue;
    double ap[6], an[6];
#pragma unroll
    for (int q = 0; q < 6; q++) {
      ap[q] = cand_p(l, cm[q], c[q], cp[q]);
      an[q] = cand_n(l, cm[q], c[q], cp[q]);
    }
    best.take(l, minval2_d(vieta_d(ap), vieta_d(an)));
  }
  return best.option();
}

// A block holds 256 consecutive cells (whole x-rows where XS: nx <= 256) and
// walks KC planes (KC > 1: planes of at least 256 cells).  The midpoint of a
// face is Cn_0 of the cell before it and Cp_1 of the cell behind, bit for bit:
// along x it comes through LDS from the neighbour, along z from the plane before
// in registers.
template <int KC, bool XS>
__global__ __launch_bounds__(256, 3) void k_select(Grid g, const double* __restrict__ C, uint8_t* __restrict__ sel) {
  __shared__ Lam s_mid[2][256];
  __shared__ unsigned s_list[3 * 256 * KC];   // cell | axis << 10 | levels << 12
  __shared__ unsigned s_sel[64 * KC];
  __shared__ unsigned s_cnt;
  const int t = threadIdx.x;
  if (t == 0) s_cnt = 0u;
  const long n = g.n, xb = xcd_block();
  const int plane = g.nx * g.ny;
  long m0 = xb * 256;
  if (KC > 1) m0 = (xb / (g.nz / KC)) * 256 + (xb % (g.nz / KC)) * (long)KC * plane;
  const bool on = m0 + t < n;                 // (grids of 64 and 128 cells)
  long m = on ? m0 + t : n - 1;
  int i, j, k;
  cell_ijk(g, m, i, j, k);
  // neighbours as signed offsets; at a wall the wrapped row is replaced
  auto step = [](int a, int d, int len, long stride) { return (long)(((a + d) & (len - 1)) - a) * stride; };
  const long xm = step(i, -1, g.nx, 1), xp = step(i, 1, g.nx, 1);
  const long ym = step(j, -1, g.ny, g.nx), yp = step(j, 1, g.ny, g.nx);
  const bool ylo = g.walls && j == 0, yhi = g.walls && j == g.ny - 1;
  const int tl = (t & ~(g.nx - 1)) | ((i - 1) & (g.nx - 1));   // XS: the thread of the cell before
  auto get = [&](double (&v)[6], long e) {
#pragma unroll
    for (int q = 0; q < 6; q++) v[q] = C[q * n + e];
  };
  auto record = [&](int d, int cell, int what, unsigned& byte) {
    const bool open = what >= 4 && on;
    if (!(what & 4)) byte |= (unsigned)what << (2 * d);
    const unsigned long long ball = __ballot(open);
    if (ball == 0ull) return;
    const int lane = t & 63;
    unsigned base = 0;
    if (lane == __builtin_ctzll(ball)) base = atomicAdd(&s_cnt, (unsigned)__popcll(ball));
    base = __shfl(base, __builtin_ctzll(ball));
    if (open) s_list[base + (unsigned)__popcll(ball & ((1ull << lane) - 1ull))] = (unsigned)(cell | d << 10 | (what >> 3) << 12);
  };
  double z[3][6];
  get(z[0], m + step(k, -1, g.nz, plane));
  get(z[1], m);
  Lam below = lowest_face(false, 1, z);
  __syncthreads();
#pragma unroll 1
  for (int kk = 0; kk < KC; kk++) {
    const int cell = kk * 256 + t;
    unsigned byte = 0;
    get(z[2], m + step(k + kk, 1, g.nz, plane));
    Lam x0, x1, x2;
    {
      double x[3][6];
      get(x[0], m + xm);
      get(x[2], m + xp);
#pragma unroll
      for (int q = 0; q < 6; q++) x[1][q] = z[1][q];
      const Lam mid = lowest_face(true, 0, x);
      if (XS) s_mid[kk & 1][t] = mid;
      x0 = level(lowest_face(false, 0, x), mid);
      x1 = lowest_face(true, 1, x);
      if (!XS) x1 = level(lowest_face(false, 1, x), x1);
      x2 = level(lowest_face(false, 2, x), lowest_face(true, 2, x));
    }
    {
      const Lam mid = lowest_face(true, 0, z);
      const Lam z0 = level(lowest_face(false, 0, z), mid), z1 = level(below, lowest_face(true, 1, z)),
                z2 = level(lowest_face(false, 2, z), lowest_face(true, 2, z));
      record(2, cell, decide(z0, z1, z2), byte);
      below = mid;
    }
    {
      double y[3][6];
      get(y[0], m + ym);
      get(y[2], m + yp);
#pragma unroll
      for (int q = 0; q < 6; q++) {
        y[1][q] = z[1][q];
        if (ylo) y[0][q] = 2.0 * y[1][q] - y[2][q];   // C_kabe
        if (yhi) y[2][q] = 2.0 * y[1][q] - y[0][q];
      }
      const Lam y0 = level(lowest_face(false, 0, y), lowest_face(true, 0, y)),
                y1 = level(lowest_face(false, 1, y), lowest_face(true, 1, y)),
                y2 = level(lowest_face(false, 2, y), lowest_face(true, 2, y));
      record(1, cell, decide(y0, y1, y2), byte);
    }
    if (XS) {
      __syncthreads();
      x1 = level(s_mid[kk & 1][tl], x1);
    }
    record(0, cell, decide(x0, x1, x2), byte);
    ((uint8_t*)s_sel)[cell] = (uint8_t)byte;
#pragma unroll
    for (int q = 0; q < 6; q++) {
      z[0][q] = z[1][q];
      z[1][q] = z[2][q];
    }
    m += plane;
  }
  __syncthreads();
  const unsigned cnt = s_cnt;
  // the cells of a pair and its place in the block
  auto pair_cells = [&](unsigned what, double (&cm)[6], double (&c)[6], double (&cp)[6]) {
    const int cell = (int)(what & 1023u), d = (int)(what >> 10 & 3u);
    const long mc = m0 + (cell & 255) + (long)(cell >> 8) * plane;
    int ci, cj, ck;
    cell_ijk(g, mc, ci, cj, ck);
#pragma unroll
    for (int q = 0; q < 6; q++) {
      const double* Cq = C + q * n;
      cm[q] = ldb(Cq, g, ci - (d == 0), cj - (d == 1), ck - (d == 2), BC_C);
      c[q] = Cq[mc];
      cp[q] = ldb(Cq, g, ci + (d == 0), cj + (d == 1), ck + (d == 2), BC_C);
    }
  };
  auto settle = [&](unsigned what, unsigned idx) {
    const int cell = (int)(what & 1023u), d = (int)(what >> 10 & 3u);
    atomicOr(&s_sel[cell >> 2], idx << (8 * (cell & 3) + 2 * d));
  };
  if (cnt <= 42) {
    // a short list: a lane per pair and face, one formula's latency instead of
    // that of all its faces.  (A long one would idle the lanes of the faces
    // that are not needed.)
    double* res = (double*)s_mid;
    const unsigned e = t / 6, l = t % 6 >> 1;
    if (e < cnt) {
      const unsigned what = s_list[e];
      if (what >> (12 + l) & 1u) {
        double cm[6], c[6], cp[6], a[6];
        pair_cells(what, cm, c, cp);
#pragma unroll
        for (int q = 0; q < 6; q++) a[q] = t & 1 ? cand_n(l, cm[q], c[q], cp[q]) : cand_p(l, cm[q], c[q], cp[q]);
        res[t] = vieta_d(a);
      }
    }
    __syncthreads();
    if ((unsigned)t < cnt) {
      Best best;
      for (int q = 0; q < 3; q++)
        if (s_list[t] >> (12 + q) & 1u) best.take(q, minval2_d(res[6 * t + 2 * q], res[6 * t + 2 * q + 1]));
      settle(s_list[t], best.option());
    }
  } else {
    for (unsigned e = t; e < cnt; e += 256) {
      const unsigned what = s_list[e];
      double cm[6], c[6], cp[6];
      pair_cells(what, cm, c, cp);
      settle(what, (unsigned)formula((int)(what >> 12), cm, c, cp));
    }
  }
  __syncthreads();
  const int words = (int)std::min<long>(64, (n - m0) >> 2);
  if (t < 64 * KC && (t & 63) < words) ((unsigned*)(sel + m0 + (long)(t >> 6) * plane))[t & 63] = s_sel[t];
}

void f64_select(Ctx& c) {
  const Grid& g = c.g;
  // as many planes a block, up to four, as leave eight blocks a CU: the midpoint
  // handed along z saves one evaluation in 17, an idle SIMD costs more
  int kc = g.nx <= 256 && g.nx * g.ny >= 256 ? 4 : 1;   // (nz is a power of two, at least 4)
  while (kc > 1 && g.n / (256 * kc) < 2048) kc >>= 1;
  auto k = g.nx > 256 ? k_select<1, false> : kc == 4 ? k_select<4, true> : kc == 2 ? k_select<2, true> : k_select<1, true>;
  const long blocks = std::max<long>(1, g.n / (256 * kc));
  hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(256), 0, c.stream, g, c.C[c.cur], c.sel);
}

}  // namespace fp
