// FP64 spectral solves of the parity path: the Crank-Nicolson Helmholtz
// problems of the three velocity components (fft_navier, fenep.f90:1430-1527;
// fft_*_kabe, fenep_2d.f90:1179-1342) and the pressure Poisson equation
// (fft_poisson, fenep.f90:1529-1560; fft_poisson_kabe and tdma,
// fenep_2d.f90:1145-1342).  Compiled with -ffp-contract=off; fused
// multiply-adds appear only where they are written out (quot, quot_finite).
// The quotients of spectrum values are quot_finite's: an infinity on the grid
// is NaN in every spectrum value.
//
// The transforms are radix-2 decimations in frequency: the butterflies, their
// twiddles and their operand order are those of the CPU restatement's Stockham
// form, so every spectrum value has its bits; only the places differ.  They
// run in place in LDS, up to three radix-2 stages per pass with the eight
// elements in registers, and leave their output bit-reversed; the inverse
// reads the bit-reversed order back, so no pass permutes anything.
//
// The half spectrum is stored [component][kx][z][y] (y fastest): an x
// transform of `nl` consecutive (y, z) lines stores runs of nl values, and a
// kx slab is contiguous.  After the z (and y) transforms the row of
// wavenumber m is row bitrev(m).
//
// Three launches serve the three Helmholtz problems and three the Poisson
// equation (its right-hand side formed in the x transform) where a kx slab
// fits in LDS, five otherwise.  Before: five per component (x, y, z with the
// division, y, x), 20 of the step's 24 launches.  Small grids are bound by those
// launches: the Newtonian 32^3 step took 127 us and takes 49, the FENE-P step
// at 64^3 340 and 228 us.  At 256 x 128 x 128 between walls the four solves
// went from 1.16 to 0.43 ms; there the line solves' serial recurrence and the
// LDS passes bound them.
#include "fp_fft.h"
#include <algorithm>
#include <cmath>

namespace fp {

namespace {

// divides a spectrum value by N and the operator of the periodic problem
// (fenep.f90:1458-1462, 1540-1548): kinds 0-2 Helmholtz, 3 Poisson.  N is a
// power of two: its reciprocal multiplies exactly.
struct Divide {
  int kind;
  double coef, rn;
  __device__ __forceinline__ double2 operator()(double k2, double2 s) const {
    const double lhs = kind == 3 ? -k2 : 1.0 + coef * k2;
    if (fabs(lhs) < 1.0e-16) return make_double2(0.0, 0.0);
    const double y = 1.0 / lhs;
    return make_double2(quot_finite(s.x * rn, lhs, y), quot_finite(s.y * rn, lhs, y));
  }
};

}  // namespace

// ------------------------------------------------------------- x transforms
// Real x-lines -> half spectrum, 2^lnl consecutive (y, z) lines per block and
// component comp + blockIdx.y.  The line values: Plain: q, one plane per
// component; Div: the divergence of u* / dt (the Poisson right-hand side,
// fenep.f90:1550-1552) of the planes u, v, w; Regular: the velocity u, v, w less
// the mean um (nullptr: none) at the cell centres.
enum class Line { Plain, Div, Regular };
template <typename T>
struct LineSrc {
  const T *u, *v, *w;
  const double* um;
};
template <int M, Line S, bool WL, typename T>
__global__ __launch_bounds__(256) void k_x_forward(Grid g, LineSrc<T> q, int comp, double2* __restrict__ spec,
                                                   const double2* __restrict__ tw, int lnl) {
  extern __shared__ double2 lds[];
  const int n = g.nx, L = g.lnx, nl = 1 << lnl, pitch = n + 1;
  double2* tws = lds + nl * pitch;
  const long plane = (long)g.ny * g.nz, l0 = (long)blockIdx.x << lnl;
  comp += blockIdx.y;
  load_tw(tws, tw, n);
  const double iy[4] = {1.0 / g.dx, 1.0 / g.dy, 1.0 / g.dz, 1.0 / g.dt};
  auto value = [&](int e) {
    const int l = e >> L, i = e & (n - 1);
    const long m = (l0 + l) * n + i;
    double v;
    int ii, j, k;
    cell_ijk(g, m, ii, j, k);
    if constexpr (S == Line::Plain) {
      v = q.u[comp * g.n + m];
    } else if constexpr (S == Line::Div) {
      v = quot((quot(-ldbw<WL>(q.u, g, i - 1, j, k, BC_U) + ldbw<WL>(q.u, g, i, j, k, BC_U), g.dx, iy[0])
                + quot(-ldbw<WL>(q.v, g, i, j - 1, k, BC_V) + ldbw<WL>(q.v, g, i, j, k, BC_V), g.dy, iy[1]))
               + quot(-ldbw<WL>(q.w, g, i, j, k - 1, BC_W) + ldbw<WL>(q.w, g, i, j, k, BC_W), g.dz, iy[2]), g.dt, iy[3]);
    } else {
      const T* f = comp == 0 ? q.u : (comp == 1 ? q.v : q.w);
      const int a = comp == 0, b = comp == 1, c = comp == 2;
      double x = (double)f[m], y = (double)ldbw<WL>(f, g, i - a, j - b, k - c, BC_U + comp);
      if (q.um) {
        const double* mean = q.um + comp * g.n;
        x = x - mean[m];
        y = y - ldbw<WL>(mean, g, i - a, j - b, k - c, BC_U + comp);
      }
      v = (x + y) / 2.0;
    }
    return v;
  };
  copy_ahead<S == Line::Plain ? 4 : 2, double>(nl << L, value, [&](int e, double v) {
    lds[(e >> L) * pitch + (e & (n - 1))] = make_double2(v, 0.0);
  });
  __syncthreads();
  const Lines<double2> f{lds, 1, pitch, lnl, L};
  dif_from_natural<M, false>(f, tws);
  double2* out = spec + blockIdx.y * (plane * g.nxh) + l0;
  for (int e = threadIdx.x; e < g.nxh << lnl; e += blockDim.x) {
    const int l = e & (nl - 1), i = e >> lnl;
    out[plane * i + l] = lds[l * pitch + brev(i, L)];
  }
}

// half spectrum -> real x-lines
template <int M>
__global__ __launch_bounds__(256) void k_x_inverse(Grid g, const double2* __restrict__ spec, double* __restrict__ out,
                                                   const double2* __restrict__ tw, int lnl) {
  extern __shared__ double2 lds[];
  const int n = g.nx, L = g.lnx, nl = 1 << lnl, pitch = n + 1, h = n / 2;
  double2* tws = lds + nl * pitch;
  const long plane = (long)g.ny * g.nz, l0 = (long)blockIdx.x << lnl;
  load_tw(tws, tw, n);
  const double2* in = spec + blockIdx.y * (plane * g.nxh) + l0;
  copy_ahead<4, double2>(g.nxh << lnl, [&](int e) { return in[plane * (e >> lnl) + (e & (nl - 1))]; },
                         [&](int e, double2 v) {
                           const int l = e & (nl - 1), i = e >> lnl;
                           if (i == 0 || i == h) v.y = 0.0;
                           lds[l * pitch + i] = v;
                           if (i > 0 && i < h) lds[l * pitch + (n - i)] = make_double2(v.x, -v.y);
                         });
  __syncthreads();
  const Lines<double2> f{lds, 1, pitch, lnl, L};
  dif_from_natural<M, true>(f, tws);
  double* o = out + blockIdx.y * g.n + l0 * n;
  for (int e = threadIdx.x; e < nl << L; e += blockDim.x) o[e] = lds[(e >> L) * pitch + brev(e & (n - 1), L)].x;
}

// -------------------------------------------------------- line solve in y
// Tridiagonal line solve along y of one (kx, kz) mode, between walls (tdma
// with the wall rows of fft_*_kabe, fenep_2d.f90:1145-1177, 1222-1331), in the
// reference's order.  Rows: 0 and ny+1 the ghosts, 1..ny the cells; the
// right-hand side of the ghost rows is zero and their solution is not needed,
// so only the cells are stored.  The pivots 1/den depend on the mode and the
// kind alone and come from a table (k_line_pivots); the recurrence for P
// follows from them with multiplies.  re and im are independent: one lane
// each.
struct LineRow {
  int kind, ny;
  double diag, off;   // the interior rows' coefficients
  __device__ __forceinline__ LineRow(const Grid& g, int kd, double k2) : kind(kd), ny(g.ny) {
    const double coef = ((g.dt * g.beta) / g.re) / 2.0, idy2 = g.dy * g.dy;
    if (kd == 3) { diag = -(k2 + 2.0 / idy2); off = 1.0 / idy2; }
    else { diag = 1.0 + coef * (k2 + 2.0 / idy2); off = -(coef / idy2); }
  }
  // P of the ghost row below; a, b, c of row r >= 1
  __device__ __forceinline__ double first() const { return kind == 3 ? 1.0 : (kind == 1 ? -0.0 : -1.0); }
  __device__ __forceinline__ void row(int r, double& a, double& b, double& c, bool& rhs) const {
    const bool inner = r <= ny - (kind == 1 ? 1 : 0);
    rhs = inner;
    a = inner ? diag : 1.0;
    b = inner ? off : 0.0;
    c = inner ? off : (kind == 3 ? -1.0 : (kind == 1 ? 0.0 : 1.0));
  }
};

// table[kx][r][row of kz], r = 0..ny (rows 1..ny+1 of the line): 1/den, 0 where the
// reference takes the row for singular
__global__ __launch_bounds__(256) void k_line_pivots(Grid g, int kind, const double* __restrict__ kx2,
                                                     const double* __restrict__ kz2, double* __restrict__ table) {
  const long t = blockIdx.x * 256L + threadIdx.x;
  if (t >= (long)g.nxh * g.nz) return;
  const int kr = (int)(t & (g.nz - 1)), i = (int)(t / g.nz);
  const LineRow lr(g, kind, kx2[i] + kz2[brev(kr, log2i(g.nz))]);
  double P = lr.first();
  double* o = table + (long)i * (g.ny + 1) * g.nz + kr;
  for (int r = 1; r <= g.ny + 1; r++) {
    double a, b, c;
    bool rhs;
    lr.row(r, a, b, c, rhs);
    const double den = a + c * P;
    const bool zero = fabs(den) < 1.0e-16;
    P = zero ? 0.0 : -b / den;
    o[(long)(r - 1) * g.nz] = zero ? 0.0 : 1.0 / den;
  }
}

// One lane's line: its values v[0..ny) (stride vs doubles) and its pivots
// lp[0..ny] (stride ps) in LDS; P takes a pivot's place once it is used.  TB rows
// (ny is a multiple) a batch: their values are read together, the next batch's
// while this one is computed, so that the recurrences wait on arithmetic only.
// (With the pivots read from memory 16 rows ahead and the values a row ahead,
// k_lines_y took 144 us for the three components at 256x128x128, now 110.)
template <int TB>
__device__ __forceinline__ void line_solve_by(const Grid& g, int kind, double k2, double rn, double* v, int vs, double* lp,
                                              int ps) {
  const LineRow lr(g, kind, k2);
  const int ny = g.ny;
  double P = lr.first(), Q = 0.0;
  double yn[TB], vn[TB];
#pragma unroll
  for (int u = 0; u < TB; u++) {
    yn[u] = lp[u * ps];
    vn[u] = v[u * vs];
  }
  // all but the last batch: interior rows of every kind
  const double off = lr.off, diag = lr.diag;
  int r0 = 1;
  for (; r0 + TB <= ny; r0 += TB) {
    double yc[TB], vc[TB];
#pragma unroll
    for (int u = 0; u < TB; u++) {
      yc[u] = yn[u];
      vc[u] = vn[u];
    }
#pragma unroll
    for (int u = 0; u < TB; u++) {
      yn[u] = lp[(r0 + TB - 1 + u) * ps];
      vn[u] = v[(r0 + TB - 1 + u) * vs];
    }
#pragma unroll
    for (int u = 0; u < TB; u++) {
      const double den = diag + off * P;
      Q = quot_finite(vc[u] * rn - off * Q, den, yc[u]);
      P = quot_finite(-off, den, yc[u]);
      v[(r0 - 1 + u) * vs] = Q;
      lp[(r0 - 1 + u) * ps] = P;   // both lanes of the line: the same value
    }
  }
#pragma unroll
  for (int u = 0; u < TB; u++) {
    double a, b, c;
    bool rhs;
    lr.row(r0 + u, a, b, c, rhs);
    const double d = rhs ? vn[u] * rn : 0.0;
    const double den = a + c * P;
    Q = quot_finite(d - c * Q, den, yn[u]);
    P = quot_finite(-b, den, yn[u]);
    v[(r0 - 1 + u) * vs] = Q;
    lp[(r0 - 1 + u) * ps] = P;
  }
  {
    double a, b, c;
    bool rhs;
    lr.row(ny + 1, a, b, c, rhs);
    Q = quot_finite(0.0 - c * Q, a + c * P, lp[ny * ps]);
  }
  double x = Q, pn[TB], qn[TB];
#pragma unroll
  for (int u = 0; u < TB; u++) {
    pn[u] = lp[(ny - 1 - u) * ps];
    qn[u] = v[(ny - 1 - u) * vs];
  }
  for (r0 = ny; r0 >= 1; r0 -= TB) {
    double pc[TB], qc[TB];
#pragma unroll
    for (int u = 0; u < TB; u++) {
      pc[u] = pn[u];
      qc[u] = qn[u];
    }
    if (r0 > TB) {
#pragma unroll
      for (int u = 0; u < TB; u++) {
        pn[u] = lp[(r0 - TB - 1 - u) * ps];
        qn[u] = v[(r0 - TB - 1 - u) * vs];
      }
    }
#pragma unroll
    for (int u = 0; u < TB; u++) {
      x = pc[u] * x + qc[u];
      v[(r0 - 1 - u) * vs] = x;
    }
  }
}
__device__ __forceinline__ void line_solve(const Grid& g, int kind, double k2, double rn, double* v, int vs, double* lp,
                                           int ps) {
  if (g.ny >= 8) line_solve_by<8>(g, kind, k2, rn, v, vs, lp, ps);
  else line_solve_by<4>(g, kind, k2, rn, v, vs, lp, ps);
}

// Line solves of 2^ltl consecutive kz rows of one kx and component per block,
// the lines staged through LDS with coalesced copies.  Bound by the serial
// recurrence of a line: 16 lines per block keep three blocks on a CU.
__global__ __launch_bounds__(128) void k_lines_y(Grid g, double2* __restrict__ spec, int kind0, double rn,
                                                 const double* __restrict__ table, long tstride, const double* __restrict__ kx2,
                                                 const double* __restrict__ kz2, int ltl) {
  extern __shared__ double2 lds[];
  const int ny = g.ny, tl = 1 << ltl, pitch = ny + 1;
  double* lp = (double*)(lds + tl * pitch);   // pivots, then P, [row][line]
  const int kind = kind0 + blockIdx.y;
  const long b0 = (long)blockIdx.x << ltl;    // first (kx, kz row) line
  const int i = (int)(b0 / g.nz), kr0 = (int)(b0 & (g.nz - 1));
  double2* base = spec + blockIdx.y * ((long)g.nxh * ny * g.nz) + b0 * ny;
  const double* y = table + (kind == 1 ? tstride : (kind == 3 ? 2 * tstride : 0)) + (long)i * (ny + 1) * g.nz + kr0;
  copy_ahead<8, double>((ny + 1) << ltl, [&](int e) { return y[(e >> ltl) * (long)g.nz + (e & (tl - 1))]; },
                        [&](int e, double v) { lp[e] = v; });
  copy_ahead<8, double2>(tl << g.lny, [&](int e) { return base[e]; },
                         [&](int e, double2 v) { lds[(e >> g.lny) * pitch + (e & (ny - 1))] = v; });
  __syncthreads();
  if (threadIdx.x < 2 * tl) {
    const int l = threadIdx.x >> 1, c = threadIdx.x & 1, kr = kr0 + l;
    line_solve(g, kind, kx2[i] + kz2[brev(kr, log2i(g.nz))], rn, (double*)(lds + l * pitch) + c, 2, lp + l, tl);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < tl << g.lny; e += blockDim.x) base[e] = lds[(e >> g.lny) * pitch + (e & (ny - 1))];
}

// ------------------------------------------------------------ one kx slab
// Everything between the x transforms for one kx and component, the [z][y]
// slab in LDS: periodic, the y and z transforms, the division and back;
// between walls, the z transforms around the line solves.  Taken where the
// slab fits in the LDS of a CU.
template <int M, bool WL>
__global__ __launch_bounds__(1024) void k_slab(Grid g, double2* __restrict__ spec, int kind0, double rn,
                                               const double2* __restrict__ twy, const double2* __restrict__ twz,
                                               const double* __restrict__ kx2, const double* __restrict__ ky2,
                                               const double* __restrict__ kz2, const double* __restrict__ table,
                                               long tstride) {
  extern __shared__ double2 lds[];
  const int ny = g.ny, nz = g.nz, pitch = ny + 1, lnz = log2i(nz);
  double2* tz = lds + nz * pitch;
  double2* ty = tz + nz / 2;                  // periodic
  double* lp = (double*)ty;                   // between walls: pivots, then P, [row][kz]
  const int i = blockIdx.x, kind = kind0 + blockIdx.y;
  double2* base = spec + (blockIdx.y * (long)g.nxh + i) * ((long)ny * nz);
  load_tw(tz, twz, nz);
  if (!WL) load_tw(ty, twy, ny);
  copy_ahead<4, double2>(ny * nz, [&](int e) { return base[e]; },
                         [&](int e, double2 v) { lds[(e >> g.lny) * pitch + (e & (ny - 1))] = v; });
  __syncthreads();
  const Lines<double2> fy{lds, 1, pitch, lnz, g.lny}, fz{lds, pitch, 1, g.lny, lnz};
  if constexpr (!WL) {
    dif_from_natural<M, false>(fy, ty);
    dif_from_natural<M, false>(fz, tz, false);
    const Divide dv{kind, ((g.dt * g.beta) / g.re) / 2.0, rn};
    const double kx = kx2[i];
    turn<M>(fz, tz, [&](int l, int kz, double2 s) { return dv((kx + ky2[brev(l, g.lny)]) + kz2[kz], s); });
    dif_from_reversed<M>(fz, tz, false);
    dif_from_reversed<M>(fy, ty);
  } else {
    const double* y = table + (kind == 1 ? tstride : (kind == 3 ? 2 * tstride : 0)) + (long)i * (ny + 1) * nz;
    copy_ahead<4, double>((ny + 1) * nz, [&](int e) { return y[e]; }, [&](int e, double v) { lp[e] = v; });
    dif_from_natural<M, false>(fz, tz);
    for (int t = threadIdx.x; t < 2 * nz; t += blockDim.x) {
      const int kr = t >> 1, c = t & 1;
      line_solve(g, kind, kx2[i] + kz2[brev(kr, lnz)], rn, (double*)(lds + kr * pitch) + c, 2, lp + kr, nz);
    }
    __syncthreads();
    dif_from_reversed<M>(fz, tz);
  }
  for (int e = threadIdx.x; e < ny * nz; e += blockDim.x) base[e] = lds[(e >> g.lny) * pitch + (e & (ny - 1))];
}

// ---------------------------------------- y and z transforms of larger grids
// y: 2^lnl consecutive contiguous lines per block (inv: bit-reversed in)
template <int M>
__global__ __launch_bounds__(256) void k_y_lines(Grid g, double2* __restrict__ spec, const double2* __restrict__ tw, int inv,
                                                 int lnl) {
  extern __shared__ double2 lds[];
  const int n = g.ny, nl = 1 << lnl, pitch = n + 1;
  double2* tws = lds + nl * pitch;
  double2* base = spec + blockIdx.y * ((long)g.nxh * n * g.nz) + ((long)blockIdx.x << (lnl + g.lny));
  load_tw(tws, tw, n);
  copy_ahead<4, double2>(nl << g.lny, [&](int e) { return base[e]; },
                         [&](int e, double2 v) { lds[(e >> g.lny) * pitch + (e & (n - 1))] = v; });
  __syncthreads();
  const Lines<double2> f{lds, 1, pitch, lnl, g.lny};
  if (inv) dif_from_reversed<M>(f, tws);
  else dif_from_natural<M, false>(f, tws);
  for (int e = threadIdx.x; e < nl << g.lny; e += blockDim.x) base[e] = lds[(e >> g.lny) * pitch + (e & (n - 1))];
}

// z: 2^lnl consecutive y columns of one kx.  mode 0 forward, 1 inverse
// (bit-reversed in), 2 forward, the periodic division, inverse
template <int M>
__global__ __launch_bounds__(256) void k_z_lines(Grid g, double2* __restrict__ spec, const double2* __restrict__ tw, int mode,
                                                 int kind0, double rn, int lnl, const double* __restrict__ kx2,
                                                 const double* __restrict__ ky2, const double* __restrict__ kz2) {
  extern __shared__ double2 lds[];
  const int n = g.nz, nl = 1 << lnl, L = log2i(n);
  double2* tws = lds + (n << lnl);
  const int lt = g.lny - lnl;                 // log2 of the tiles per kx
  const int i = blockIdx.x >> lt, j0 = (blockIdx.x & ((1 << lt) - 1)) << lnl;
  double2* base = spec + (blockIdx.y * (long)g.nxh + i) * ((long)g.ny * n) + j0;
  load_tw(tws, tw, n);
  copy_ahead<4, double2>(n << lnl, [&](int e) { return base[((long)(e >> lnl) << g.lny) + (e & (nl - 1))]; },
                         [&](int e, double2 v) { lds[e] = v; });
  __syncthreads();
  const Lines<double2> f{lds, nl, 1, lnl, L};
  if (mode == 0) {
    dif_from_natural<M, false>(f, tws);
  } else if (mode == 1) {
    dif_from_reversed<M>(f, tws);
  } else {
    dif_from_natural<M, false>(f, tws, false);
    const Divide dv{kind0 + (int)blockIdx.y, ((g.dt * g.beta) / g.re) / 2.0, rn};
    const double kx = kx2[i];
    turn<M>(f, tws, [&](int l, int kz, double2 s) { return dv((kx + ky2[brev(j0 + l, g.lny)]) + kz2[kz], s); });
    dif_from_reversed<M>(f, tws, false);
  }
  for (int e = threadIdx.x; e < n << lnl; e += blockDim.x) base[((long)(e >> lnl) << g.lny) + (e & (nl - 1))] = lds[e];
}

// -------------------------------------------------------------------- host
namespace {

size_t lds_slab64(const Grid& g) {
  size_t w = sizeof(double2) * ((size_t)g.nz * (g.ny + 1) + g.nz / 2);
  return w + (g.walls ? sizeof(double) * (size_t)(g.ny + 1) * g.nz : sizeof(double2) * (g.ny / 2));
}
constexpr int LNL_Y = 4;   // lines per block of k_lines_y (log2)
size_t lds_lines_y(int ny, int ltl) { return (sizeof(double2) + sizeof(double)) * (ny + 1) << ltl; }

template <typename F>
void allow_lds(F* f, int bytes) {
  FP_HIP_CHECK(hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
}

int lnl_lines_y(const Grid& g) {
  int l = std::min(LNL_Y, lg(g.nz));
  while (l > 0 && lds_lines_y(g.ny, l) > 64 * 1024) l--;
  return l;
}

// words of one kind's table of pivots
long piv_words(const Grid& g) { return (long)g.nxh * (g.ny + 1) * g.nz; }
void line_pivots(Ctx& c) {
  const Grid& g = c.g;
  const long stride = piv_words(g);
  const int kinds[3] = {0, 1, 3};   // U and W share a table
  for (int t = 0; t < 3; t++)
    hipLaunchKernelGGL(k_line_pivots, dim3((unsigned)(((long)g.nxh * g.nz + 255) / 256)), dim3(256), 0, c.stream, g, kinds[t],
                       c.kx2, c.kz2, c.piv + t * stride);
  c.piv_beta = g.beta;
}

// Stages per pass: two where the launch has few points per CU (a pass of
// three would leave SIMDs without a thread), three above.
int stages_per_pass(const Grid& g, int comps) { return g.n * comps <= (1L << 20) ? 2 : 3; }
int threads_for(long points, int M) { return (int)std::max(64L, std::min(256L, points >> M)); }

// the transforms along one axis of `comps` components
template <Line S, bool WL, typename T>
void x_forward(Ctx& c, int comp, int comps, const LineSrc<T>& q) {
  const Grid& g = c.g;
  const long lines = (long)g.ny * g.nz;
  const int lx = lines_log2(g.nx, lines, comps), M = stages_per_pass(g, comps);
  auto k = M == 2 ? k_x_forward<2, S, WL, T> : k_x_forward<3, S, WL, T>;
  if (lds_lines(g.nx, lx) > 65536) allow_lds(k, (int)lds_lines(g.nx, lx));
  hipLaunchKernelGGL(k, dim3((unsigned)(lines >> lx), comps), dim3(threads_for((long)g.nx << lx, M)), lds_lines(g.nx, lx),
                     c.stream, g, q, comp, c.spec, c.twx, lx);
}
void x_inverse(Ctx& c, int comps, double* x) {
  const Grid& g = c.g;
  const long lines = (long)g.ny * g.nz;
  const int lx = lines_log2(g.nx, lines, comps), M = stages_per_pass(g, comps);
  hipLaunchKernelGGL(M == 2 ? k_x_inverse<2> : k_x_inverse<3>, dim3((unsigned)(lines >> lx), comps),
                     dim3(threads_for((long)g.nx << lx, M)), lds_lines(g.nx, lx), c.stream, g, c.spec, x, c.twx, lx);
}
void y_lines(Ctx& c, int comps, int inv) {
  const Grid& g = c.g;
  // (the lines of a block share their kx)
  const int l = std::min(lines_log2(g.ny, (long)g.nxh * g.nz, comps), lg(g.nz)), M = stages_per_pass(g, comps);
  hipLaunchKernelGGL(M == 2 ? k_y_lines<2> : k_y_lines<3>, dim3((unsigned)((long)g.nxh * g.nz >> l), comps),
                     dim3(threads_for((long)g.ny << l, M)), lds_lines(g.ny, l), c.stream, g, c.spec, c.twy, inv, l);
}
void z_lines(Ctx& c, int comps, int mode, int kind0, double rn) {
  const Grid& g = c.g;
  const int l = std::min(lines_log2(g.nz, (long)g.nxh * g.ny, comps), g.lny), M = stages_per_pass(g, comps);
  hipLaunchKernelGGL(M == 2 ? k_z_lines<2> : k_z_lines<3>, dim3((unsigned)((long)g.nxh * g.ny >> l), comps),
                     dim3(threads_for((long)g.nz << l, M)), sizeof(double2) * (((size_t)g.nz << l) + g.nz / 2), c.stream, g, c.spec,
                     c.twz, mode, kind0, rn, l, c.kx2, c.ky2, c.kz2);
}

// the solves of `comps` components, kinds kind0, kind0 + 1, ..., at once
void solve(Ctx& c, int kind0, int comps, const double* q, double* x, bool div) {
  const Grid& g = c.g;
  hipStream_t s = c.stream;
  const LineSrc<double> src{q, q + g.n, q + 2 * g.n, nullptr};
  if (!div) x_forward<Line::Plain, false>(c, 0, comps, src);
  else if (g.walls) x_forward<Line::Div, true>(c, 0, comps, src);
  else x_forward<Line::Div, false>(c, 0, comps, src);
  const double rn = 1.0 / (double)(g.walls ? (long)g.nx * g.nz : g.n);
  const long tstride = piv_words(g);
  if (g.walls && c.piv_beta != g.beta) line_pivots(c);
  if (c.slab64) {
    const int threads = std::max(64, std::min(1024, g.ny * g.nz / 4));
    // three stages a pass where both axes divide into them: 64^3's step of 80 us
    // is 2 us shorter, elsewhere two and three measure the same
    const bool three = g.lny % 3 == 0 && lg(g.nz) % 3 == 0;
    auto slab = g.walls ? k_slab<2, true> : (three ? k_slab<3, false> : k_slab<2, false>);
    hipLaunchKernelGGL(slab, dim3(g.nxh, comps), dim3(threads), lds_slab64(g), s, g,
                       c.spec, kind0, rn, c.twy, c.twz, c.kx2, c.ky2, c.kz2, c.piv, tstride);
  } else if (!g.walls) {
    y_lines(c, comps, 0);
    z_lines(c, comps, 2, kind0, rn);
    y_lines(c, comps, 1);
  } else {
    const int lt = lnl_lines_y(g);
    z_lines(c, comps, 0, kind0, rn);
    hipLaunchKernelGGL(k_lines_y, dim3((unsigned)((long)g.nxh * g.nz >> lt), comps), dim3(128), lds_lines_y(g.ny, lt), s, g,
                       c.spec, kind0, rn, c.piv, tstride, c.kx2, c.kz2, lt);
    z_lines(c, comps, 1, kind0, rn);
  }
  x_inverse(c, comps, x);
}

}  // namespace

// The spectrum holds three components where that is small beside the state
// (their solves then share launches); one above it, where a component alone
// fills the device, and in a mixed context, whose step makes no FP64 solve
// (its shell spectrum goes a component at a time) until it records for the
// adjoint.
static int solve_components(const Grid& g) { return (size_t)g.nxh * g.ny * g.nz <= ((size_t)1 << 24) ? 3 : 1; }
static size_t spectrum_bytes(const Grid& g, int comps) { return sizeof(double2) * (size_t)g.nxh * g.ny * g.nz * comps; }

void f64_spectral_reserve(Ctx& c) {
  const int comps = solve_components(c.g);
  if (c.nspec >= comps) return;
  double2* more = nullptr;
  if (hipMalloc((void**)&more, spectrum_bytes(c.g, comps)) != hipSuccess) {
    (void)hipGetLastError();   // the solves go on one component at a time
    return;
  }
  FP_HIP_CHECK(hipStreamSynchronize(c.stream));
  (void)hipFree(c.spec);
  c.spec = more;
  c.nspec = comps;
}

void f64_spectral_create(Ctx& c) {
  const Grid& g = c.g;
  c.nspec = c.p.precision == FP_PREC_F64 ? solve_components(g) : 1;
  FP_HIP_CHECK(hipMalloc((void**)&c.spec, spectrum_bytes(g, c.nspec)));
  // the pivots' tables: only the FP64 step solves between walls; filled by
  // the first solve and when beta has changed
  if (g.walls && c.p.precision == FP_PREC_F64) FP_HIP_CHECK(hipMalloc((void**)&c.piv, sizeof(double) * 3 * piv_words(g)));
  int lds_max = 0, dev = 0;
  FP_HIP_CHECK(hipGetDevice(&dev));
  FP_HIP_CHECK(hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
  c.slab64 = lds_slab64(g) <= (size_t)lds_max;
  allow_lds(k_slab<2, false>, lds_max);
  allow_lds(k_slab<2, true>, lds_max);
  allow_lds(k_slab<3, false>, lds_max);
  allow_lds(k_x_inverse<2>, lds_max);
  allow_lds(k_x_inverse<3>, lds_max);
  allow_lds(k_y_lines<2>, lds_max);
  allow_lds(k_y_lines<3>, lds_max);
  allow_lds(k_z_lines<2>, lds_max);
  allow_lds(k_z_lines<3>, lds_max);
  allow_lds(k_lines_y, lds_max);
}

void f64_solve(Ctx& c, int kind, const double* q, double* x) { solve(c, kind, 1, q, x, false); }

// the three components' Helmholtz problems: q and x of 3 planes
void f64_helmholtz(Ctx& c, const double* q, double* x) {
  if (c.nspec == 3) {
    solve(c, 0, 3, q, x, false);
    return;
  }
  for (int comp = 0; comp < 3; comp++) solve(c, comp, 1, q + comp * c.g.n, x + comp * c.g.n, false);
}

// the Poisson equation lap_h x = div_h up / dt
void f64_poisson(Ctx& c, const double* up, double* x) { solve(c, 3, 1, up, x, true); }

// forward transforms of the regular-grid velocity (periodic grids; the
// wavenumbers m of y and z at bitrev(m))
template <typename T>
static void forward_regular(Ctx& c, const T* U, const T* V, const T* W, int comp, int comps) {
  x_forward<Line::Regular, false>(c, comp, comps, LineSrc<T>{U, V, W, c.mean_u});
  y_lines(c, comps, 0);
  z_lines(c, comps, 0, 3, 1.0);
}
void f64_forward_regular(Ctx& c, const double* U, const double* V, const double* W, int comp, int comps) {
  forward_regular(c, U, V, W, comp, comps);
}
void f64_forward_regular(Ctx& c, const float* U, const float* V, const float* W, int comp, int comps) {
  forward_regular(c, U, V, W, comp, comps);
}

}  // namespace fp
