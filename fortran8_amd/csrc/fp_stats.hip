// Diagnostics, time-series statistics and spectra of the current state.  The
// kernels read the state in its stored type (FP64, or the mixed step's FP32
// fields) and compute in FP64; a mixed state is not widened in memory first.
// Sums: registers over a thread's cells, shuffles over a wavefront, one
// partial per block and a second kernel over the partials, always in the same
// order; the shell spectrum alone adds into a block's bins with LDS atomics, so
// its last bits depend on the order in which wavefronts arrive.  Compiled with
// -ffp-contract=off.
#include "fp_fft.h"
#include "fp_mixed.h"
#include <algorithm>
#include <cmath>
#include <type_traits>

namespace fp {

namespace {

inline int nblk(long n, int t) { return (int)((n + t - 1) / t); }

// the state's fields; C: 6 planes
template <typename T>
struct Fields {
  const T *U, *V, *W, *C;
  __host__ __device__ static T zero() { return T(0); }
};
template <typename F>
void with_fields(Ctx& c, F run) {
  if (c.mixed) {
    Fields<float> f;
    mixed_fields(c, &f.U, &f.V, &f.W, &f.C);
    run(f);
  } else {
    run(Fields<double>{c.U, c.V, c.W, c.C[c.cur]});
  }
}

// walls and a subtracted mean as compile-time constants: one kernel for all
// held the loads of every kind in registers
template <typename F>
void with_kind(Ctx& c, F run) {
  using Y = std::true_type;
  using N = std::false_type;
  if (c.g.walls) { if (c.mean_u) run(Y{}, Y{}); else run(Y{}, N{}); }
  else { if (c.mean_u) run(N{}, Y{}); else run(N{}, N{}); }
}

// device workspace of `words` doubles, kept by the context (grown as needed)
double* stat_ws(Ctx& c, size_t words) {
  if (c.stat_words < words) {
    FP_HIP_CHECK(hipStreamSynchronize(c.stream));
    if (c.stat) (void)hipFree(c.stat);
    c.stat = nullptr;
    c.stat_words = 0;
    FP_HIP_CHECK(hipMalloc((void**)&c.stat, sizeof(double) * words));
    c.stat_words = words;
  }
  return c.stat;
}

// blocks of a reduction over n cells: eight a CU, each thread several cells
inline int stat_blocks(long n) { return std::min(nblk(n, 256), 2048); }

enum class Red { Sum, Max, Min };
template <Red R>
__device__ __forceinline__ double combine(double a, double b) {
  return R == Red::Sum ? a + b : (R == Red::Max ? fmax(a, b) : fmin(a, b));
}
template <Red R>
__device__ __forceinline__ double wave_red(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = combine<R>(v, __shfl_xor(v, o));
  return v;
}
// one value per block of 256 threads from a value per thread, stored by thread 0
// (sh: 4 words of the value's own)
template <Red R>
__device__ __forceinline__ void block_red(double v, double* sh) {
  v = wave_red<R>(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
}
template <Red R>
__device__ __forceinline__ double block_get(const double* sh) {
  return combine<R>(combine<R>(sh[0], sh[1]), combine<R>(sh[2], sh[3]));
}

// rows of nb partials to one value each (one block per row), out[row]
__global__ __launch_bounds__(256) void k_row_sums(const double* __restrict__ part, int nb, double* __restrict__ out) {
  __shared__ double sh[4];
  const double* row = part + (long)blockIdx.x * nb;
  double v = 0.0;
  for (int b = threadIdx.x; b < nb; b += 256) v += row[b];
  block_red<Red::Sum>(v, sh);
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = block_get<Red::Sum>(sh);
}

// spacings and their multiples with correctly rounded reciprocals (quot)
struct StatConst {
  double h[3], ih[3], h4[3], ih4[3];
};
StatConst stat_const(const Grid& g) {
  StatConst k;
  const double h[3] = {g.dx, g.dy, g.dz};
  for (int d = 0; d < 3; d++) {
    k.h[d] = h[d]; k.ih[d] = 1.0 / h[d];
    k.h4[d] = 4 * h[d]; k.ih4[d] = 1.0 / k.h4[d];
  }
  return k;
}

}  // namespace

// =============================================== time-series statistics ===
// Per-cell terms of all_time_dif / all_time_dif_map (fenep_mpi.f90:2200-2564)
// for the velocity fluctuation u' = u - u_mean (u_mean = nullptr: none, the
// 'same' records; otherwise the 'diff' records): 0-2 regular-grid u'^2,
// 3-5 squared staggered gradients of u', 6 S:S with S = D + D^T of the
// 4-point gradient of u', 7 |u|^2 on the staggered grid (raw u, the
// K_staggered term), 8 log f(C), 9 tr C.  The ghosts of u' are those of u
// minus those of the mean, each by the boundary rules.
constexpr int TS_N = 10;
template <bool WL, bool MEAN, typename T>
__device__ __forceinline__ void stat_cell(const Grid& g, const StatConst& K, const Fields<T>& f, const double* __restrict__ Um,
                                          int i, int j, int k, long m, double* s) {
  const double *Vm = Um + g.n, *Wm = Um + 2 * g.n;
  auto get = [&](const T* F, const double* M, int a, int b, int c, int kind) {
    const double v = (double)ldbw<WL>(F, g, i + a, j + b, k + c, kind);
    return MEAN ? v - ldbw<WL>(M, g, i + a, j + b, k + c, kind) : v;
  };
  auto UG = [&](int a, int b, int c) { return get(f.U, Um, a, b, c, BC_U); };
  auto VG = [&](int a, int b, int c) { return get(f.V, Vm, a, b, c, BC_V); };
  auto WG = [&](int a, int b, int c) { return get(f.W, Wm, a, b, c, BC_W); };
  const double u0 = UG(0, 0, 0), v0 = VG(0, 0, 0), w0 = WG(0, 0, 0);
  const double ur = (u0 + UG(-1, 0, 0)) / 2.0, vr = (v0 + VG(0, -1, 0)) / 2.0, wr = (w0 + WG(0, 0, -1)) / 2.0;
  s[0] = ur * ur; s[1] = vr * vr; s[2] = wr * wr;
  double D[3][3];
#define Q1(d, x) quot(x, K.h[d], K.ih[d])
#define Q4(d, x) quot(x, K.h4[d], K.ih4[d])
  D[0][0] = Q1(0, u0 - UG(-1, 0, 0));
  D[0][1] = Q4(1, UG(0, 1, 0) - UG(0, -1, 0) + UG(-1, 1, 0) - UG(-1, -1, 0));
  D[0][2] = Q4(2, UG(0, 0, 1) - UG(0, 0, -1) + UG(-1, 0, 1) - UG(-1, 0, -1));
  D[1][0] = Q4(0, VG(1, 0, 0) - VG(-1, 0, 0) + VG(1, -1, 0) - VG(-1, -1, 0));
  D[1][1] = Q1(1, v0 - VG(0, -1, 0));
  D[1][2] = Q4(2, VG(0, 0, 1) - VG(0, 0, -1) + VG(0, -1, 1) - VG(0, -1, -1));
  D[2][0] = Q4(0, WG(1, 0, 0) - WG(-1, 0, 0) + WG(1, 0, -1) - WG(-1, 0, -1));
  D[2][1] = Q4(1, WG(0, 1, 0) - WG(0, -1, 0) + WG(0, 1, -1) - WG(0, -1, -1));
  D[2][2] = Q1(2, w0 - WG(0, 0, -1));
#undef Q1
#undef Q4
  s[3] = D[0][0] * D[0][0]; s[4] = D[1][1] * D[1][1]; s[5] = D[2][2] * D[2][2];
  s[6] = 0.0;
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) { const double sab = D[a][b] + D[b][a]; s[6] += sab * sab; }
  const double u = f.U[m], v = f.V[m], w = f.W[m];
  s[7] = u * u + v * v + w * w;
  const double t = ((double)f.C[m] + (double)f.C[3 * g.n + m]) + (double)f.C[5 * g.n + m];
  const double L2 = g.lp * g.lp;
  s[8] = log((L2 - 3.0) / (L2 - t));
  s[9] = t;
}

// part[q nb + block]: the block's sums
template <bool WL, bool MEAN, typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_time_stats(Grid g, StatConst K, Fields<T> f, const double* __restrict__ Um,
                                                    double* __restrict__ part) {
  double acc[TS_N], s[TS_N];
#pragma unroll
  for (int q = 0; q < TS_N; q++) acc[q] = 0.0;
  const long nb = gridDim.x;
  for (long m = xcd_cell(); m < g.n; m += nb * 256) {
    int i, j, k;
    cell_ijk(g, m, i, j, k);
    stat_cell<WL, MEAN>(g, K, f, Um, i, j, k, m, s);
#pragma unroll
    for (int q = 0; q < TS_N; q++) acc[q] += s[q];
  }
  __shared__ double sh[TS_N][4];
#pragma unroll
  for (int q = 0; q < TS_N; q++) block_red<Red::Sum>(acc[q], sh[q]);
  __syncthreads();
  if (threadIdx.x < TS_N) part[(long)threadIdx.x * nb + blockIdx.x] = block_get<Red::Sum>(sh[threadIdx.x]);
}

// sum of (tr C - sum/n)^2, per block
template <typename T>
__global__ __launch_bounds__(256) void k_trc_var(Grid g, const T* __restrict__ C, const double* __restrict__ sum,
                                                 double* __restrict__ part) {
  const double mean = *sum / (double)g.n;
  double v = 0.0;
  for (long m = blockIdx.x * 256L + threadIdx.x; m < g.n; m += gridDim.x * 256L) {
    const double t = ((double)C[m] + (double)C[3 * g.n + m]) + (double)C[5 * g.n + m] - mean;
    v += t * t;
  }
  __shared__ double sh[4];
  block_red<Red::Sum>(v, sh);
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = block_get<Red::Sum>(sh);
}

void f64_time_stats(Ctx& c, double* out) {
  const Grid& g = c.g;
  hipStream_t s = c.stream;
  const int nb = stat_blocks(g.n);
  double* part = stat_ws(c, (size_t)(TS_N + 1) * nb + TS_N + 1);
  double* red = part + (size_t)(TS_N + 1) * nb;
  double r[TS_N + 1];
  with_fields(c, [&](auto f) {
    with_kind(c, [&](auto wl, auto mean) {
      auto k = k_time_stats<wl.value, mean.value, decltype(f.zero())>;
      hipLaunchKernelGGL(k, dim3(nb), dim3(256), 0, s, g, stat_const(g), f, c.mean_u, part);
    });
    hipLaunchKernelGGL(k_row_sums, dim3(TS_N), dim3(256), 0, s, part, nb, red);
    hipLaunchKernelGGL(k_trc_var, dim3(nb), dim3(256), 0, s, g, f.C, red + 9, part + (long)TS_N * nb);
    hipLaunchKernelGGL(k_row_sums, dim3(1), dim3(256), 0, s, part + (long)TS_N * nb, nb, red + TS_N);
  });
  FP_HIP_CHECK(hipMemcpyAsync(r, red, sizeof(r), hipMemcpyDeviceToHost, s));
  FP_HIP_CHECK(hipStreamSynchronize(s));
  const double N = (double)g.n, nu = 1.0 / c.p.re, L2 = c.p.lp * c.p.lp;
  const double urms = r[0] / N, vrms = r[1] / N, wrms = r[2] / N;
  const double all_rms = (urms + vrms + wrms) / 3.0, all_grad = (r[3] / N + r[4] / N + r[5] / N) / 3.0;
  const double eps = nu / 2.0 * r[6] / N;
  const double lambda = std::sqrt(all_rms / all_grad);
  out[0] = (double)c.step;
  out[1] = c.step * c.p.dt;
  out[2] = (urms + vrms + wrms) / 2.0;
  out[3] = r[7] / (2.0 * N);
  out[4] = lambda;
  out[5] = std::sqrt(all_rms) * lambda / nu;
  out[6] = eps;
  out[7] = std::pow(nu * nu * nu / eps, 0.25);
  out[8] = std::sqrt(nu / eps);
  out[9] = std::pow(nu * eps, 0.25);
  out[10] = 0.5 * (1.0 - c.p.beta) / c.p.re / c.p.wi * (L2 - 3.0) * r[8] / N;
  out[11] = r[9] / N;
  out[12] = std::sqrt(r[TS_N] / N);
}

// all_time_dif_map (fenep_mpi.f90:2350-2500): the per-cell terms summed over
// z for each (i, j) column, then the z variance of tr C about the column
// mean.  col[q * nx*ny + i + nx*j]: q = 0..9 as stat_cell (7 unused), q = 10 the
// sum of (tr C - column mean)^2.  A block holds 32 columns, Z threads each
// walking a part of the planes (256x128x128, mixed: one thread per column, 128
// blocks, took 1278 us; eight, with a kernel per boundary kind and four waves per
// SIMD, 87 us).
constexpr int COL_N = 11;
template <bool WL, bool MEAN, int Z, typename T>
__global__ __launch_bounds__(32 * Z) __attribute__((amdgpu_waves_per_eu(4))) void k_column_stats(Grid g, StatConst K, Fields<T> f, const double* __restrict__ Um,
                                                         double* __restrict__ col) {
  const int l = threadIdx.x & 31, z = threadIdx.x >> 5;
  const long nxy = (long)g.nx * g.ny;
  const long ij = xcd_block() * 32 + l;
  const bool valid = ij < nxy;   // (whole columns: the threads of a column agree)
  const int i = (int)(ij & (g.nx - 1)), j = (int)(ij >> g.lnx);
  const int k0 = g.nz / Z * z, k1 = k0 + g.nz / Z;
  double acc[TS_N], s[TS_N];
#pragma unroll
  for (int q = 0; q < TS_N; q++) acc[q] = 0.0;
  if (valid)
    for (int k = k0; k < k1; k++) {
      stat_cell<WL, MEAN>(g, K, f, Um, i, j, k, ij + nxy * k, s);
#pragma unroll
      for (int q = 0; q < TS_N; q++) acc[q] += s[q];
    }
  __shared__ double sh[TS_N + 1][Z][32];
#pragma unroll
  for (int q = 0; q < TS_N; q++) sh[q][z][l] = acc[q];
  __syncthreads();
  double tr = 0.0;
#pragma unroll
  for (int u = 0; u < Z; u++) tr += sh[9][u][l];
  const double mean = tr / (double)g.nz;
  double var = 0.0;
  if (valid)
    for (int k = k0; k < k1; k++) {
      const long m = ij + nxy * k;
      const double t = ((double)f.C[m] + (double)f.C[3 * g.n + m]) + (double)f.C[5 * g.n + m] - mean;
      var += t * t;
    }
  sh[TS_N][z][l] = var;
  __syncthreads();
  for (int q = z; q < COL_N; q += Z) {
    double v = 0.0;
#pragma unroll
    for (int u = 0; u < Z; u++) v += sh[q][u][l];
    if (valid) col[q * nxy + ij] = v;
  }
}

// mask(i, j) = 0 within 1.5 radii of a cylinder centre (fenep_mpi.f90:2530-2537,
// with the centres given instead of the reference's four fixed ones, and dY
// for y); part[block]: the block's sum
__global__ __launch_bounds__(256) void k_plane_mask(Grid g, int ncyl, const double* __restrict__ xy, double r2,
                                                    double* __restrict__ mask, double* __restrict__ part) {
  const long ij = blockIdx.x * 256L + threadIdx.x, nxy = (long)g.nx * g.ny;
  double v = 0.0;
  if (ij < nxy) {
    const int i = (int)(ij & (g.nx - 1)), j = (int)(ij >> g.lnx);
    v = 1.0;
    for (int c = 0; c < ncyl; c++) {
      const double dxc = (i + 0.5) * g.dx - xy[2 * c], dyc = (j + 0.5) * g.dy - xy[2 * c + 1];
      if (dxc * dxc + dyc * dyc < r2) v = 0.0;
    }
    mask[ij] = v;
  }
  __shared__ double sh[4];
  block_red<Red::Sum>(v, sh);
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = block_get<Red::Sum>(sh);
}
// the mask and its per-block sums (nblk(nxy, 256) of them) from the host's
// centres; xyd: 2 ncyl device words
static void plane_mask(Ctx& c, int ncyl, const double* xy, double diameter, double* xyd, double* mask, double* part) {
  const double r = diameter * 1.5 / 2.0;
  if (ncyl) FP_HIP_CHECK(hipMemcpyAsync(xyd, xy, sizeof(double) * 2 * ncyl, hipMemcpyHostToDevice, c.stream));
  hipLaunchKernelGGL(k_plane_mask, dim3(nblk((long)c.g.nx * c.g.ny, 256)), dim3(256), 0, c.stream, c.g, ncyl, xyd, r * r, mask,
                     part);
}

// all_time_dif_map (fenep_mpi.f90:2350-2564): the statistics of each column
// from its sums, as 18-value records (j outer, i inner: x, y, ten statistics,
// the mask, 0 x 5), and their masked sums per block, part[q gridDim.x + block].
constexpr int MAP_N = 10;
__global__ __launch_bounds__(256) void k_map_records(Grid g, const double* __restrict__ col, const double* __restrict__ mask,
                                                     double nu, double epc, double* __restrict__ map18,
                                                     double* __restrict__ part) {
  const long ij = blockIdx.x * 256L + threadIdx.x, nxy = (long)g.nx * g.ny;
  double vals[MAP_N + 1];
#pragma unroll
  for (int q = 0; q <= MAP_N; q++) vals[q] = 0.0;
  if (ij < nxy) {
    const double NZ = (double)g.nz;
    auto C_ = [&](int q) { return col[(long)q * nxy + ij]; };
    const double urms = C_(0) / NZ, vrms = C_(1) / NZ, wrms = C_(2) / NZ;
    const double all_rms = (urms + vrms + wrms) / 3.0;
    const double all_grad = (C_(3) / NZ + C_(4) / NZ + C_(5) / NZ) / 3.0;
    const double eps = nu / 2.0 * C_(6) / NZ;
    const double lam = sqrt(all_rms / all_grad);
    vals[0] = (urms + vrms + wrms) / 2.0;          // K
    vals[1] = lam;
    vals[2] = sqrt(all_rms) * lam / nu;
    vals[3] = eps;
    vals[4] = pow(nu * nu * nu / eps, 0.25);       // Kolmogorov length, time, velocity
    vals[5] = sqrt(nu / eps);
    vals[6] = pow(nu * eps, 0.25);
    vals[7] = epc * (C_(8) / NZ);                  // Ep
    vals[8] = C_(9) / NZ;                          // tr C mean, std
    vals[9] = sqrt(C_(10) / NZ);
    vals[10] = mask[ij];
    if (map18) {
      double* row = map18 + 18 * ij;
      row[0] = ((int)(ij & (g.nx - 1)) + 0.5) * g.dx;
      row[1] = ((int)(ij >> g.lnx) + 0.5) * g.dy;
#pragma unroll
      for (int q = 0; q <= MAP_N; q++) row[2 + q] = vals[q];
#pragma unroll
      for (int q = 13; q < 18; q++) row[q] = 0.0;
    }
  }
  __shared__ double sh[MAP_N][4];
#pragma unroll
  for (int q = 0; q < MAP_N; q++) block_red<Red::Sum>(ij < nxy ? vals[q] * vals[10] : 0.0, sh[q]);
  __syncthreads();
  if (threadIdx.x < MAP_N) part[(long)threadIdx.x * gridDim.x + blockIdx.x] = block_get<Red::Sum>(sh[threadIdx.x]);
}

int f64_time_stats_map(Ctx& c, int ncyl, const double* xy, double diameter, double* map18, double* out13) {
  const Grid& g = c.g;
  hipStream_t s = c.stream;
  const long nxy = (long)g.nx * g.ny;
  const int nbp = nblk(nxy, 256);
  double* col = stat_ws(c, (size_t)(COL_N + 1 + 18) * nxy + (size_t)(MAP_N + 1) * nbp + MAP_N + 1 + 2 * (size_t)ncyl);
  double *mask = col + COL_N * nxy, *map = mask + nxy, *part = map + 18 * nxy, *red = part + (MAP_N + 1) * nbp;
  plane_mask(c, ncyl, xy, diameter, red + MAP_N + 1, mask, part + MAP_N * nbp);
  with_fields(c, [&](auto f) {
    with_kind(c, [&](auto wl, auto mean) {
      typedef decltype(f.zero()) T;
      auto k = g.nz >= 8 ? k_column_stats<wl.value, mean.value, 8, T> : k_column_stats<wl.value, mean.value, 4, T>;
      hipLaunchKernelGGL(k, dim3((unsigned)((nxy + 31) / 32)), dim3(g.nz >= 8 ? 256 : 128), 0, s, g, stat_const(g), f, c.mean_u,
                         col);
    });
  });
  const double nu = 1.0 / c.p.re, L2 = c.p.lp * c.p.lp;
  const double epc = 0.5 * (1.0 - c.p.beta) / c.p.re / c.p.wi * (L2 - 3.0);
  hipLaunchKernelGGL(k_map_records, dim3(nbp), dim3(256), 0, s, g, col, mask, nu, epc, map18 ? map : nullptr, part);
  hipLaunchKernelGGL(k_row_sums, dim3(MAP_N + 1), dim3(256), 0, s, part, nbp, red);
  double acc[MAP_N + 1];
  FP_HIP_CHECK(hipMemcpyAsync(acc, red, sizeof(acc), hipMemcpyDeviceToHost, s));
  FP_HIP_CHECK(hipStreamSynchronize(s));
  const double msum = acc[MAP_N];
  if (msum == 0.0) return 1;
  if (map18) {
    FP_HIP_CHECK(hipMemcpyAsync(map18, map, sizeof(double) * 18 * nxy, hipMemcpyDeviceToHost, s));
    FP_HIP_CHECK(hipStreamSynchronize(s));
  }
  if (out13) {
    out13[0] = (double)c.step;
    out13[1] = c.step * c.p.dt;
    out13[2] = acc[0] / msum;   // K
    out13[3] = 0.0;             // no K_staggered in the masked record
    for (int q = 1; q < MAP_N; q++) out13[3 + q] = acc[q] / msum;
  }
  return 0;
}

// fft_energy_dif_map (fenep_mpi.f90:2670-2797): the z transform of the
// regular-grid fluctuation velocity of every (i, j) column, normalised by
// 1/NZ (fft_z, fenep_mpi.f90:1442-1463); energy (|u^|^2 + |v^|^2 + |w^|^2)/2 per
// |kz| = 0..NZ/2, doubled for 0 < kz < NZ/2 (the +-kz pair).  A block transforms
// 2^lnl columns in LDS, u + i v as one complex line (|Z(kz)|^2 + |Z(-kz)|^2 =
// 2 (|u^|^2 + |v^|^2)), then w, and sums the masked columns:
// part[kz gridDim.x + block]; first[kz]: column (1, 1).  (Every column and kz
// as a direct sum over z took 2075 us at 256x128x128, mixed, and the masked sums
// 53; this takes 79, its LDS passes bound it.)
template <typename T>
__global__ __launch_bounds__(256) void k_zspec(Grid g, Fields<T> f, const double* __restrict__ Um, const double* __restrict__ mask,
                                               const double2* __restrict__ tw, int lnl, double* __restrict__ part,
                                               double* __restrict__ first) {
  extern __shared__ double2 lds[];
  const int n = g.nz, L = log2i(n), nl = 1 << lnl, nk = n / 2 + 1;
  double2* tws = lds + (n << lnl);
  double* en = (double*)(tws + n / 2);        // [kz][column]
  const long nxy = (long)g.nx * g.ny, ij0 = (long)blockIdx.x << lnl;
  const double *Vm = Um ? Um + g.n : nullptr, *Wm = Um ? Um + 2 * g.n : nullptr;
  load_tw(tws, tw, n);
  auto regular = [&](const T* F, const double* M, int i, int j, int k, int d, int kind) {
    const int a = d == 0, b = d == 1, c = d == 2;
    double x = (double)ldb(F, g, i, j, k, kind), y = (double)ldb(F, g, i - a, j - b, k - c, kind);
    if (M) { x = x - ldb(M, g, i, j, k, kind); y = y - ldb(M, g, i - a, j - b, k - c, kind); }
    return (x + y) / 2.0;
  };
  const Lines<double2> ln{lds, nl, 1, lnl, L};
  for (int pass = 0; pass < 2; pass++) {
    for (int e = threadIdx.x; e < n << lnl; e += 256) {
      const int l = e & (nl - 1), k = e >> lnl;
      const long ij = ij0 + l;
      const int i = (int)(ij & (g.nx - 1)), j = (int)(ij >> g.lnx);
      lds[e] = pass == 0 ? make_double2(regular(f.U, Um, i, j, k, 0, BC_U), regular(f.V, Vm, i, j, k, 1, BC_V))
                         : make_double2(regular(f.W, Wm, i, j, k, 2, BC_W), 0.0);
    }
    __syncthreads();
    dif_from_natural<3, false>(ln, tws);
    for (int e = threadIdx.x; e < nk << lnl; e += 256) {
      const int l = e & (nl - 1), kz = e >> lnl;
      auto power = [&](int m) {
        const double2 v = lds[(brev(m, L) << lnl) + l];
        const double re = v.x / (double)n, im = v.y / (double)n;
        return re * re + im * im;
      };
      if (pass == 0) {
        en[e] = (power(kz) + power((n - kz) & (n - 1))) / 2.0;
      } else {
        const double v = en[e] + power(kz);
        en[e] = (kz == 0 || kz == n / 2) ? v / 2.0 : v;
      }
    }
    __syncthreads();
  }
  for (int kz = threadIdx.x; kz < nk; kz += 256) {
    double v = 0.0;
    for (int l = 0; l < nl; l++) v += en[(kz << lnl) + l] * mask[ij0 + l];
    part[(long)kz * gridDim.x + blockIdx.x] = v;
    if (blockIdx.x == 0) first[kz] = en[kz << lnl];
  }
}

// fft_energy_dif_map (fenep_mpi.f90:2670-2797) of the current state:
// Emask[kz] = masked plane average of the column z spectra, Efirst[kz] = the
// spectrum of column (1, 1); kz = 0..NZ-1 (zero above NZ/2).
int f64_energy_spectrum_z(Ctx& c, int ncyl, const double* xy, double diameter, double* Emask, double* Efirst) {
  const Grid& g = c.g;
  hipStream_t s = c.stream;
  const long nxy = (long)g.nx * g.ny;
  const int nk = g.nz / 2 + 1, nbp = nblk(nxy, 256);
  const int lnl = std::max(2, std::min(4, 11 - lg(g.nz)));
  const int nb = (int)(nxy >> lnl);
  std::vector<double> r(2 * nk + 1);
  double* dmask = stat_ws(c, (size_t)nxy + (size_t)nk * nb + nbp + 2 * nk + 1 + 2 * (size_t)ncyl);
  double *part = dmask + nxy, *mpart = part + (size_t)nk * nb, *out = mpart + nbp;
  plane_mask(c, ncyl, xy, diameter, out + 2 * nk + 1, dmask, mpart);
  const size_t sh = sizeof(double2) * (((size_t)g.nz << lnl) + g.nz / 2) + sizeof(double) * ((size_t)nk << lnl);
  with_fields(c, [&](auto f) {
    auto k = k_zspec<decltype(f.zero())>;
    if (sh > 65536) FP_HIP_CHECK(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh));
    hipLaunchKernelGGL(k, dim3(nb), dim3(256), sh, s, g, f, c.mean_u, dmask, c.twz, lnl, part, out + nk);
  });
  hipLaunchKernelGGL(k_row_sums, dim3(nk), dim3(256), 0, s, part, nb, out);
  hipLaunchKernelGGL(k_row_sums, dim3(1), dim3(256), 0, s, mpart, nbp, out + 2 * nk);
  FP_HIP_CHECK(hipMemcpyAsync(r.data(), out, sizeof(double) * (2 * nk + 1), hipMemcpyDeviceToHost, s));
  FP_HIP_CHECK(hipStreamSynchronize(s));
  const double msum = r[2 * nk];
  if (msum == 0.0) return 1;
  for (int k = 0; k < g.nz; k++) {
    if (Emask) Emask[k] = k < nk ? r[k] / msum : 0.0;
    if (Efirst) Efirst[k] = k < nk ? r[nk + k] : 0.0;
  }
  return 0;
}

// time-mean accumulation of the velocity (fenep_mpi.f90:2969-2971)
template <typename T>
__global__ __launch_bounds__(256) void k_mean_acc(long n, const T* __restrict__ U, const T* __restrict__ V,
                                                  const T* __restrict__ W, double* __restrict__ acc) {
  const long m = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (m >= n) return;
  acc[m] += (double)U[m];
  acc[n + m] += (double)V[m];
  acc[2 * n + m] += (double)W[m];
}

// mean = acc / count, then (zavg) its z average for every (i, j) (ave_mean,
// fenep_mpi.f90:2010-2033), in k order
__global__ __launch_bounds__(256) void k_mean_finish(Grid g, const double* __restrict__ acc, double count, int zavg,
                                                     double* __restrict__ mean) {
  const long nxy = (long)g.nx * g.ny;
  const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (t >= 3 * nxy) return;
  const int comp = (int)(t / nxy);
  const long ij = t % nxy;
  const double* a = acc + comp * g.n;
  double* o = mean + comp * g.n;
  if (!zavg) {
    for (int k = 0; k < g.nz; k++) o[ij + nxy * k] = a[ij + nxy * k] / count;
    return;
  }
  double s = 0.0;
  for (int k = 0; k < g.nz; k++) s += a[ij + nxy * k] / count;
  s = s / (double)g.nz;
  for (int k = 0; k < g.nz; k++) o[ij + nxy * k] = s;
}

// time mean of the velocity for the mean-subtracted statistics
void f64_mean_accumulate(Ctx& c, const float* u32, const float* v32, const float* w32) {
  const Grid& g = c.g;
  if (!c.mean_acc) {
    FP_HIP_CHECK(hipMalloc((void**)&c.mean_acc, sizeof(double) * 3 * g.n));
    zero_words(c.mean_acc, 6 * g.n, c.stream);
    c.mean_count = 0;
  }
  if (u32)
    hipLaunchKernelGGL(k_mean_acc<float>, dim3(nblk(g.n, 256)), dim3(256), 0, c.stream, g.n, u32, v32, w32, c.mean_acc);
  else
    hipLaunchKernelGGL(k_mean_acc<double>, dim3(nblk(g.n, 256)), dim3(256), 0, c.stream, g.n, (const double*)c.U,
                       (const double*)c.V, (const double*)c.W, c.mean_acc);
  c.mean_count++;
}

int f64_mean_apply(Ctx& c, int mode) {
  const Grid& g = c.g;
  if (mode == 0) {
    if (c.mean_u) (void)hipFree(c.mean_u);
    c.mean_u = nullptr;
  } else {
    if (!c.mean_acc || c.mean_count == 0) return 1;
    if (!c.mean_u) FP_HIP_CHECK(hipMalloc((void**)&c.mean_u, sizeof(double) * 3 * g.n));
    const long nxy = (long)g.nx * g.ny;
    hipLaunchKernelGGL(k_mean_finish, dim3(nblk(3 * nxy, 256)), dim3(256), 0, c.stream, g, c.mean_acc,
                       (double)c.mean_count, mode == 1 ? 1 : 0, c.mean_u);
  }
  if (c.mean_acc) {
    FP_HIP_CHECK(hipStreamSynchronize(c.stream));
    (void)hipFree(c.mean_acc);
    c.mean_acc = nullptr;
  }
  c.mean_count = 0;
  FP_HIP_CHECK(hipStreamSynchronize(c.stream));
  return 0;
}

// ===================================================== energy spectrum =====
// fft_energy_dif (fenep_mpi.f90:2566-2665): the regular-grid velocity, its
// forward transform / N (f64_forward_regular), |u^|^2 summed over the three
// components into integer shells nint(|k|), half weight on the kx = 0 and
// Nyquist planes of the half spectrum.  One row of nbins sums per block and
// component.
__global__ __launch_bounds__(256) void k_spec_shells(Grid g, const double2* __restrict__ spec, int nbins,
                                                     double* __restrict__ part) {
  extern __shared__ double bins[];
  for (int b = threadIdx.x; b < nbins; b += blockDim.x) bins[b] = 0.0;
  __syncthreads();
  const long total = (long)g.nxh * g.ny * g.nz;
  const double2* sp = spec + blockIdx.y * total;
  const double rn = 1.0 / (double)g.n;        // exact: N is a power of two
  const int lnz = log2i(g.nz);
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    // [kx][z][y], the wavenumbers of y and z bit-reversed
    const int j = brev((int)(e & (g.ny - 1)), g.lny);
    const int k = brev((int)((e >> g.lny) & (g.nz - 1)), lnz);
    const int i = (int)(e >> (g.lny + lnz));
    const int ky = j <= g.ny / 2 ? j : j - g.ny, kz = k <= g.nz / 2 ? k : k - g.nz;
    // nint(|k|): (2 idx - 1)^2 <= 4 |k|^2 < (2 idx + 1)^2, an FP32 root put right
    const int k2 = i * i + ky * ky + kz * kz;
    int idx = (int)(sqrtf((float)k2) + 0.5f);
    idx += (4 * k2 >= (2 * idx + 1) * (2 * idx + 1)) - (idx > 0 && 4 * k2 < (2 * idx - 1) * (2 * idx - 1));
    const double2 s = sp[e];
    const double re = s.x * rn, im = s.y * rn;
    const double w = (i == 0 || i == g.nxh - 1) ? 0.5 : 1.0;
    if (idx < nbins) atomicAdd(&bins[idx], (re * re + im * im) * w);
  }
  __syncthreads();
  double* row = part + (long)(blockIdx.y * gridDim.x + blockIdx.x) * nbins;
  for (int b = threadIdx.x; b < nbins; b += blockDim.x) row[b] = bins[b];
}
// E[b] = sum of column b of the rows (16 columns per block, 64 threads each)
__global__ __launch_bounds__(1024) void k_bin_sums(const double* __restrict__ part, int rows, int nbins, double* __restrict__ E) {
  __shared__ double sh[64][16];
  const int l = threadIdx.x & 15, z = threadIdx.x >> 4, b = blockIdx.x * 16 + l;
  double v = 0.0;
  if (b < nbins)
    for (int r = z; r < rows; r += 64) v += part[(long)r * nbins + b];
  sh[z][l] = v;
  __syncthreads();
  if (z == 0 && b < nbins) {
    for (int u = 1; u < 64; u++) v += sh[u][l];
    E[b] = v;
  }
}

void f64_energy_spectrum(Ctx& c, double* E, int nbins) {
  const Grid& g = c.g;
  hipStream_t s = c.stream;
  const long total = (long)g.nxh * g.ny * g.nz;
  const int sb = (int)std::min<long>(256, (total + 255) / 256);
  double* part = stat_ws(c, (size_t)3 * sb * nbins + nbins);
  double* dE = part + (size_t)3 * sb * nbins;
  for (int comp = 0; comp < 3; comp += c.nspec) {
    with_fields(c, [&](auto f) { f64_forward_regular(c, f.U, f.V, f.W, comp, c.nspec); });
    hipLaunchKernelGGL(k_spec_shells, dim3(sb, c.nspec), dim3(256), sizeof(double) * nbins, s, g, c.spec, nbins,
                       part + (size_t)comp * sb * nbins);
  }
  hipLaunchKernelGGL(k_bin_sums, dim3(nblk(nbins, 16)), dim3(1024), 0, s, part, 3 * sb, nbins, dE);
  FP_HIP_CHECK(hipMemcpyAsync(E, dE, sizeof(double) * nbins, hipMemcpyDeviceToHost, s));
  FP_HIP_CHECK(hipStreamSynchronize(s));
}

// ===================================================== diagnostics ========
// sums: ke, trsum, trsq, nitr, nan, Newton stopped at the cap; maxima: u v w
// tr C, the minimum of tr C, the maximum of |div u|.  part[a nb + block]
template <typename T>
__global__ __launch_bounds__(256) void k_diag(Grid g, StatConst K, Fields<T> f, const int* __restrict__ nitr, int polymer,
                                              double* __restrict__ part) {
  double s[6] = {0, 0, 0, 0, 0, 0};
  double mx[6] = {-1e300, -1e300, -1e300, -1e300, 1e300, 0.0};
  const long nb = gridDim.x;
  for (long m = xcd_cell(); m < g.n; m += nb * 256) {
    int i, j, k;
    cell_ijk(g, m, i, j, k);
    const double u = ldb(f.U, g, i, j, k, BC_U), v = ldb(f.V, g, i, j, k, BC_V), w = ldb(f.W, g, i, j, k, BC_W);
    const double um = ldb(f.U, g, i - 1, j, k, BC_U), vm = ldb(f.V, g, i, j - 1, k, BC_V), wm = ldb(f.W, g, i, j, k - 1, BC_W);
    const double ur = (u + um) / 2.0, vr = (v + vm) / 2.0, wr = (w + wm) / 2.0;
    s[0] += ur * ur + vr * vr + wr * wr;
    const double tr = ((double)f.C[m] + (double)f.C[3 * g.n + m]) + (double)f.C[5 * g.n + m];
    s[1] += tr; s[2] += tr * tr;
    if (polymer) {
      const int it = nitr[m];
      s[3] += (double)abs(it);
      s[5] += it < 0 ? 1.0 : 0.0;
    }
    s[4] += isnan((double)f.U[m]) ? 1.0 : 0.0;
    mx[0] = fmax(mx[0], u); mx[1] = fmax(mx[1], v); mx[2] = fmax(mx[2], w); mx[3] = fmax(mx[3], tr);
    mx[4] = fmin(mx[4], tr);
    const double dv = (quot(u - um, K.h[0], K.ih[0]) + quot(v - vm, K.h[1], K.ih[1])) + quot(w - wm, K.h[2], K.ih[2]);
    mx[5] = fmax(mx[5], fabs(dv));
  }
  __shared__ double sh[12][4];
#pragma unroll
  for (int a = 0; a < 6; a++) {
    block_red<Red::Sum>(s[a], sh[a]);
    if (a == 4) block_red<Red::Min>(mx[a], sh[6 + a]);
    else block_red<Red::Max>(mx[a], sh[6 + a]);
  }
  __syncthreads();
  const int a = threadIdx.x;
  if (a < 12)
    part[a * nb + blockIdx.x] = a < 6 ? block_get<Red::Sum>(sh[a]) : (a == 10 ? block_get<Red::Min>(sh[a]) : block_get<Red::Max>(sh[a]));
}

// the 12 per-block partials of k_diag reduced to one value each (one block
// per value), and the sums of the x and y marker forces (two more blocks:
// drag and lift before the -dX^3 factor)
template <typename T>
__global__ __launch_bounds__(256) void k_diag_reduce(const double* __restrict__ part, int nb, const T* __restrict__ mf, long nmk,
                                                     double* __restrict__ out) {
  const int a = blockIdx.x;
  __shared__ double sh[4];
  if (a >= 12) {
    double v = 0.0;
    for (long id = threadIdx.x; id < nmk; id += 256) v += (double)mf[(a - 12) * nmk + id];
    block_red<Red::Sum>(v, sh);
  } else {
    const double* row = part + (long)a * nb;
    double v = a < 6 ? 0.0 : (a == 10 ? 1e300 : -1e300);
    for (int b = threadIdx.x; b < nb; b += 256) {
      const double x = row[b];
      v = a < 6 ? v + x : (a == 10 ? fmin(v, x) : fmax(v, x));
    }
    if (a < 6) block_red<Red::Sum>(v, sh);
    else if (a == 10) block_red<Red::Min>(v, sh);
    else block_red<Red::Max>(v, sh);
  }
  __syncthreads();
  if (threadIdx.x == 0)
    out[a] = a < 6 || a >= 12 ? block_get<Red::Sum>(sh) : (a == 10 ? block_get<Red::Min>(sh) : block_get<Red::Max>(sh));
}

size_t diag_scratch_words(const Grid& g) { return (size_t)12 * stat_blocks(g.n) + 16; }

// log_progress quantities (fenep.f90:2279-2311) and the drag and lift of the
// marker forces, reduced on the device in `scratch` (diag_scratch_words
// doubles, owned by the caller); 14 doubles come back.
void f64_diag(Ctx& c, fp_diag* d, double* scratch) {
  const Grid& g = c.g;
  const int nb = stat_blocks(g.n), rows = c.nmk ? 14 : 12;
  double* out = scratch + (size_t)12 * nb;
  with_fields(c, [&](auto f) {
    typedef decltype(f.zero()) T;
    const T* mf = nullptr;
    if constexpr (sizeof(T) == 4) mf = mixed_marker_forces32(c);
    else mf = c.mf;
    hipLaunchKernelGGL(k_diag<T>, dim3(nb), dim3(256), 0, c.stream, g, stat_const(g), f, c.nitr, c.p.beta != 1.0 ? 1 : 0, scratch);
    hipLaunchKernelGGL(k_diag_reduce<T>, dim3(rows), dim3(256), 0, c.stream, scratch, nb, mf, c.nmk, out);
  });
  double h[14] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  FP_HIP_CHECK(hipMemcpyAsync(h, out, sizeof(double) * rows, hipMemcpyDeviceToHost, c.stream));
  FP_HIP_CHECK(hipStreamSynchronize(c.stream));
  const double N = (double)g.n;
  d->ke = (h[0] / 2.0) / N;
  d->cfl = std::max(h[6] * g.dt / g.dx, std::max(h[7] * g.dt / g.dy, h[8] * g.dt / g.dz)) * 6.0;
  d->trc_mean = h[1] / N;
  d->trc_std = std::sqrt(std::max(0.0, h[2] / N - d->trc_mean * d->trc_mean));
  d->trc_max = h[9];
  d->trc_min = h[10];
  d->div_max = h[11];
  d->newton_itr_mean = h[3] / N;
  d->newton_unconverged = h[5];
  d->nan_flag = h[4] > 0 ? 1 : 0;
  if (c.nmk) {
    d->drag = -(h[12] * g.sw);
    d->lift = -(h[13] * g.sw);
  }
}

}  // namespace fp
