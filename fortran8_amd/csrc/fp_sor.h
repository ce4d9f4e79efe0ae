// Red-black SOR sweeps on tiles held in LDS (the SOR variant of the Poisson
// equation, fenep.f90:848-905), for the FP64 path and, in FP32, the mixed one.
//
// A launch per colour and one for the residual's sum made a sweep of a 128 x
// 64 x 64 grid 16 us long, for arrays of 2 MB that never leave the caches:
// launches and latency.  Here a block holds whole x-lines of a TY x TZ tile in
// (y, z) and two halo rows on each side and makes a full sweep: red on the
// tile and one row around it, black on the tile.  The halo's updates are its
// neighbours' own, operation for operation, so every cell's value is the one a
// colour at a time gives.  In and out are two arrays.  One sweep of 128 x 64 x
// 64 in FP32 takes 6.2 us (4 x 4 tiles, one block per CU; 7.0 in 4 x 2 tiles),
// of 64 x 64 x 32 in FP64 5.0 us (4 x 2; 5.9 in 2 x 2), where the two colours
// took 9.4 and 8.2 and their sum 2.8.  Two sweeps a launch with four halo rows
// took 13.5 and 10.4 us: the halo's work grows faster than the launches shrink.
#pragma once
#include "fp_device.h"
#include <algorithm>

namespace fp {

template <typename T>
struct SorCoef {
  T bx, by, bz, b0;
  T om, ib0;   // FP64: omega and RN(1/b0); FP32: omega/b0 and unused
};
__device__ __forceinline__ double sor_update(const SorCoef<double>& k, double p0, double e) {
  return p0 + quot(k.om * e, k.b0, k.ib0);
}
__device__ __forceinline__ float sor_update(const SorCoef<float>& k, float p0, float e) { return p0 + k.om * e; }

template <typename T, int TY, int TZ>
struct SorTile {
  static constexpr int H = 2;                           // halo rows
  static constexpr int WY = TY + 2 * H, WZ = TZ + 2 * H;   // rows of the iterate; two fewer of the right-hand side
  static size_t lds(const Grid& g) { return sizeof(T) * (size_t)g.nx * (WY * WZ + (WY - 2) * (WZ - 2)); }
};

// stop: nonzero ends the launch at once (converged); part[block]: the block's
// sum of E^2, E taken before each update; zero_in: the iterate starts from zero and `in` is not read.
// A row lies in LDS with its even x first, then the odd: the lanes of a
// half-sweep read runs.  LN: log2 nx where it is one of the usual ones (row
// strides are constants then), 0 for any.  From nx = 128 on a wavefront holds
// part of one row, whose number and place are scalars.
template <typename T, bool WL, int TY, int TZ, int LN>
__global__ __launch_bounds__(1024) void k_sor_tile(Grid g, SorCoef<T> co, const T* __restrict__ q, const T* __restrict__ in,
                                                   T* __restrict__ out, double* __restrict__ part, int zero_in,
                                                   const int* __restrict__ stop) {
  using Tile = SorTile<T, TY, TZ>;
  constexpr int H = Tile::H, WY = Tile::WY, WZ = Tile::WZ, QY = WY - 2, QZ = WZ - 2;
  constexpr int THREADS = LN ? std::min(1024, std::max(64, TY * TZ << (LN - 1))) : 0;
  extern __shared__ double sor_lds[];
  __shared__ double s_sum[16];
  if (*stop) return;
  T* E = (T*)sor_lds;
  const int lnx = LN ? LN : g.lnx, nx = 1 << lnx, h2 = nx >> 1, lh = lnx - 1;
  T* Q = E + WY * WZ * nx;
  const int lty = g.lny - __builtin_ctz(TY);
  const long b = xcd_block();
  const int j0 = (int)(b & ((1 << lty) - 1)) * TY, k0 = (int)(b >> lty) * TZ;
  struct alignas(2 * sizeof(T)) Pair { T a, b; };
  auto row_of = [&](int e) { return LN >= 7 ? __builtin_amdgcn_readfirstlane(e >> lh) : e >> lh; };
  // all of a thread's loads are issued before the first is stored: each would
  // wait a memory latency on its own
  const int th = LN ? THREADS : (int)blockDim.x;
  constexpr int NE = LN ? (WY * WZ * (1 << (LN - 1)) + THREADS - 1) / THREADS : 8;
  // (a trip loads NE and NQ pairs a thread: as many of the right-hand side, in
  // proportion, as of the iterate, whose count ends the loop)
  constexpr int NQ = LN ? (QY * QZ * (1 << (LN - 1)) + THREADS - 1) / THREADS : (NE * QY * QZ + WY * WZ - 1) / (WY * WZ);
  static_assert((LN ? WY * WZ * (1 << (LN - 1)) <= NE * THREADS && QY * QZ * (1 << (LN - 1)) <= NQ * THREADS
                    : NQ * WY * WZ >= NE * QY * QZ), "every row of the right-hand side is loaded");
  for (int e0 = threadIdx.x, q0 = threadIdx.x; e0 < (WY * WZ) << lh; e0 += NE * th, q0 += NQ * th) {
    Pair pe[NE], pq[NQ];
#pragma unroll
    for (int u = 0; u < NE; u++) {
      // (rows beyond a wall are loaded, wrapped, and not used)
      const int row = min(row_of(e0 + u * th), WY * WZ - 1), h = (e0 + u * th) & (h2 - 1);
      const int jw = (j0 - H + row % WY) & (g.ny - 1), kk = (k0 - H + row / WY) & (g.nz - 1);
      pe[u] = zero_in ? Pair{T(0), T(0)} : ((const Pair*)(in + ((size_t)(jw + (kk << g.lny)) << lnx)))[h];
    }
#pragma unroll
    for (int u = 0; u < NQ; u++) {
      const int row = min(row_of(q0 + u * th), QY * QZ - 1), h = (q0 + u * th) & (h2 - 1);
      const int jw = (j0 - H + 1 + row % QY) & (g.ny - 1), kk = (k0 - H + 1 + row / QY) & (g.nz - 1);
      pq[u] = ((const Pair*)(q + ((size_t)(jw + (kk << g.lny)) << lnx)))[h];
    }
#pragma unroll
    for (int u = 0; u < NE; u++) {
      const int row = row_of(e0 + u * th), h = (e0 + u * th) & (h2 - 1);
      if (row < WY * WZ) {
        E[row * nx + h] = pe[u].a;
        E[row * nx + h2 + h] = pe[u].b;
      }
    }
#pragma unroll
    for (int u = 0; u < NQ; u++) {
      const int row = row_of(q0 + u * th), h = (q0 + u * th) & (h2 - 1);
      if (row < QY * QZ) {
        Q[row * nx + h] = pq[u].a;
        Q[row * nx + h2 + h] = pq[u].b;
      }
    }
  }
  __syncthreads();
  double sum = 0.0;
#pragma unroll
  for (int s = 0; s < 2; s++) {
    const int wy = WY - 2 - 2 * s, wz = WZ - 2 - 2 * s;   // rows updated
    for (int e = threadIdx.x; e < (wy * wz) << lh; e += blockDim.x) {
      const int row = row_of(e), h = e & (h2 - 1);
      const int ry = s + 1 + row % wy, rz = s + 1 + row / wy;
      const int jj = j0 - H + ry, kk = k0 - H + rz;
      if (WL && (jj < 0 || jj >= g.ny)) continue;
      const int par = (jj + kk + s) & 1;    // colour s: (i + j + k) % 2
      T* R = E + (rz * WY + ry) * nx;
      T* c = R + par * h2 + h;
      const T* o = R + (1 - par) * h2;      // the x neighbours
      const int hm = (h - 1) & (h2 - 1), hp = (h + 1) & (h2 - 1);
      const T p0 = *c;
      const T xm = o[par ? h : hm], xp = o[par ? hp : h];
      // P_kabe: a wall's ghost is the cell's own value
      const T ym = WL && jj == 0 ? p0 : c[-nx], yp = WL && jj == g.ny - 1 ? p0 : c[nx];
      const T zm = c[-WY * nx], zp = c[WY * nx];
      const T v = (((((co.bz * zm + co.by * ym) + co.bx * xm) - co.b0 * p0) + co.bx * xp) + co.by * yp) + co.bz * zp -
                  Q[((rz - 1) * QY + (ry - 1)) * nx + par * h2 + h];
      *c = sor_update(co, p0, v);
      if (ry >= H && ry < H + TY && rz >= H && rz < H + TZ) sum += (double)v * (double)v;
    }
    __syncthreads();
  }
  for (int e = threadIdx.x; e < (TY * TZ) << lh; e += blockDim.x) {
    const int row = row_of(e), h = e & (h2 - 1);
    const int ry = row % TY, rz = row / TY;
    const T* R = E + ((rz + H) * WY + ry + H) * nx;
    ((Pair*)(out + ((size_t)((j0 + ry) + ((k0 + rz) << g.lny)) << lnx)))[h] = Pair{R[h], R[h2 + h]};
  }
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_down(sum, o);
  if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = 0.0;
    for (unsigned t = 0; t < blockDim.x >> 6; t++) v += s_sum[t];
    part[blockIdx.x] = v;
  }
}

// Sums of `rows` rows (at most 16) of nb partials, a wavefront per row, into
// res[] for the calling block of 1024 threads (ends with a barrier).
__device__ __forceinline__ void sor_row_sums(const double* __restrict__ part, int nb, int rows, double* res) {
  const int r = threadIdx.x >> 6;
  double v = 0.0;
  if (r < rows)
    for (int i = threadIdx.x & 63; i < nb; i += 64) v += part[(long)r * nb + i];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o);
  if ((threadIdx.x & 63) == 0 && r < rows) res[r] = v;
  __syncthreads();
}

// The kernels a grid takes: the largest tile that fits in a block's LDS and
// leaves a block per CU, whole otherwise; none for long FP64 x-lines (a colour
// per launch there).
template <typename T>
struct SorPlan {
  typedef void (*Kernel)(Grid, SorCoef<T>, const T*, const T*, T*, double*, int, const int*);
  Kernel k = nullptr;
  size_t lds = 0;
  long blocks = 0;
  int threads = 0;
};
template <typename T, int TY, int TZ>
inline bool sor_fit(const Grid& g, size_t lds_max, long least, SorPlan<T>& p) {
  const size_t lds = SorTile<T, TY, TZ>::lds(g);
  const long blocks = (long)(g.ny / TY) * (g.nz / TZ);
  if (lds > lds_max || blocks < least) return false;
#define SOR_K(WL)                                                                                   \
  (g.lnx == 7 ? k_sor_tile<T, WL, TY, TZ, 7> : g.lnx == 6 ? k_sor_tile<T, WL, TY, TZ, 6> \
   : g.lnx == 8 ? k_sor_tile<T, WL, TY, TZ, 8> : k_sor_tile<T, WL, TY, TZ, 0>)
  p.k = g.walls ? SOR_K(true) : SOR_K(false);
#undef SOR_K
  p.lds = lds;
  p.blocks = blocks;
  p.threads = (int)std::max(64L, std::min(1024L, (long)TY * TZ * (g.nx / 2)));
  FP_HIP_CHECK(hipFuncSetAttribute((const void*)p.k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_max));
  return true;
}
template <typename T>
inline SorPlan<T> sor_plan(const Grid& g) {
  SorPlan<T> p;
  int lds = 0, dev = 0;
  FP_HIP_CHECK(hipGetDevice(&dev));
  FP_HIP_CHECK(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
  const size_t lds_max = (size_t)lds - 1024;   // beside the kernel's own sums
  sor_fit<T, 4, 4>(g, lds_max, 256, p) || sor_fit<T, 4, 2>(g, lds_max, 256, p) ||
      sor_fit<T, 2, 2>(g, lds_max, 1, p);
  return p;
}

// `sweeps` sweeps from buf[0] (zero_in: from zero), alternating between the
// two arrays; part receives one row of p.blocks sums per sweep.  Returns the
// launches made: the iterate is in buf[launches & 1].
template <typename T>
inline int sor_launch(const Grid& g, const SorPlan<T>& p, const SorCoef<T>& co, const T* q, T* const (&buf)[2], double* part,
                      int sweeps, bool zero_in, const int* stop, hipStream_t s) {
  int l = 0;
  for (; l < sweeps; l++)
    hipLaunchKernelGGL(p.k, dim3((unsigned)p.blocks), dim3(p.threads), p.lds, s, g, co, q, buf[l & 1], buf[(l + 1) & 1],
                       part + l * p.blocks, zero_in && l == 0 ? 1 : 0, stop);
  return l;
}

}  // namespace fp
