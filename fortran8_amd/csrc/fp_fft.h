// Transforms of lines held in LDS, in place: radix-2 decimations in frequency,
// two or three stages per pass with the elements in registers, natural order
// in and bit-reversed out, or bit-reversed in and natural out.  V: the complex
// type (double2 for the FP64 path, float2 for the mixed one).
#pragma once
#include "fp_device.h"
#include <algorithm>

namespace fp {

__device__ __forceinline__ int brev(int v, int bits) { return bits ? (int)(__brev((unsigned)v) >> (32 - bits)) : 0; }

// one radix-2 butterfly of the Stockham form: (a, b) -> (a + b, (a - b) w)
template <bool CONJ, typename V>
__device__ __forceinline__ void bfly(V& a, V& b, V w) {
  const auto wi = CONJ ? -w.y : w.y;
  const auto dr = a.x - b.x, di = a.y - b.y;
  a.x = a.x + b.x;
  a.y = a.y + b.y;
  b.x = dr * w.x - di * wi;
  b.y = dr * wi + di * w.x;
}

// LR radix-2 stages, spans len/2, len/4, ..., on the 2^LR elements p + c
// len/2^LR of one block: p the first one's place in the block, sh = log2(n /
// len)
template <int LR, bool CONJ, typename V>
__device__ __forceinline__ void stages(V (&v)[1 << LR], int p, int step, int sh, const V* tws) {
  constexpr int R = 1 << LR;
#pragma unroll
  for (int s = 0; s < LR; s++) {
    const int half = R >> (s + 1);
#pragma unroll
    for (int c = 0; c < half; c++) {
      const V w = tws[(p + c * step) << (sh + s)];
#pragma unroll
      for (int b = 0; b < R; b += 2 * half) bfly<CONJ>(v[b + c], v[b + c + half], w);
    }
  }
}

// A set of 2^lnl lines of n = 2^L points in LDS: point r of line l at
// X[r rs + l ls].  Consecutive threads take consecutive lines, whose stride
// (1, or an odd pitch) keeps the 16-byte accesses off each other's banks.
template <typename V>
struct Lines {
  V* X;
  int rs, ls, lnl, L;
};

// the LR stages from blocks of 2^ll points on; REV: the points lie
// bit-reversed
template <int LR, bool CONJ, bool REV, typename V>
__device__ __forceinline__ void dif_pass(const Lines<V>& f, int ll, const V* tws) {
  constexpr int R = 1 << LR;
  const int n = 1 << f.L, step = 1 << (ll - LR);
  for (int e = threadIdx.x; e < (n >> LR) << f.lnl; e += blockDim.x) {
    const int l = e & ((1 << f.lnl) - 1), t = e >> f.lnl;
    const int p = t & (step - 1), base = ((t >> (ll - LR)) << ll) + p;
    V* x = f.X + l * f.ls;
    V v[R];
    int at[R];
#pragma unroll
    for (int c = 0; c < R; c++) {
      const int o = base + c * step;
      at[c] = (REV ? brev(o, f.L) : o) * f.rs;
      v[c] = x[at[c]];
    }
    stages<LR, CONJ>(v, p, step, f.L - ll, tws);
#pragma unroll
    for (int c = 0; c < R; c++) x[at[c]] = v[c];
  }
  __syncthreads();
}

// The stages of a transform of 2^L points in passes of M (2 or 3): forward,
// what is left over comes first, as one shorter pass (M = 3, L = 1 mod 3: two
// of two stages); the inverse mirrors it.
__device__ __forceinline__ int lead_stages(int M, int L) { return M == 2 ? (L & 1) : (L % 3 == 1 ? 4 : L % 3); }
// stages of the last forward pass and of the first inverse one
__device__ __forceinline__ int last_stages(int M, int L) { return M == 3 && L != 2 && L != 4 ? 3 : 2; }

// natural order in, bit-reversed out; all passes, or all but the last one
template <int M, bool CONJ, typename V>
__device__ __forceinline__ void dif_from_natural(const Lines<V>& f, const V* tws, bool all = true) {
  const int stop = all ? 0 : last_stages(M, f.L);
  const int rest = f.L - lead_stages(M, f.L);
  int ll = f.L;
  if constexpr (M == 2) {
    if (ll > rest) { dif_pass<1, CONJ, false>(f, ll, tws); ll--; }
  } else {
    for (; ll > rest && ll > stop; ll -= 2) dif_pass<2, CONJ, false>(f, ll, tws);
  }
  for (; ll > stop; ll -= M) dif_pass<M, CONJ, false>(f, ll, tws);
}
// bit-reversed in, natural order out; all passes, or all but the first one
template <int M, typename V>
__device__ __forceinline__ void dif_from_reversed(const Lines<V>& f, const V* tws, bool all = true) {
  const int lead = lead_stages(M, f.L);
  int ll = f.L - (all ? 0 : last_stages(M, f.L));
  for (; ll > lead; ll -= M) dif_pass<M, true, true>(f, ll, tws);
  if constexpr (M == 2) {
    if (ll > 0) dif_pass<1, true, true>(f, ll, tws);
  } else {
    for (; ll > 0; ll -= 2) dif_pass<2, true, true>(f, ll, tws);
  }
}

// The last forward pass, op on every spectrum value, the first inverse pass:
// both work on the same 2^LR elements (places t R + c, wavenumbers bitrev(c)
// n/R + bitrev(t)), which stay in registers between them.
template <int LR, typename V, typename Op>
__device__ __forceinline__ void turn_pass(const Lines<V>& f, const V* tws, Op op) {
  constexpr int R = 1 << LR;
  const int n = 1 << f.L;
  for (int e = threadIdx.x; e < (n >> LR) << f.lnl; e += blockDim.x) {
    const int l = e & ((1 << f.lnl) - 1), t = e >> f.lnl;
    V* x = f.X + l * f.ls + t * R * f.rs;
    V v[R], u[R];
#pragma unroll
    for (int c = 0; c < R; c++) v[c] = x[c * f.rs];
    stages<LR, false>(v, 0, 1, f.L - LR, tws);
    const int p = brev(t, f.L - LR), step = n >> LR;
#pragma unroll
    for (int c = 0; c < R; c++) {
      // static bit reversal of c in LR bits
      const int rc = LR == 2 ? ((c & 1) << 1 | c >> 1) : ((c & 1) << 2 | (c & 2) | c >> 2);
      u[rc] = op(l, p + rc * step, v[c]);
    }
    stages<LR, true>(u, p, step, 0, tws);
#pragma unroll
    for (int c = 0; c < R; c++) {
      const int rc = LR == 2 ? ((c & 1) << 1 | c >> 1) : ((c & 1) << 2 | (c & 2) | c >> 2);
      x[c * f.rs] = u[rc];
    }
  }
  __syncthreads();
}
template <int M, typename V, typename Op>
__device__ __forceinline__ void turn(const Lines<V>& f, const V* tws, Op op) {
  if (M == 2 || last_stages(M, f.L) == 2) turn_pass<2>(f, tws, op);
  else turn_pass<3>(f, tws, op);
}

__device__ __forceinline__ int log2i(int n) { return __ffs(n) - 1; }

// store(e, load(e)) for e < total over the block, U loads of a thread in
// flight: one at a time, the copy of 33 KB into the LDS by 128 threads waits 16
// times on memory
template <int U, typename V, typename Load, typename Store>
__device__ __forceinline__ void copy_ahead(int total, Load load, Store store) {
  const int nt = blockDim.x;
  for (int e = threadIdx.x; e < total; e += U * nt) {
    V v[U];
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = load(min(e + u * nt, total - 1));
#pragma unroll
    for (int u = 0; u < U; u++)
      if (e + u * nt < total) store(e + u * nt, v[u]);
  }
}

// twiddles exp(-2 pi i t/n), t < n/2, into LDS (no barrier)
template <typename V>
__device__ __forceinline__ void load_tw(V* tws, const V* __restrict__ tw, int n) {
  for (int e = threadIdx.x; e < n / 2; e += blockDim.x) tws[e] = tw[e];
}

// ---- host: launch shapes
static inline int lg(int n) { int l = 0; while ((1 << l) < n) l++; return l; }

// log2 of the lines of n points a block holds: 16 where they take at most 33
// KB of LDS (four blocks per CU), fewer for long lines, and fewer (4 at
// least) while the launch would leave CUs without a block
static inline int lines_log2(int n, long lines, int comps) {
  int l = std::max(2, std::min(4, 11 - lg(n)));
  while (l > 2 && (lines >> l) * comps < 512) l--;
  while (l > 0 && (1L << l) > lines) l--;
  return l;
}
static inline size_t lds_lines(int n, int lnl) { return sizeof(double2) * (((size_t)(n + 1) << lnl) + n / 2); }

}  // namespace fp
