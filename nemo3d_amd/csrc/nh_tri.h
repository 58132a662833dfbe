// Eigenvalues of a symmetric tridiagonal matrix in two windows, and the last
// two components of their eigenvectors, on the device: the convergence check
// of the Lanczos runs.
//
// A workgroup of four wavefronts per eigenvalue.  Its lanes count the
// eigenvalues below 256 points of the interval at a time (signs of the leading
// minors, three-term recurrence with rescaling), which cuts the interval by
// 257 a pass; then two wavefronts run the pivots from both ends, and the
// eigenvector follows from the position where they meet best (twisted
// factorisation), without inverse iteration.  The kernel uses no LDS and few
// registers, so that it runs beside a Lanczos step that fills the LDS of every
// compute unit; the wavefronts meet in the scratch memory.  (Three workgroups of
// an FP32 step leave 56 registers of a SIMD; with 80 of them for the check, for
// a loop over eigenvalues, the step went from 239 to 255 us, 786,520 atoms.)
// Bound by the serial recurrences, 38 cycles a row and pass (6 passes) and
// about 85 a row for the pivots: 0.30 ms at 1,375 rows.  (One wavefront, 64
// points, the pivots and the components by two lanes: 547 us; four points a
// lane: 776 us, the FP64 units are busy with one; rows handed out by readlane
// instead of scalar loads: 145 cycles a row.)  On 8 host threads (bisection
// with a division a row, threads started for each check) a check took longer
// than the 25 steps between two of them: a whole solve of 3,888 atoms 57 ms,
// now 24, a mixed one of 172,032 atoms 355 ms, now 230.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace nh {

struct TriWindows {
  double lo[2], hi[2];
  int want[2];  // at most so many: the highest of window 0, the lowest of 1
};
// results: kTriHead doubles (eigenvalues taken of windows 0, 1), then 3 an
// eigenvalue: value, last and last but one component
constexpr int kTriHead = 2, kTriOut = 3;
constexpr int kTriThreads = 256;
constexpr int kTriGroups = 512;  // workgroups of a launch at most (their scratch)
// scratch of a workgroup, in doubles: pivots from both ends, and what the
// wavefronts tell each other
inline int64_t tri_scratch(int m) { return 2 * (int64_t)m + 32; }

// eigenvalues of T_m (a diagonal, b off-diagonal) below x
__device__ inline int tri_count(int m, const double *__restrict__ a,
                                const double *__restrict__ b, double x) {
  double p0 = 0.0, p1 = 1.0, e = 0.0;
  int cnt = 0;
  uint32_t signs = 0;  // sign bits of the last minors, the newest lowest
  auto row = [&](double d, double off) {
    const double t = e * p0;
    const double p = __builtin_fma(d - x, p1, -(e * t));
    p0 = p1;
    p1 = p;
    e = off;
    signs = signs << 1 | (uint32_t)(__double_as_longlong(p) >> 63 & 1);
  };
  constexpr int kU = 8;
  double d[kU], f[kU];
  const int full = m / kU * kU;
  if (full > 0)
#pragma unroll
    for (int u = 0; u < kU; ++u) d[u] = a[u], f[u] = b[u];
  for (int i = 0; i < full; i += kU) {
    // the next rows are requested before these are used
    double dn[kU], fn[kU];
    const int nx = i + kU < full ? i + kU : i;
#pragma unroll
    for (int u = 0; u < kU; ++u) dn[u] = a[nx + u], fn[u] = b[nx + u];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kU; ++u) row(d[u], f[u]);
    cnt += __builtin_popcount((signs ^ signs >> 1) & ((1u << kU) - 1));
    const int s = __builtin_amdgcn_frexp_exp(fmax(fabs(p0), fabs(p1)));
    p0 = __builtin_amdgcn_ldexp(p0, -s);
    p1 = __builtin_amdgcn_ldexp(p1, -s);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      // opaque, or the compiler moves the loads behind the loop's back edge
      asm volatile("" : "+s"(dn[u]), "+s"(fn[u]));
      d[u] = dn[u], f[u] = fn[u];
    }
  }
  for (int i = full; i < m; ++i) {
    row(a[i], b[i]);
    cnt += (signs ^ signs >> 1) & 1;
  }
  return cnt;
}

// Pivots of T_m - v from the front (BACK: from the back) by one wavefront, the
// lanes alike; to q[0 .. m)
template <bool BACK>
__device__ inline void tri_pivots(int m, const double *__restrict__ a,
                                  const double *__restrict__ b, double v, double *q) {
  const int lane = threadIdx.x & 63;
  double p = 1.0, keep = 0.0;
  auto row = [&](int t, double d, double e) {
    // 1 / p to rounding: the hardware's approximation and two Newton steps
    double r = __builtin_amdgcn_rcp(p);
    r = __builtin_fma(__builtin_fma(-p, r, 1.0), r, r);
    r = __builtin_fma(__builtin_fma(-p, r, 1.0), r, r);
    p = __builtin_fma(-(e * e), r, d - v);
    if (fabs(p) < 1e-280) p = 1e-280;  // its inverse must be finite
    if (lane == (t & 63)) keep = p;
  };
  auto flush = [&](int t) {  // rows t & ~63 .. t
    const int s = (t & ~63) + lane;
    if (s <= t) q[BACK ? m - 1 - s : s] = keep;
  };
  constexpr int kU = 8;
  double d[kU], e[kU];
  auto load = [&](int t0, double (&dd)[kU], double (&ee)[kU]) {
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int i = BACK ? m - 1 - t0 - u : t0 + u;
      dd[u] = a[i];
      ee[u] = BACK ? b[i] : b[i > 0 ? i - 1 : 0];
    }
  };
  const int full = m / kU * kU;
  if (full > 0) load(0, d, e);
  for (int t0 = 0; t0 < full; t0 += kU) {
    double dn[kU], en[kU];
    load(t0 + kU < full ? t0 + kU : t0, dn, en);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kU; ++u) row(t0 + u, d[u], t0 + u > 0 ? e[u] : 0.0);
    if ((t0 & 63) == 56) flush(t0 + 7);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      asm volatile("" : "+s"(dn[u]), "+s"(en[u]));  // as in tri_count
      d[u] = dn[u], e[u] = en[u];
    }
  }
  for (int t = full; t < m; ++t) {
    const int i = BACK ? m - 1 - t : t;
    row(t, a[i], t == 0 ? 0.0 : b[BACK ? i : i - 1]);
  }
  if ((m & 63) != 0) flush(m - 1);
}

// Products of the n ratios f[0], f[dir], f[2 dir], .. by one wavefront: the
// sum of their squares, the first, the last and the last but one
struct TriProducts {
  double sum, first, last, before;
};
__device__ inline TriProducts tri_products(const double *f, int dir, int n) {
  const int lane = threadIdx.x & 63;
  double carry = 1.0, sum = 0.0, first = 1.0, last = 1.0, before = 1.0;
  for (int c = 0; c < n; c += 64) {
    const int t = c + lane;
    double p = t < n ? f[(int64_t)dir * t] : 1.0;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const double o = __shfl_up(p, off, 64);
      if (lane >= off) p *= o;
    }
    p *= carry;
    if (t < n) sum = __builtin_fma(p, p, sum);
    if (t == 0) first = p;
    if (t == n - 1) last = p;
    if (t == n - 2) before = p;
    carry = __shfl(p, 63, 64);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  return {sum, __shfl(first, 0, 64), n > 0 ? __shfl(last, (n - 1) & 63, 64) : 1.0,
          n > 1 ? __shfl(before, (n - 2) & 63, 64) : 1.0};
}

// Eigenvalues first, first + 1, .. of the windows' want[0] + want[1], one a
// workgroup.  S: tri_scratch(m) doubles a workgroup
__global__ __launch_bounds__(kTriThreads) void k_tri_windows(
    int m, const double *__restrict__ a, const double *__restrict__ b, TriWindows win,
    int first, double *S, double *__restrict__ out) {
  constexpr int kPts = kTriThreads, kWaves = kTriThreads / 64;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int idx = first + (int)blockIdx.x;
  const int w = idx >= win.want[0], j = idx - (w ? win.want[0] : 0);
  double *F = S + (int64_t)blockIdx.x * (2 * (int64_t)m + 32), *B = F + m, *talk = B + m;
  // the first point with more than k eigenvalues below (kPts: none); slot: of
  // the talk, in turn
  auto first_above = [&](int cnt, int k, int slot) {
    const uint64_t above = __ballot(cnt > k);
    if (lane == 0)
      talk[slot * kWaves + wave] = above ? 64 * wave + __builtin_ctzll(above) : kPts;
    __syncthreads();
    double l = kPts;
#pragma unroll
    for (int q = 0; q < kWaves; ++q) l = fmin(l, talk[slot * kWaves + q]);
    return (int)l;
  };
  // numbers of the eigenvalues in the window, and this workgroup's, from a
  // first pass with points from end to end of the window
  double lo = win.lo[w], hi = win.hi[w];
  // window ends beyond T's Gershgorin bounds (an open window: +-1e99, infinity)
  // are moved to them: eight minors at such a point leave the range of a double
  {
    double mn = INFINITY, mx = -INFINITY;
    for (int i = tid; i < m; i += kTriThreads) {
      const double r = (i > 0 ? fabs(b[i - 1]) : 0.0) + (i + 1 < m ? fabs(b[i]) : 0.0);
      mn = fmin(mn, a[i] - r);
      mx = fmax(mx, a[i] + r);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      mn = fmin(mn, __shfl_xor(mn, off, 64));
      mx = fmax(mx, __shfl_xor(mx, off, 64));
    }
    double *ends = talk + 5 * kWaves;
    if (lane == 0) {
      ends[2 * wave] = mn;
      ends[2 * wave + 1] = mx;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kWaves; ++q) {
      mn = fmin(mn, ends[2 * q]);
      mx = fmax(mx, ends[2 * q + 1]);
    }
    const double eps = 1e-12 * (fabs(mn) + fabs(mx)) + 1e-30;
    auto inside = [&](double x) { return x < mn - eps ? mn - eps : x > mx + eps ? mx + eps : x; };
    lo = inside(lo);
    hi = inside(hi);
  }
  auto point = [&](double h, int i) { return __builtin_fma(h, (double)i, lo); };
  int k, n;
  {
    const double h = (hi - lo) / (kPts - 1);
    const int cnt = tri_count(m, a, b, tid == kPts - 1 ? hi : point(h, tid));
    if (tid == 0) talk[4 * kWaves] = cnt;
    if (tid == kPts - 1) talk[4 * kWaves + 1] = cnt;
    __syncthreads();
    const int klo = (int)talk[4 * kWaves], khi = (int)talk[4 * kWaves + 1];
    n = min(khi - klo, win.want[w]);
    k = w == 0 ? khi - n + j : klo + j;
    if (j == 0 && tid == 0) out[w] = n > 0 ? (double)n : 0.0;
    if (j >= n) return;
    const int l = max(first_above(cnt, k, 0), 1);  // klo <= k < khi
    const double nlo = point(h, l - 1), nhi = l < kPts - 1 ? point(h, l) : hi;
    lo = nlo;
    hi = nhi;
  }
  for (int it = 1; it < 64 && hi - lo > 1e-13; ++it) {
    const double h = (hi - lo) / (kPts + 1);
    const int l = first_above(tri_count(m, a, b, point(h, tid + 1)), k, it & 1);
    const double nlo = l > 0 ? point(h, l) : lo;
    const double nhi = l < kPts ? point(h, l + 1) : hi;
    if (!(nhi - nlo < hi - lo)) break;
    lo = nlo;
    hi = nhi;
  }
  const double v = 0.5 * (lo + hi);

  if (wave == 0) tri_pivots<false>(m, a, b, v, F);
  if (wave == 1) tri_pivots<true>(m, a, b, v, B);
  __syncthreads();
  // where they meet best
  double best = INFINITY;
  int r = 0;
  for (int i = tid; i < m; i += kTriThreads) {
    const double g = fabs(F[i] + B[i] - (a[i] - v));
    if (g < best) {
      best = g;
      r = i;
    }
  }
  auto better = [&](double g, int o) {
    if (g < best || (g == best && o < r)) {
      best = g;
      r = o;
    }
  };
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double g = __shfl_xor(best, off, 64);
    better(g, __shfl_xor(r, off, 64));
  }
  if (lane == 0) {
    talk[2 * kWaves + 2 * wave] = best;
    talk[2 * kWaves + 2 * wave + 1] = r;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kWaves; ++q)
    better(talk[2 * kWaves + 2 * q], (int)talk[2 * kWaves + 2 * q + 1]);
  // component ratios away from it
  for (int i = tid; i < m; i += kTriThreads) {
    if (i < r) F[i] = -b[i] / F[i];
    else if (i > r) F[i] = -b[i - 1] / B[i];
  }
  __syncthreads();
  if (wave == 0) {
    const TriProducts down = tri_products(F + (r > 0 ? r - 1 : 0), -1, r);
    if (lane == 0) {
      talk[0] = down.sum;
      talk[1] = down.first;
    }
  }
  TriProducts up{0.0, 1.0, 1.0, 1.0};
  if (wave == 1) up = tri_products(F + (r < m - 1 ? r + 1 : m - 1), 1, m - 1 - r);
  __syncthreads();
  if (wave == 1 && lane == 0) {
    const double norm = sqrt(1.0 + talk[0] + up.sum);
    double *o = out + kTriHead + (int64_t)idx * kTriOut;
    o[0] = v;
    o[1] = up.last / norm;
    // the row before the last: the first one down if the last is r
    o[2] = m >= 2 ? (r == m - 1 ? talk[1] : up.before) / norm : 0.0;
  }
}

}  // namespace nh
