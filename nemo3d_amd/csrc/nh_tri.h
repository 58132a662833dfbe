// Eigenvalues of a symmetric tridiagonal matrix in two windows, and the last
// two components of their eigenvectors, on the device: the convergence check
// of the Lanczos runs.
//
// One wavefront per eigenvalue.  The 64 lanes count the eigenvalues below 64
// points of its interval at a time (signs of the leading minors, three-term
// recurrence with rescaling), which cuts the interval by 65 a pass; then two
// lanes run the pivots from both ends, and the eigenvector follows from the
// position where they meet best (twisted factorisation), without inverse
// iteration.  The kernel uses no LDS and few registers, so that it runs beside
// a Lanczos step that fills the LDS of every compute unit.
// Bound by the serial recurrences: about 30 cycles a row and pass (9 passes)
// and 200 cycles a row for the vector: 0.2 ms at 1,100 rows.  On 8 host
// threads (bisection with a division a row, threads started for each check) a
// check took longer than the 25 steps between two of them: a whole solve of
// 3,888 atoms 57 ms, now 26, a mixed one of 172,032 atoms 355 ms, now 241.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace nh {

struct TriWindows {
  double lo[2], hi[2];
  int want[2];  // at most so many: the highest of window 0, the lowest of 1
};
// results: kTriHead doubles (eigenvalues taken of windows 0, 1), then 3 a
// wavefront: value, last and last but one component
constexpr int kTriHead = 2, kTriOut = 3;

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

// S: 2 m doubles a wavefront (stride ld)
__global__ __launch_bounds__(64) void k_tri_windows(int m, const double *__restrict__ a,
                                                    const double *__restrict__ b,
                                                    TriWindows win, double *S, int64_t ld,
                                                    double *__restrict__ out) {
  const int lane = threadIdx.x;
  const int w = (int)blockIdx.x >= win.want[0], j = (int)blockIdx.x - (w ? win.want[0] : 0);
  // numbers of the eigenvalues in the window, and this wavefront's
  int k, n;
  double lo = win.lo[w], hi = win.hi[w];
  {
    const int c = tri_count(m, a, b, lane == 0 ? lo : hi);
    const int klo = __shfl(c, 0, 64), khi = __shfl(c, 1, 64);
    n = min(khi - klo, win.want[w]);
    k = w == 0 ? khi - n + j : klo + j;
    if (j == 0 && lane == 0) out[w] = n > 0 ? (double)n : 0.0;
  }
  if (j >= n) return;
  for (int it = 0; it < 64 && hi - lo > 1e-13; ++it) {
    const double h = (hi - lo) / 65.0;
    const double x = __builtin_fma(h, lane + 1.0, lo);
    const uint64_t above = __ballot(tri_count(m, a, b, x) > k);
    const int l = above ? __builtin_ctzll(above) : 64;  // first point above it
    const double nlo = l > 0 ? __builtin_fma(h, (double)l, lo) : lo;
    const double nhi = l < 64 ? __builtin_fma(h, l + 1.0, lo) : hi;
    if (!(nhi - nlo < hi - lo)) break;
    lo = nlo;
    hi = nhi;
  }
  const double v = 0.5 * (lo + hi);

  // pivots from the front (lane 0) and from the back (lane 1)
  double *F = S + (int64_t)blockIdx.x * ld, *B = F + m;
  if (lane < 2) {
    double q = 0.0;
    double *to = lane ? B : F;
    constexpr int kU = 8;
    double d[kU], e[kU];
    auto load = [&](int t0) {
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int t = min(t0 + u, m - 1), i = lane ? m - 1 - t : t;
        d[u] = a[i];
        e[u] = t == 0 ? 0.0 : b[lane ? i : i - 1];
      }
    };
    load(0);
    for (int t0 = 0; t0 < m; t0 += kU) {
      double dc[kU], ec[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) dc[u] = d[u], ec[u] = e[u];
      load(t0 + kU);
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int t = t0 + u;
        if (t < m) {
          q = dc[u] - v - (t == 0 ? 0.0 : ec[u] * ec[u] / q);
          if (q == 0.0) q = 1e-300;
          to[lane ? m - 1 - t : t] = q;
        }
      }
    }
  }
  __syncthreads();
  // where they meet best
  double best = INFINITY;
  int r = 0;
  for (int i = lane; i < m; i += 64) {
    const double g = fabs(F[i] + B[i] - (a[i] - v));
    if (g < best) {
      best = g;
      r = i;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double g = __shfl_xor(best, off, 64);
    const int o = __shfl_xor(r, off, 64);
    if (g < best || (g == best && o < r)) {
      best = g;
      r = o;
    }
  }
  // component ratios away from it
  __syncthreads();
  for (int i = lane; i < m; i += 64) {
    if (i < r) F[i] = -b[i] / F[i];
    else if (i > r) F[i] = -b[i - 1] / B[i];
  }
  __syncthreads();
  double x = 1.0, x1 = 1.0, sum = 0.0, first = 0.0;  // lane 0 down, lane 1 up from r
  if (lane < 2) {
    const int cnt = lane ? m - 1 - r : r;
    constexpr int kU = 8;
    double q[kU];
    auto load = [&](int t0) {
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int t = t0 + u;
        q[u] = t < cnt ? F[lane ? r + 1 + t : r - 1 - t] : 0.0;
      }
    };
    load(0);
    for (int t0 = 0; t0 < cnt; t0 += kU) {
      double c[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) c[u] = q[u];
      load(t0 + kU);
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (t0 + u < cnt) {
          x1 = x;
          x *= c[u];
          sum = __builtin_fma(x, x, sum);
          if (t0 + u == 0) first = x;
        }
    }
  }
  const double norm = sqrt(1.0 + __shfl(sum, 0, 64) + __shfl(sum, 1, 64));
  const double last = __shfl(x, 1, 64);  // 1 if r is the last row
  const double before = r == m - 1 ? __shfl(first, 0, 64) : __shfl(x1, 1, 64);
  if (lane == 0) {
    double *o = out + kTriHead + (int64_t)blockIdx.x * kTriOut;
    o[0] = v;
    o[1] = last / norm;
    o[2] = m >= 2 ? before / norm : 0.0;
  }
}

}  // namespace nh
