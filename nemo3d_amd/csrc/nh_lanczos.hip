// Device-resident Lanczos eigensolver (no reorthogonalisation), the
// counterpart of eigensolve_lanczos (NEMO_3D/eigen/src/lanczos.c:1823-2089).
//
// One iteration (single_lanczos_iteration, lanczos.c:421-757) is two fused
// kernels plus two one-workgroup reductions, all on one stream:
//   k_lz_hv     q = r / beta_{k-1} (written into a ring slot), y = H q, and
//               per-workgroup partials of alpha = Re<q, y>;
//   k_lz_update r = y - alpha q - beta_{k-1} q_prev with partials of |r|^2.
// In the SK and matrix-free layouts it is one kernel (k_lz_sk, Paige's order;
// FP32 products keep FP32 vectors): the product sums the previous step's
// partials to alpha_{k-1} and beta_k, forms r_k from u_{k-1} and r_{k-1} as it
// reads them, computes u_k = H q_k - beta_k q_{k-1} and the partials of
// alpha_k and beta_{k+1} (LzPart3).
// The reference's REDUCE_OPT variant of the iteration (lanczos.c:441-456)
// defers the vector update into the next iteration in the same spirit, to
// merge its two reductions into one.
// alpha and beta stay in device arrays; every ConvCheckSkipRate iterations
// the tridiagonal is analysed on a second stream (k_tri_windows, nh_tri.h:
// eigenvalues in the Erange windows, convergence by the trailing components
// of the tridiagonal eigenvector, find_converged_eigval Method 2,
// lanczos.c:764-996).  Eigenvectors come from a second pass over the same
// recurrence (eigenvectorsLanczos, lanczos.c:1364-1689): the Lanczos
// vectors land in a ring (K = 128 steps, fewer when memory is short) and
// every K iterations one kernel adds Ring * Z to the eigenvector block.
// The second pass reuses alpha and beta, so with the SK and matrix-free layouts
// its H*v kernel writes r_{k+1} straight into the ring (no reductions), and the
// ring holds the r vectors themselves.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <type_traits>
#include <vector>

#include "nh_hv_row.h"
#include "nh_hv_sk.h"
#include "nh_tri.h"
#include "nh_vector.h"

namespace nh {
namespace {

constexpr int kRingMax = 128;
constexpr int kMaxVec = 64;

template <int WAVES, int NSP, typename TB, typename TA>
__global__ __launch_bounds__(64 * WAVES, 3) void k_lz_hv(
    int A, const double *__restrict__ onsite, const TB *__restrict__ blocks,
    const int32_t *__restrict__ nbr, const double2 *__restrict__ R,
    double2 *__restrict__ Q, double2 *__restrict__ Y,
    const double *__restrict__ beta_prev, double *__restrict__ part) {
  constexpr int NB = NSP * 10;
  __shared__ RowLds<NSP, TB> L[WAVES];
  __shared__ double sums[WAVES];
  const int wave = threadIdx.x >> 6;
  const int a0 = (blockIdx.x * WAVES + wave) * kRowAtoms;
  const double inv = beta_prev ? 1.0 / beta_prev[0] : 1.0;
  double local = 0.0;
  if (a0 < A) {
    double acc_re[NSP], acc_im[NSP];
    double2 xi[NSP];
    const Rows<NSP, TB> rows(a0, A, blocks, nbr);
    rows.template apply<TA>(onsite, 0.0, R, L[wave], acc_re, acc_im, xi);
    if (rows.atom >= 0) {
      const int64_t base = (int64_t)rows.atom * NB + rows.o;
#pragma unroll
      for (int s = 0; s < NSP; ++s) {
        const double2 q = make_double2(xi[s].x * inv, xi[s].y * inv);
        const double2 y = make_double2(acc_re[s] * inv, acc_im[s] * inv);
        if (Q) Q[base + s * 10] = q;
        Y[base + s * 10] = y;
        local += q.x * y.x + q.y * y.y;
      }
    }
  }
  if (part) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) local += __shfl_down(local, off, 64);
    if ((threadIdx.x & 63) == 0) sums[wave] = local;
    __syncthreads();
    if (threadIdx.x == 0) {
      local = 0.0;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) local += sums[w];
      part[blockIdx.x] = local;
    }
  }
}
// Wavefronts of a workgroup of k_lz_hv: four, and up to eight where with more
// the compute units take the atoms in one round (one workgroup on each; a
// second one on some of them holds up the whole step: 60 steps, FP64, 6,720
// atoms 1475 us with four, 1379 with six; 9,984 atoms 1666, with eight 1594).
inline int hv_waves(int A) {
  for (int w : {4, 6, 8})
    if ((A + w * kRowAtoms - 1) / (w * kRowAtoms) <= 256) return w;
  return 4;
}

// One element of the three-term step y - alpha q - beta_prev q_prev with
// q_prev = r_prev * (1 / beta_prev2); rp null on the first step.  The
// operations are spelled out (explicit fma, y kept opaque) so that the
// separate update kernel and the H*v kernel of the eigenvector pass, which
// fuses the step, round identically: the second pass must retrace the first
// pass's trajectory bit for bit.
__device__ __forceinline__ double2 lz_three_term_v(double2 y, double2 q,
                                                   bool has_p, double2 r,
                                                   double al, double be,
                                                   double invp) {
  asm volatile("" : "+v"(y.x), "+v"(y.y));
  if (has_p) {
    const double2 p = make_double2(r.x * invp, r.y * invp);
    y.x = y.x - __builtin_fma(al, q.x, be * p.x);
    y.y = y.y - __builtin_fma(al, q.y, be * p.y);
  } else {
    y.x = __builtin_fma(-al, q.x, y.x);
    y.y = __builtin_fma(-al, q.y, y.y);
  }
  return y;
}
// the same step with r_prev read from rp (null: first step; FP64 or FP32
// storage)
template <typename XO>
__device__ __forceinline__ double2 lz_three_term(double2 y, double2 q,
                                                 const XO *rp, double al,
                                                 double be, double invp) {
  return lz_three_term_v(y, q, rp != nullptr,
                         rp ? widen2(*rp) : make_double2(0.0, 0.0), al, be, invp);
}

// Paige's order of the step: u_k = H q_k - beta_k q_{k-1} (FP64 arithmetic,
// rounded once to FP32 vectors), alpha_k = <q_k, u_k>, r_{k+1} = u_k -
// alpha_k q_k (lz_defer1).
__device__ __forceinline__ double lz_u(double y, double rp, double be, double invp) {
  return __builtin_fma(-be, rp * invp, y);
}
// partials of an eigenvalue-pass step: with w = u_k - sigma_k q_k, <q_k, w>,
// |w|^2 and |q_k|^2 (lz_alpha_beta).  sigma_k = alpha_{k-1}: u's part along q_k
// is gone but for alpha_k - alpha_{k-1}, and beta as exact as from |r_{k+1}|^2
// (600 steps, N = 20,000: 7.5e-17 root mean square against 8.5e-17; without
// sigma 1.9e-16, and 8e-14 with H shifted by 300 eV)
struct LzPart3 {
  double a = 0.0, w2 = 0.0, q2 = 0.0;
  __device__ __forceinline__ void add(double sigma, double qv, double uv) {
    const double w = __builtin_fma(-sigma, qv, uv);
    a = __builtin_fma(qv, w, a);
    w2 = __builtin_fma(w, w, w2);
    q2 = __builtin_fma(qv, qv, q2);
  }
};
// alpha_k = <q, u> and beta_{k+1}^2 = |u - alpha_k q|^2 from the partials' sums;
// d: <q, u> - sigma
__device__ __forceinline__ void lz_alpha_beta(const double (&s)[3], double sigma, double &alpha,
                                              double &beta) {
  const double d = __builtin_fma(sigma, s[2] - 1.0, s[0]);
  alpha = sigma + d;
  beta = sqrt(fmax(__builtin_fma(d, __builtin_fma(d, s[2], -2.0 * s[0]), s[1]), 0.0));
}
// sums of three values over a workgroup of kRedThreads in a fixed order, in
// every thread; scratch: 3 * kRedThreads / 64 doubles
__device__ __forceinline__ void lz_block_sum3(double (&s)[3], double *scratch) {
  constexpr int kWaves = kRedThreads / 64;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s[c] += __shfl_xor(s[c], off, 64);
    if ((threadIdx.x & 63) == 0) scratch[c * kWaves + (threadIdx.x >> 6)] = s[c];
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    s[c] = scratch[c * kWaves];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) s[c] += scratch[c * kWaves + w];
  }
}
// alpha_k and beta_{k+1} from the partials of nparts workgroups (fixed order:
// every workgroup that evaluates it gets the same bits)
__device__ __forceinline__ void lz_scalars3(int nparts, const double *__restrict__ part,
                                            double sigma, double *scratch, double &alpha,
                                            double &beta) {
  double s[3] = {0.0, 0.0, 0.0};
  for (int k = threadIdx.x; k < nparts; k += kRedThreads)
#pragma unroll
    for (int c = 0; c < 3; ++c) s[c] += part[3 * k + c];
  lz_block_sum3(s, scratch);
  lz_alpha_beta(s, sigma, alpha, beta);
}
__global__ __launch_bounds__(kRedThreads) void k_lz_scalars3(
    int nparts, const double *__restrict__ part, double *__restrict__ alpha,
    double *__restrict__ beta) {
  __shared__ double scratch[3 * kRedThreads / 64];
  double a, b;
  lz_scalars3(nparts, part, alpha[-1], scratch, a, b);
  if (threadIdx.x == 0) {
    alpha[0] = a;
    beta[0] = b;
  }
}

// The SK / matrix-free product of a Lanczos step (block mapping of
// nh_hv_sk.h), V: storage of the vectors.
//  Deferred (Paige's order; FP64 vectors with FP64 products, FP32 vectors
//  with FP32 products):
//   kLzValues  eigenvalue pass, the whole step in one launch: the previous
//     launch's partials give alpha_{k-1}, beta_k (each workgroup sums them,
//     workgroup 0 stores them); r_k = u_{k-1} - .. r_{k-1} is formed from x =
//     u_{k-1} and rp = r_{k-1} as the block is staged, u_k goes to out, r_k to
//     rout, the partials to part;
//   kLzVectors eigenvector pass: x = r_k, rp = r_{k-1}, r_{k+1} to out.
//  Classic (FP64 vectors; products of either precision):
//   kLzProduct eigenvalue pass, before k_lz_update: y = H q_k to out, partials
//     of alpha_k;
//   kLzFused   eigenvector pass: with the three-term step, r_{k+1} to out.
// In both pairs the second pass evaluates the first one's expressions on the
// same operands and so retraces it bit for bit (sk_apply and the step spell
// their multiply-adds out).
// Why deferred: an FP64 step moves H and four vectors (u, r read, u, r
// written) instead of H and six in two launches with two reductions between
// them: 786,520 atoms, SK 0.528 -> 0.366 ms a step, 4,336,640 atoms,
// matrix-free 3.07 -> 2.07 ms, 3,888 atoms 21 -> 10 us.
enum { kLzProduct = 0, kLzFused = 1, kLzValues = 2, kLzVectors = 3 };
template <typename V>
struct LzArgs {
  const V *x, *rp;
  V *out, *rout;
  const double *alpha, *beta_prev, *beta_prev2;  // beta null: 1 (start vector)
  const double *part_prev;  // kLzValues: partials of the previous step (null: none)
  int nparts;
  // .. whose alpha and beta go here; alpha_out[-1]: its sigma, or (no previous
  // step) this one's is alpha_out[0]
  double *alpha_out, *beta_out;
  double *part;
};
template <int MODE, int NSP, typename R, typename V, typename SRC>
__global__ __launch_bounds__(kSkThreads, sizeof(V) == 8 ? 3 : 2) void k_lz_sk(
    SkTable tab, const double *__restrict__ onsite, const SRC src, const LzArgs<V> g) {
  constexpr bool VALUES = MODE == kLzValues, DEFER = MODE >= kLzValues;
  static_assert(DEFER || sizeof(V) == 16, "the classic step keeps FP64 vectors");
  static_assert(sizeof(R) == sizeof(V) / 2 || !DEFER, "deferred vectors have the products' type");
  static_assert(kSkThreads == kRedThreads, "block sums");
  using S = SkX<NSP, V>;
  __shared__ SkLds<NSP, R, V> L;
  const SkThread t;
  SkWalk w(tab);
  const bool cat = __builtin_amdgcn_readfirstlane(t.Q) < kSkOwn / 2;
  uint4 *own = L.x + t.Q * S::kStride, *halo = L.x + (kSkOwn + t.Q) * S::kStride;
  double *scratch = reinterpret_cast<double *>(L.rec);
  double be = g.beta_prev ? g.beta_prev[0] : 0.0;
  double inv = g.beta_prev ? 1.0 / be : 1.0;
  const double invp = g.beta_prev2 ? 1.0 / g.beta_prev2[0] : 1.0;
  const double al = MODE == kLzFused || MODE == kLzVectors ? g.alpha[0] : 0.0;
  SkIndex<SRC> ix;
  if (w.b < w.end) ix.read(tab, src, w.b, t.Q);
  LzCoef<V> ap{};
  double sigma = 0.0;
  if constexpr (VALUES) {
    double alp = 0.0;
    if (!g.part_prev) {
      sigma = g.alpha_out[0];
    } else {
      lz_scalars3(g.nparts, g.part_prev, g.alpha_out[-1], scratch, alp, be);
      sigma = alp;
      inv = 1.0 / be;
      if (blockIdx.x == 0 && threadIdx.x == 0) {
        g.alpha_out[0] = alp;
        g.beta_out[0] = be;
      }
      __syncthreads();  // the scratch is the records' place
    }
    ap = lz_defer_coef<V>(alp, invp);
  }
  const LzCoef<V> af = lz_defer_coef<V>(al, inv);
  LzPart3 p3;
  double local = 0.0;
  while (w.b < w.end) {
    const int atom = ix.own;
    typename SRC::Data rec;
    uint4 xo[S::kLoads], xh[S::kLoads], os[3];
    sk_load_x<NSP>(atom, t.c, g.x, xo);
    sk_load_x<NSP>(ix.halo, t.c, g.x, xh);
    if constexpr (VALUES) {
      uint4 po[S::kLoads], ph[S::kLoads];
      sk_load_x<NSP>(atom, t.c, g.rp, po);
      sk_load_x<NSP>(ix.halo, t.c, g.rp, ph);
      src.load(ix.rec, rec);
      sk_load_onsite(atom, t.c, onsite, os);
      sk_defer<V>(xo, po, ap);
      sk_defer<V>(xh, ph, ap);
      if (g.rout && atom >= 0) {
        uint4 *o = reinterpret_cast<uint4 *>(g.rout) + (int64_t)atom * S::kChunks;
#pragma unroll
        for (int i = 0; i < S::kLoads; ++i)
          if (4 * i + t.c < S::kChunks) o[4 * i + t.c] = xo[i];
      }
    } else {
      src.load(ix.rec, rec);
      sk_load_onsite(atom, t.c, onsite, os);
    }
    const uint2 lc = ix.local;
    const bool surface = sk_surface(atom, lc);
    w.b += w.step;
    if (w.b < w.end) ix.read(tab, src, w.b, t.Q);
    src.stage(rec, L.rec);
    sk_stage_x<NSP, V>(own, t.c, xo);
    sk_stage_x<NSP, V>(halo, t.c, xh);
    __syncthreads();
    double acc[10];
    if (cat) sk_bonds<NSP, R, true, V>(t, lc, L, acc);
    else sk_bonds<NSP, R, false, V>(t, lc, L, acc);
    // own r_{k-1}, requested before the barrier of sk_finish
    constexpr int kSpins = sizeof(V) == 8 ? NSP : 1;      // FP32: a spin at a time
    constexpr int kPer = S::kChunks / kSpins, kPl = (kPer + 3) / 4;
    uint4 rp[kSpins][kPl];
#pragma unroll
    for (int s = 0; s < kSpins; ++s)
#pragma unroll
      for (int i = 0; i < kPl; ++i) {
        rp[s][i] = make_uint4(0, 0, 0, 0);
        if (MODE != kLzProduct && g.rp && atom >= 0 && 4 * i + t.c < kPer)
          rp[s][i] = reinterpret_cast<const uint4 *>(g.rp)[(int64_t)atom * S::kChunks + s * kPer +
                                                           4 * i + t.c];
      }
    sk_finish<NSP, R, V>(t, L, os, 0.0, surface, acc);
    uint4 *out = reinterpret_cast<uint4 *>(g.out) + (int64_t)atom * S::kChunks;
#pragma unroll
    for (int s = 0; s < kSpins; ++s) {
      // entries of y = H r_k in the halo place: all of them, or those of spin s
      if (kSpins == 1 ? NSP == 2 || t.h == 0 : t.h == s)
        sk_entries(halo, t.comp, kSpins == 1 && NSP == 2 ? 10 * t.h : 0, acc);
      wave_sync();
      if (atom >= 0) {
#pragma unroll
        for (int i = 0; i < kPl; ++i) {
          const int q = 4 * i + t.c;
          if (q >= kPer) break;
          const uint4 rk4 = own[S::at(s * kPer + q)];
          uint4 o4;
          if constexpr (sizeof(V) == 16) {
            const double2 y = *reinterpret_cast<const double2 *>(&halo[q]);
            const double2 rk = *reinterpret_cast<const double2 *>(&rk4);
            const double2 rm = *reinterpret_cast<const double2 *>(&rp[s][i]);
            const double2 qk = make_double2(rk.x * inv, rk.y * inv);
            double2 o = make_double2(y.x * inv, y.y * inv);
            if constexpr (MODE == kLzFused) {
              o = lz_three_term_v(o, qk, g.rp != nullptr, rm, al, be, invp);
            } else if constexpr (DEFER) {
              o = make_double2(lz_u(o.x, rm.x, be, invp), lz_u(o.y, rm.y, be, invp));
              if constexpr (MODE == kLzVectors) {
                o = make_double2(lz_defer1(o.x, rk.x, af), lz_defer1(o.y, rk.y, af));
              } else {
                p3.add(sigma, qk.x, o.x);
                p3.add(sigma, qk.y, o.y);
              }
            } else {
              local += qk.x * o.x + qk.y * o.y;
            }
            o4 = *reinterpret_cast<const uint4 *>(&o);
          } else {
            const float *rk = reinterpret_cast<const float *>(&rk4);
            const float *rm = reinterpret_cast<const float *>(&rp[s][i]);
            const double *y = reinterpret_cast<const double *>(&halo[2 * q]);
            float *o = reinterpret_cast<float *>(&o4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float u = (float)lz_u(y[e] * inv, (double)rm[e], be, invp);
              if constexpr (MODE == kLzVectors) {
                o[e] = lz_defer1(u, rk[e], af);
              } else {
                o[e] = u;
                p3.add(sigma, (double)rk[e] * inv, (double)u);
              }
            }
          }
          out[s * kPer + q] = o4;
        }
      }
      wave_sync();
    }
  }
  if constexpr (VALUES || MODE == kLzProduct) {
    double s[3] = {VALUES ? p3.a : local, p3.w2, p3.q2};
    __syncthreads();  // the last block's records have been read
    lz_block_sum3(s, scratch);
    if (threadIdx.x == 0) {
      if constexpr (VALUES) {
#pragma unroll
        for (int c = 0; c < 3; ++c) g.part[3 * blockIdx.x + c] = s[c];
      } else {
        g.part[blockIdx.x] = s[0];
      }
    }
  }
}

// y <- y - alpha q - beta_prev q_prev with q = r * (1 / beta_prev) and
// q_prev = r_prev * (1 / beta_prev2) formed on the fly (the same products
// as the fused H·v kernel's q, so the trajectory does not depend on whether
// q was stored), partial sums of |y|^2.  Rp may be null (first step), and
// beta_prev / beta_prev2 null mean 1 (the start vector is normalised).
__global__ __launch_bounds__(kRedThreads) void k_lz_update(
    int64_t n, double2 *__restrict__ Y, const double2 *__restrict__ Rk,
    const double2 *__restrict__ Rp, const double *__restrict__ alpha,
    const double *__restrict__ beta_prev, const double *__restrict__ beta_prev2,
    double *__restrict__ part) {
  const double al = alpha[0];
  const double be = beta_prev ? beta_prev[0] : 0.0;
  const double inv = beta_prev ? 1.0 / beta_prev[0] : 1.0;
  const double invp = beta_prev2 ? 1.0 / beta_prev2[0] : 1.0;
  double s = 0.0, z = 0.0;
  for (int64_t k = blockIdx.x * (int64_t)kRedThreads + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * kRedThreads) {
    const double2 r = Rk[k];
    const double2 q = make_double2(r.x * inv, r.y * inv);
    const double2 y = lz_three_term(Y[k], q, Rp ? Rp + k : nullptr, al, be, invp);
    Y[k] = y;
    s += y.x * y.x + y.y * y.y;
  }
  if (part) {
    block_sum2(s, z);
    if (threadIdx.x == 0) part[2 * blockIdx.x] = s;
  }
}

// out[0] = sum of nparts partials (stride `stride`); sqrt if take_sqrt.
__global__ __launch_bounds__(kRedThreads) void k_lz_scalar(
    int nparts, int stride, const double *__restrict__ part,
    double *__restrict__ out, int take_sqrt) {
  // eight independent partial sums per thread (all loads of a trip in
  // flight together), combined in a fixed order
  double p[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  int k = threadIdx.x;
  for (; k + 7 * kRedThreads < nparts; k += 8 * kRedThreads) {
#pragma unroll
    for (int u = 0; u < 8; ++u) p[u] += part[(k + u * kRedThreads) * stride];
  }
  for (int u = 0; k < nparts; k += kRedThreads, ++u) p[u & 7] += part[k * stride];
  double a = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7])), b = 0.0;
  block_sum2(a, b);
  if (threadIdx.x == 0) out[0] = take_sqrt ? sqrt(a) : a;
}

// V[e] += sum_k Z[e][k] Ring[k] for e < ne, k < K <= kRingMax (ring of
// FP64 q or of the FP32 copies of r).  Eight eigenvectors at a time stay in
// registers while the ring streams past in groups of eight slots.
template <typename T>
__global__ __launch_bounds__(256) void k_lz_accum(
    int64_t n, int ne, int K, const double *__restrict__ Z,
    const T *__restrict__ ring, int64_t ring_ld, double2 *__restrict__ V,
    int64_t v_ld) {
  __shared__ double zs[8 * kRingMax];
  const int K8 = (K + 7) / 8 * 8;
  for (int e0 = 0; e0 < ne; e0 += 8) {
    const int nb = min(8, ne - e0);
    __syncthreads();
    for (int t = threadIdx.x; t < 8 * K8; t += blockDim.x) {
      const int e = t / K8, k = t % K8;
      zs[t] = e < nb && k < K ? Z[(e0 + e) * K + k] : 0.0;
    }
    __syncthreads();
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
      double2 v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e)
        v[e] = e < nb ? V[(int64_t)(e0 + e) * v_ld + i] : make_double2(0.0, 0.0);
      for (int k0 = 0; k0 < K8; k0 += 8) {
        double2 q[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          q[j] = make_double2(0.0, 0.0);
          if (k0 + j < K) {
            const T r = ring[(int64_t)(k0 + j) * ring_ld + i];
            q[j] = make_double2(r.x, r.y);
          }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const double z = zs[e * K8 + k0 + j];
            v[e].x += z * q[j].x;
            v[e].y += z * q[j].y;
          }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e < nb) V[(int64_t)(e0 + e) * v_ld + i] = v[e];
    }
  }
}

// The FP32 ring (copies of r) accumulated two rows per thread, so each
// ring load is 16 bytes; n even.
__global__ __launch_bounds__(256) void k_lz_accum32(
    int64_t n, int ne, int K, const double *__restrict__ Z,
    const float2 *__restrict__ ring, int64_t ring_ld, double2 *__restrict__ V,
    int64_t v_ld) {
  __shared__ double zs[8 * kRingMax];
  const int K8 = (K + 7) / 8 * 8;
  const int64_t n2 = n / 2;
  const float4 *r4 = reinterpret_cast<const float4 *>(ring);
  const int64_t ld4 = ring_ld / 2;
  for (int e0 = 0; e0 < ne; e0 += 8) {
    const int nb = min(8, ne - e0);
    __syncthreads();
    for (int t = threadIdx.x; t < 8 * K8; t += blockDim.x) {
      const int e = t / K8, k = t % K8;
      zs[t] = e < nb && k < K ? Z[(e0 + e) * K + k] : 0.0;
    }
    __syncthreads();
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n2;
         i += (int64_t)gridDim.x * blockDim.x) {
      double2 v0[8], v1[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        v0[e] = v1[e] = make_double2(0.0, 0.0);
        if (e < nb) {
          v0[e] = V[(int64_t)(e0 + e) * v_ld + 2 * i];
          v1[e] = V[(int64_t)(e0 + e) * v_ld + 2 * i + 1];
        }
      }
      for (int k0 = 0; k0 < K8; k0 += 8) {
        float4 q[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          q[j] = k0 + j < K ? r4[(int64_t)(k0 + j) * ld4 + i] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const double z = zs[e * K8 + k0 + j];
            v0[e].x += z * (double)q[j].x;
            v0[e].y += z * (double)q[j].y;
            v1[e].x += z * (double)q[j].z;
            v1[e].y += z * (double)q[j].w;
          }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e < nb) {
          V[(int64_t)(e0 + e) * v_ld + 2 * i] = v0[e];
          V[(int64_t)(e0 + e) * v_ld + 2 * i + 1] = v1[e];
        }
    }
  }
}

__global__ void k_scale(int64_t n, double2 *__restrict__ x, double s) {
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * blockDim.x) {
    x[k].x *= s;
    x[k].y *= s;
  }
}

// ---------------- host-side tridiagonal analysis ---------------------------

// Eigenvector of T_m at lambda by inverse iteration (tridiagonal Gaussian
// elimination with partial pivoting), from a fixed pseudo-random start.
void tri_eigvec(const std::vector<double> &d, const std::vector<double> &e,
                int m, double lambda, std::vector<double> &x) {
  x.assign(m, 0.0);
  uint64_t s = 0x9E3779B97F4A7C15ull;
  for (int i = 0; i < m; ++i) {
    s = s * 6364136223846793005ull + 1442695040888963407ull;
    x[i] = 0.5 + (double)(s >> 11) * (1.0 / 9007199254740992.0);
  }
  const double pert = 1e-13 * (std::fabs(lambda) + 1.0);
  std::vector<double> a(m), b(m), c(m), c2(m), rhs(m);
  std::vector<char> swapped(m);
  for (int sweep = 0; sweep < 3; ++sweep) {
    // (T - lambda') x_new = x with a tridiagonal LU (a: sub, b: diag, c: sup)
    for (int i = 0; i < m; ++i) {
      b[i] = d[i] - lambda - pert;
      a[i] = i > 0 ? e[i - 1] : 0.0;
      c[i] = i + 1 < m ? e[i] : 0.0;
      c2[i] = 0.0;
      rhs[i] = x[i];
    }
    for (int i = 0; i + 1 < m; ++i) {
      // rows i and i+1; eliminate a[i+1]
      if (std::fabs(a[i + 1]) > std::fabs(b[i])) {
        std::swap(b[i], a[i + 1]);
        std::swap(c[i], b[i + 1]);
        std::swap(c2[i], c[i + 1]);
        std::swap(rhs[i], rhs[i + 1]);
      }
      if (b[i] == 0.0) b[i] = 1e-300;
      const double f = a[i + 1] / b[i];
      b[i + 1] -= f * c[i];
      c[i + 1] -= f * c2[i];
      rhs[i + 1] -= f * rhs[i];
    }
    if (b[m - 1] == 0.0) b[m - 1] = 1e-300;
    x[m - 1] = rhs[m - 1] / b[m - 1];
    if (m > 1) x[m - 2] = (rhs[m - 2] - c[m - 2] * x[m - 1]) / b[m - 2];
    for (int i = m - 3; i >= 0; --i)
      x[i] = (rhs[i] - c[i] * x[i + 1] - c2[i] * x[i + 2]) / b[i];
    double nrm = 0.0;
    for (int i = 0; i < m; ++i) nrm += x[i] * x[i];
    nrm = std::sqrt(nrm);
    for (int i = 0; i < m; ++i) x[i] /= nrm;
  }
}

struct Converged {
  double value;
  int iter;
  int window;
};

class LanczosRun {
 public:
  // classic: no deferred step
  LanczosRun(nh_context *c, bool classic) : c_(c), classic_(classic) {}
  ~LanczosRun() {
    release_events();
    // a check that nobody waited for (error returns) still uses the buffers
    if (c_->side) (void)hipStreamSynchronize(c_->side);
    for (void *p : allocs_) pool_release(c_, p);
    if (tri_s_) pool_release(c_, tri_s_);
    if (pin_) (void)hipHostFree(pin_);
    for (hipEvent_t e : {fetch_ev_, check_ev_, look_ev_})
      if (e) (void)hipEventDestroy(e);
  }
  nh_status run(const nh_lanczos_opts *o, nh_eig_result *res);
  // run() ended because the deferred step's beta has lost digits
  bool small_beta() const { return small_beta_; }
  // a restart's vectors are not those of its tridiagonal
  bool stale() const { return stale_; }
  int matvecs() const { return matvecs_; }

 private:
  // from the context's workspace pool, handed back when the run ends
  nh_status alloc(void **p, size_t bytes) {
    NH_TRY(pool_alloc(c_, p, bytes));
    allocs_.push_back(*p);
    return NH_OK;
  }
  void release(void *p) {
    pool_release(c_, p);
    allocs_.erase(std::remove(allocs_.begin(), allocs_.end(), p), allocs_.end());
  }
  nh_status iterate(int k, bool with_reductions);
  nh_status collect_timing();
  nh_status fetch(int m);
  nh_status check(int m);
  nh_status look(bool wait);
  // whether the deferred step's beta_i has lost digits (LzPart3)
  static bool lost(double sigma, double alpha, double beta) {
    const double d = alpha - sigma;
    return !(beta * beta >= 0.125 * (d * d + beta * beta));
  }
  hipStream_t check_stream() const { return alone_ ? c_->stream : c_->side; }
  bool alone_ = false;
  nh_status analyse(int m, const nh_lanczos_opts *o);
  bool window_done(int w, int req, int rule) const;

  nh_context *c_;
  bool classic_;
  std::vector<void *> allocs_;
  int64_t n_ = 0;
  double2 *R_ = nullptr, *Y_ = nullptr, *Rm1_ = nullptr, *ring_ = nullptr;
  // SK and matrix-free layouts: the deferred step (k_lz_sk), with vectors of
  // the products' type (vbytes_ an entry).  The eigenvalue pass keeps r_{k-1},
  // u_{k-1} in r_[0], u_[0] and writes r_k, u_k to r_[1], u_[1]; part_ holds
  // the partials of two steps in turn, grid_ of each.
  bool defer_ = false, small_beta_ = false, stale_ = false;
  size_t vbytes_ = sizeof(double2);
  char *r_[2] = {nullptr, nullptr}, *u_[2] = {nullptr, nullptr};
  int waves_ = 4;  // of a workgroup of k_lz_hv
  int grid_ = 0, last_ = -1;  // the last step of the eigenvalue pass queued
  // ring length of the eigenvector pass (<= kRingMax)
  int ring_k_ = kRingMax;
  // SK and matrix-free layouts: the eigenvector pass keeps the r vectors
  // themselves in 2 K slots, slot k % (2 K) holding r_k: read as own entries
  // and gathered at step k, r_(k-1) from slot k - 1, r_(k+1) written to slot
  // k + 1; the accumulation reads them as its ring (1 / beta_{k-1} folded into
  // the coefficients), so no q is stored
  char *ringr_ = nullptr;
  char *slot(int k) const { return ringr_ + (size_t)((k + 2 * ring_k_) % (2 * ring_k_)) * n_ * vbytes_; }
  template <int NSP, typename R, typename V, typename SRC>
  void launch_sk(int k, bool red, const SRC &src);
  template <int NSP>
  void launch_sk(int k, bool red);
  nh_status build_start(const nh_lanczos_opts *o);
  nh_status upload_start(void *r, size_t bytes);
  double2 *R0_ = nullptr;  // the normalised start vector (device)
  double *alpha_ = nullptr, *beta_ = nullptr, *part_ = nullptr;  // (alpha_[-1]: sigma_0)
  int nparts_ = 0;
  std::vector<double> ha_, hb_;
  // pinned staging of sigma_0 and alpha, of beta (pin_cap_ each, filled up to
  // fetched_) and of the last check's results; fetch_ev_: alpha and beta are there on the
  // context's stream, check_ev_: the check of checked_ steps is done
  double *pin_ = nullptr;
  int pin_cap_ = 0, fetched_ = 0;
  hipEvent_t fetch_ev_ = nullptr, check_ev_ = nullptr, look_ev_ = nullptr;
  int matvecs_ = 0;
  int checked_ = 0;
  TriWindows win_{};
  // no more eigenvalues are asked for than T_m has
  TriWindows win_at(int m) const {
    TriWindows w = win_;
    for (int &n : w.want) n = std::min(n, m);
    return w;
  }
  double *tri_out_ = nullptr, *tri_s_ = nullptr;  // results, scratch of the check
  int64_t tri_cap_ = 0;                           // doubles in tri_s_
  std::vector<Converged> conv_;
  std::vector<double> lastRitz_[2];
  std::vector<char> lastConv_[2];
  // sampled H·v timing: one event pair every kTimeEvery iterations, per
  // pass (eigenvalue pass, eigenvector pass)
  static constexpr int kTimeEvery = 16;
  struct Timed {
    hipEvent_t start, stop;
    bool value_pass;
  };
  std::vector<Timed> ev_;
  double hv_ms_sum_[2] = {0.0, 0.0};
  int hv_timed_[2] = {0, 0};

 public:
  // pass 0: eigenvalue pass, 1: eigenvector pass
  double hv_ms(int pass = 0) const {
    return hv_timed_[pass] ? hv_ms_sum_[pass] / hv_timed_[pass] : 0.0;
  }
  int hv_timed(int pass = 0) const { return hv_timed_[pass]; }
  void release_events() {
    for (auto &e : ev_) {
      (void)hipEventDestroy(e.start);
      (void)hipEventDestroy(e.stop);
    }
    ev_.clear();
  }
};

nh_status LanczosRun::collect_timing() {
  NH_HIP(hipStreamSynchronize(c_->stream));
  for (auto &e : ev_) {
    float ms = 0.f;
    NH_HIP(hipEventElapsedTime(&ms, e.start, e.stop));
    const int pass = e.value_pass ? 0 : 1;
    hv_ms_sum_[pass] += ms;
    ++hv_timed_[pass];
  }
  release_events();
  return NH_OK;
}

__global__ __launch_bounds__(256) void k_to_f32(int64_t n,
                                                const double2 *__restrict__ x,
                                                float2 *__restrict__ y) {
  for (int64_t k = blockIdx.x * (int64_t)256 + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * 256)
    y[k] = make_float2((float)x[k].x, (float)x[k].y);
}

// start vector (lanczos_initialize, eigsys3d_par.c:113-215) built and
// normalised in device memory: CyclicRandom r0[j] = (s[2j mod L],
// s[2j+1 mod L]), Const1 (1, 1), or a caller's host or device vector
__global__ __launch_bounds__(256) void k_start_fill(int64_t n, int kind, int L,
                                                   const double *__restrict__ cyc,
                                                   double2 *__restrict__ r) {
  for (int64_t j = blockIdx.x * (int64_t)256 + threadIdx.x; j < n;
       j += (int64_t)gridDim.x * 256)
    r[j] = kind == 0 ? make_double2(cyc[(2 * j) % L], cyc[(2 * j + 1) % L])
                     : make_double2(1.0, 1.0);
}
// (and sigma_0, see LzPart3: the mean diagonal entry of 256 atoms)
__global__ __launch_bounds__(256) void k_div(int64_t n, double2 *__restrict__ r,
                                             double s, int A, const double *__restrict__ onsite,
                                             double *__restrict__ sigma) {
  for (int64_t j = blockIdx.x * (int64_t)256 + threadIdx.x; j < n;
       j += (int64_t)gridDim.x * 256)
    r[j] = make_double2(r[j].x / s, r[j].y / s);
  if (blockIdx.x == 0) {
    const double *os = onsite + (int64_t)threadIdx.x * A / 256 * kOnsiteStride;
    double d = 0.0, z = 0.0;
#pragma unroll
    for (int k = 0; k < 10; ++k) d += os[k];
    block_sum2(d, z);
    if (threadIdx.x == 0) sigma[0] = d / 2560.0;
  }
}

nh_status LanczosRun::build_start(const nh_lanczos_opts *o) {
  NH_TRY(alloc((void **)&R0_, n_ * sizeof(double2)));
  const int g = reduce_blocks(n_);
  if (o->start == 0 || o->start == 1) {
    double *cyc = nullptr;
    int L = 1;
    if (o->start == 0) {
      NH_CHECK(o->cyclic_len > 0 && o->cyclic_string, NH_ERR_ARG,
               "CyclicRandom start needs CyclicString");
      L = o->cyclic_len;
      NH_TRY(alloc((void **)&cyc, (size_t)L * sizeof(double)));
      NH_HIP(hipMemcpyAsync(cyc, o->cyclic_string, (size_t)L * sizeof(double),
                            hipMemcpyHostToDevice, c_->stream));
    }
    hipLaunchKernelGGL(k_start_fill, dim3(g), dim3(256), 0, c_->stream, n_,
                       o->start, L, cyc, R0_);
    NH_HIP(hipGetLastError());
    // the host CyclicString may be released on return
    NH_HIP(hipStreamSynchronize(c_->stream));
  } else if (o->start == 4) {
    // Random: glibc rand() after srand(random_seed), drawn on the host in
    // the reference's order (one number per entry, real part)
    std::vector<nh_cplx> h((size_t)n_);
    rand_start(o->random_seed, n_, h.data());
    NH_HIP(hipMemcpyAsync(R0_, h.data(), n_ * sizeof(double2),
                          hipMemcpyHostToDevice, c_->stream));
    NH_HIP(hipStreamSynchronize(c_->stream));  // h is released on return
  } else {
    NH_CHECK(o->start == 2 || o->start == 3, NH_ERR_ARG, "bad start %d", o->start);
    NH_CHECK(o->start_vector, NH_ERR_ARG, "start vector missing");
    NH_HIP(hipMemcpyAsync(R0_, o->start_vector, n_ * sizeof(double2),
                          o->start == 2 ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice,
                          c_->stream));
  }
  double s = 0.0;
  NH_TRY(reduce_nrm2sq(c_, n_, reinterpret_cast<const nh_cplx *>(R0_), &s));
  NH_CHECK(s > 0, NH_ERR_ARG, "zero start vector");
  hipLaunchKernelGGL(k_div, dim3(g), dim3(256), 0, c_->stream, n_, R0_, std::sqrt(s),
                     c_->n_atoms, c_->onsite, alpha_ - 1);
  NH_HIP(hipGetLastError());
  return NH_OK;
}

// r <- r0 as FP64 or FP32 entries
nh_status LanczosRun::upload_start(void *r, size_t bytes) {
  if (bytes == sizeof(double2)) {
    NH_HIP(hipMemcpyAsync(r, R0_, n_ * sizeof(double2), hipMemcpyDeviceToDevice,
                          c_->stream));
  } else {
    hipLaunchKernelGGL(k_to_f32, dim3(reduce_blocks(n_)), dim3(256), 0,
                       c_->stream, n_, R0_, reinterpret_cast<float2 *>(r));
    NH_HIP(hipGetLastError());
  }
  return NH_OK;
}

// One product of the SK / matrix-free layouts in the run's mode.
// Eigenvalue pass, step 0 of the deferred step: u_{-1} = r_{-1} = r_0 with
// alpha_{-1} = beta_0 = 0, which leaves r_0 as it is; nothing is written back
// for it.  Eigenvector pass: r_{-1} is slot 0 itself (the eigenvalue pass's
// operands), none in the classic step.
template <int NSP, typename R, typename V, typename SRC>
void LanczosRun::launch_sk(int k, bool red, const SRC &src) {
  nh_context *c = c_;
  LzArgs<V> g{};
  g.alpha = alpha_ + k;
  g.beta_prev = k > 0 ? beta_ + (k - 1) : nullptr;
  g.beta_prev2 = k > 1 ? beta_ + (k - 2) : nullptr;
  g.part = part_ + (size_t)(k & 1) * 3 * nparts_;
  auto vec = [](char *p) { return reinterpret_cast<V *>(p); };
  if (red && defer_) {
    g.x = vec(k == 0 ? r_[0] : u_[0]);
    g.rp = vec(r_[0]);
    g.out = vec(u_[1]);
    g.rout = k == 0 ? nullptr : vec(r_[1]);
    g.beta_prev = nullptr;  // summed by this launch
    g.alpha_out = alpha_ + (k - 1);
    g.beta_out = beta_ + (k - 1);
    if (k > 0) {
      g.part_prev = part_ + (size_t)((k - 1) & 1) * 3 * nparts_;
      g.nparts = grid_;
    }
  } else if (red) {
    g.x = reinterpret_cast<V *>(R_);
    g.out = reinterpret_cast<V *>(Y_);
    g.part = part_;
  } else {
    g.x = vec(slot(k));
    g.rp = k > 0 ? vec(slot(k - 1)) : defer_ ? g.x : nullptr;
    g.out = vec(slot(k + 1));
  }
  const SkTable tab = sk_table_of(c);
#define LZ_SK(MODE)                                                            \
  hipLaunchKernelGGL((k_lz_sk<MODE, NSP, R, V, SRC>), dim3(grid_),             \
                     dim3(kSkThreads), 0, c->stream, tab, c->onsite, src, g)
  if constexpr (sizeof(V) == 2 * sizeof(R)) {
    if (defer_) {
      if (red) LZ_SK(kLzValues);
      else LZ_SK(kLzVectors);
      return;
    }
  }
  if constexpr (sizeof(V) == 16) {
    if (red) LZ_SK(kLzProduct);
    else LZ_SK(kLzFused);
  }
#undef LZ_SK
}

template <int NSP>
void LanczosRun::launch_sk(int k, bool red) {
  nh_context *c = c_;
  const bool f64 = c->precision == NH_PREC_FP64, v64 = vbytes_ == sizeof(double2);
#define LZ_SRC(S64, S32)                                                       \
  do {                                                                         \
    if (f64) launch_sk<NSP, double, double2>(k, red, S64);                     \
    else if (v64) launch_sk<NSP, float, double2>(k, red, S32);                 \
    else launch_sk<NSP, float, float2>(k, red, S32);                           \
  } while (0)
  if (c->layout == NH_LAYOUT_MATRIX_FREE)
    LZ_SRC(mf_src<double>(c), mf_src<float>(c));
  else
    LZ_SRC((SkSrc<double>{c->sk64, c->blk_bonds}), (SkSrc<float>{c->sk32, c->blk_bonds}));
#undef LZ_SRC
}

nh_status LanczosRun::iterate(int k, bool red) {
  nh_context *c = c_;
  const bool sk = sk_like(c);
  const double *bprev = k > 0 ? beta_ + (k - 1) : nullptr;
  const double *bprev2 = k > 1 ? beta_ + (k - 2) : nullptr;
  const bool timed = (k % kTimeEvery) == 0;
  Timed evp{nullptr, nullptr, red};
  if (timed) {
    NH_HIP(hipEventCreate(&evp.start));
    NH_HIP(hipEventCreate(&evp.stop));
    NH_HIP(hipEventRecord(evp.start, c->stream));
  }
  if (sk) {
    if (c->nb == 20) launch_sk<2>(k, red);
    else launch_sk<1>(k, red);
  } else {
    // q_k is stored (ring slot) only in the eigenvector pass, which
    // accumulates from it; the update forms q_k, q_{k-1} from r_k, r_{k-1}
    double2 *Q = red ? nullptr : ring_ + (int64_t)(k % ring_k_) * n_;
    double *part = red ? part_ : nullptr;
#define LZ_HVW(W, NSP, TB, BLK)                                                \
  hipLaunchKernelGGL((k_lz_hv<W, NSP, TB, TB>), dim3(grid_), dim3(64 * W), 0,  \
                     c->stream, c->n_atoms, c->onsite, BLK, c->nbr, R_, Q, Y_, \
                     bprev, part)
#define LZ_HV(NSP, TB, BLK)                                                    \
  do {                                                                         \
    if (waves_ == 8) LZ_HVW(8, NSP, TB, BLK);                                  \
    else if (waves_ == 6) LZ_HVW(6, NSP, TB, BLK);                             \
    else LZ_HVW(4, NSP, TB, BLK);                                              \
  } while (0)
    if (c->precision == NH_PREC_FP64) {
      if (c->nb == 20) LZ_HV(2, double, c->blocks64);
      else LZ_HV(1, double, c->blocks64);
    } else {
      if (c->nb == 20) LZ_HV(2, float, c->blocks32);
      else LZ_HV(1, float, c->blocks32);
    }
#undef LZ_HV
#undef LZ_HVW
  }
  NH_HIP(hipGetLastError());
  if (timed) {
    NH_HIP(hipEventRecord(evp.stop, c->stream));
    ev_.push_back(evp);
  }
  if (red) last_ = k;
  if (sk && defer_) {
    // rotate (r_{k-1}, u_{k-1}) <- (r_k, u_k) (step 0: r_0 stays); the
    // eigenvector pass rotates its slots by index
    if (red) {
      if (k > 0) std::swap(r_[0], r_[1]);
      std::swap(u_[0], u_[1]);
    }
    return NH_OK;
  }
  if (sk && !red) return NH_OK;
  if (red)
    hipLaunchKernelGGL(k_lz_scalar, dim3(1), dim3(kRedThreads), 0, c->stream,
                       grid_, 1, part_, alpha_ + k, 0);
  const int nb = reduce_blocks(n_);
  hipLaunchKernelGGL(k_lz_update, dim3(nb), dim3(kRedThreads), 0, c->stream,
                     n_, Y_, R_, k > 0 ? Rm1_ : nullptr, alpha_ + k, bprev,
                     bprev2, red ? part_ : nullptr);
  if (red)
    hipLaunchKernelGGL(k_lz_scalar, dim3(1), dim3(kRedThreads), 0, c->stream,
                       nb, 2, part_, beta_ + k, 1);
  NH_HIP(hipGetLastError());
  // r_{k+1} is in Y: rotate (r_{k-1}, r_k, y) -> (r_k, r_{k+1}, free)
  double2 *free_buf = Rm1_;
  Rm1_ = R_;
  R_ = Y_;
  Y_ = free_buf;
  return NH_OK;
}

bool LanczosRun::window_done(int w, int req, int rule) const {
  if (req <= 0) return true;
  if (rule == 0) {
    // reference rule (lanczos.c:1231-1232): enough converged values found
    // anywhere in the window
    int cnt = 0;
    for (const auto &x : conv_) cnt += x.window == w;
    return cnt >= req;
  }
  // the `req` Ritz values nearest the gap (top of the vb window, bottom of
  // the cb window) must all be converged
  const auto &r = lastRitz_[w];
  const auto &cv = lastConv_[w];
  if ((int)r.size() < req) return false;
  for (int t = 0; t < req; ++t) {
    const int idx = w == 0 ? (int)r.size() - 1 - t : t;
    if (!cv[idx]) return false;
  }
  return true;
}

// queue the copy of alpha and beta up to step m into the pinned staging
nh_status LanczosRun::fetch(int m) {
  if (m > fetched_) {
    // deferred step: the last step's alpha and beta are still partials (the
    // next step would sum them)
    if (defer_ && last_ == m - 1)
      hipLaunchKernelGGL(k_lz_scalars3, dim3(1), dim3(kRedThreads), 0, c_->stream, grid_,
                         part_ + (size_t)(last_ & 1) * 3 * nparts_, alpha_ + last_,
                         beta_ + last_);
    NH_HIP(hipGetLastError());
    if (!alone_) {
      NH_HIP(hipEventRecord(fetch_ev_, c_->stream));
      NH_HIP(hipStreamWaitEvent(c_->side, fetch_ev_, 0));
    }
    const int from = fetched_ > 0 ? fetched_ : -1;
    NH_HIP(hipMemcpyAsync(pin_ + 1 + from, alpha_ + from, (m - from) * sizeof(double),
                          hipMemcpyDeviceToHost, check_stream()));
    NH_HIP(hipMemcpyAsync(pin_ + pin_cap_ + fetched_, beta_ + fetched_,
                          (m - fetched_) * sizeof(double), hipMemcpyDeviceToHost, check_stream()));
    fetched_ = m;
  }
  return check(m);
}

// queue the check of the first m steps (fetched before) on the side stream
// (alone_: the run's only check, with no steps beside it, on the run's own);
// the earlier one has been waited for
nh_status LanczosRun::check(int m) {
  const TriWindows win = win_at(m);
  const int count = win.want[0] + win.want[1];
  if (count > 0) {
    const int groups = std::min(count, kTriGroups);
    const int64_t need = groups * tri_scratch(m);
    if (need > tri_cap_) {
      if (tri_s_) pool_release(c_, tri_s_);
      tri_s_ = nullptr;
      tri_cap_ = 0;
      const int64_t cap = groups * tri_scratch(std::max(2 * m, 2048));
      NH_TRY(pool_alloc(c_, (void **)&tri_s_, cap * sizeof(double)));
      tri_cap_ = cap;
    }
    for (int first = 0; first < count; first += groups)
      hipLaunchKernelGGL(k_tri_windows, dim3(std::min(groups, count - first)), dim3(kTriThreads),
                         0, check_stream(), m, alpha_, beta_, win, first, tri_s_, tri_out_);
    NH_HIP(hipGetLastError());
    NH_HIP(hipMemcpyAsync(pin_ + 2 * (size_t)pin_cap_, tri_out_,
                          (kTriHead + (size_t)count * kTriOut) * sizeof(double),
                          hipMemcpyDeviceToHost, check_stream()));
  }
  NH_HIP(hipEventRecord(check_ev_, check_stream()));
  checked_ = m;
  return NH_OK;
}

// A caller's start vector may lie in an almost invariant subspace (an
// eigenvector): a look at the first step beside the ones that follow, so that
// such a run is not first taken to its first check
nh_status LanczosRun::look(bool wait) {
  double *first = pin_ + 2 * (size_t)pin_cap_ - 3;  // the places of the last beta
  if (!wait) {
    NH_HIP(hipEventRecord(fetch_ev_, c_->stream));
    NH_HIP(hipStreamWaitEvent(c_->side, fetch_ev_, 0));
    NH_HIP(hipMemcpyAsync(first, alpha_ - 1, 2 * sizeof(double), hipMemcpyDeviceToHost, c_->side));
    NH_HIP(hipMemcpyAsync(first + 2, beta_, sizeof(double), hipMemcpyDeviceToHost, c_->side));
    NH_HIP(hipEventRecord(look_ev_, c_->side));
    return NH_OK;
  }
  NH_HIP(hipEventSynchronize(look_ev_));
  small_beta_ = lost(first[0], first[1], first[2]);
  return small_beta_ ? NH_ERR_STATE : NH_OK;
}

// analyse the tridiagonal of the first m steps (fetch(m) queued before)
nh_status LanczosRun::analyse(int m, const nh_lanczos_opts *o) {
  NH_CHECK(fetched_ >= m, NH_ERR_STATE, "Lanczos: tridiagonal not fetched");
  if (checked_ != m) NH_TRY(check(m));
  NH_HIP(hipEventSynchronize(check_ev_));
  ha_.assign(pin_ + 1, pin_ + 1 + m);
  hb_.assign(pin_ + pin_cap_, pin_ + pin_cap_ + m);
  // The deferred FP64 step has beta^2 as a difference of sums, |w|^2 - (alpha -
  // sigma)^2 (LzPart3): below |w|^2 / 8 (a start vector in an almost invariant
  // subspace; 0.83 |w|^2 was the least in 1,400 steps from ordinary ones) three
  // of its bits are lost, and the run is repeated with the classic step, which
  // sums |r|^2 itself.  (FP32 vectors: their rounding is far above what is lost.)
  if (defer_ && vbytes_ == sizeof(double2))
    for (int i = 0; i < m; ++i)
      if (lost(pin_[i], ha_[i], hb_[i])) small_beta_ = true;
  if (small_beta_) return NH_ERR_STATE;
  const double tol = o->conv_tolerance;
  const double resolution = 100.0 * tol;  // lanczos.c:1970
  const double bias = 1e-80;
  const int req[2] = {o->num_eig_vb, o->num_eig_cb};
  const double *tri = pin_ + 2 * (size_t)pin_cap_;
  // nearest-the-gap rule: two converged copies of one level differ by up to
  // about 2 tol ||T|| (each Ritz value within beta tol of it), which the
  // reference's relative resolution misses for levels near 0 eV; that rule
  // merges copies within this bound as well (the reference rule keeps the
  // reference's check)
  double dup_abs = 0.0;
  if (o->stop_rule == 1) {
    double tn = 0.0;
    for (int i = 0; i < m; ++i)
      tn = std::max(tn, std::fabs(ha_[i]) + (i > 0 ? std::fabs(hb_[i - 1]) : 0.0) +
                            (i + 1 < m ? std::fabs(hb_[i]) : 0.0));
    dup_abs = 2.0 * tol * tn;
  }
  for (int w = 0; w < 2; ++w) {
    lastRitz_[w].clear();
    lastConv_[w].clear();
    if (req[w] <= 0) continue;
    // the candidates nearest the gap: top of vb, bottom of cb
    std::vector<double> ev((size_t)tri[w]);
    const double *o3 = tri + kTriHead + (w ? win_at(m).want[0] : 0) * kTriOut;
    for (size_t i = 0; i < ev.size(); ++i) ev[i] = o3[kTriOut * i];
    auto duplicate = [&](size_t i) {
      // copies of one eigenvalue (ghosts, degeneracies) count once
      return i > 0 && std::fabs(ev[i - 1] - ev[i]) <
                          std::max(std::fabs(bias + ev[i]) * resolution, dup_abs);
    };
    auto known_value = [&](double v) {
      for (const auto &cv : conv_)
        if (std::fabs(cv.value - v) < resolution) return true;
      return false;
    };
    for (size_t i = 0; i < ev.size(); ++i) {
      if (duplicate(i)) continue;
      const bool known = known_value(ev[i]);
      bool ok = known;
      if (!known) {
        ok = std::fabs(o3[kTriOut * i + 1]) <= tol && std::fabs(o3[kTriOut * i + 2]) <= tol;
        if (ok) conv_.push_back({ev[i], m, w});
      }
      lastRitz_[w].push_back(ev[i]);
      lastConv_[w].push_back(ok);
    }
  }
  return NH_OK;
}

nh_status LanczosRun::run(const nh_lanczos_opts *o, nh_eig_result *res) {
  nh_context *c = c_;
  const auto t0 = std::chrono::steady_clock::now();
  NH_CHECK(c->layout == NH_LAYOUT_BLOCKS || sk_like(c), NH_ERR_STATE,
           "Lanczos: build the Hamiltonian first");
  NH_CHECK(o->max_iter > 2 && o->conv_tolerance > 0, NH_ERR_ARG,
           "Lanczos: bad max_iter / tolerance");
  n_ = c->n;
  // FP32 products with FP64 vectors (NH_SET_LZ_VECTORS = 0) and stored blocks
  // take the classic step
  const bool fp32 = c->precision == NH_PREC_FP32;
  defer_ = sk_like(c) && !classic_ && (!fp32 || lz_fp32_vectors(c));
  vbytes_ = defer_ && fp32 ? sizeof(float2) : sizeof(double2);
  if (!defer_) {
    NH_TRY(alloc((void **)&R_, n_ * sizeof(double2)));
    NH_TRY(alloc((void **)&Rm1_, n_ * sizeof(double2)));
    NH_TRY(alloc((void **)&Y_, n_ * sizeof(double2)));
  }
  NH_TRY(alloc((void **)&alpha_, (size_t)(o->max_iter + 2) * sizeof(double)));
  ++alpha_;  // alpha_[-1]: sigma_0
  NH_TRY(alloc((void **)&beta_, (size_t)(o->max_iter + 1) * sizeof(double)));
  // workgroups of the products: as many as run at a time (LDS: 2 a CU with
  // FP64 entries, 3 with FP32 ones)
  waves_ = hv_waves(c->n_atoms);
  grid_ = sk_like(c) ? sk_grid(c, vbytes_ == sizeof(float2) ? 3 : 2)
                     : (c->n_atoms + waves_ * kRowAtoms - 1) / (waves_ * kRowAtoms);
  nparts_ = std::max(grid_, 2 * kRedMaxBlocks) + 64;
  NH_TRY(alloc((void **)&part_, (size_t)nparts_ * 6 * sizeof(double)));

  NH_TRY(build_start(o));
  if (defer_) {
    for (char **p : {&r_[0], &r_[1], &u_[0], &u_[1]})
      NH_TRY(alloc((void **)p, n_ * vbytes_));
    NH_TRY(upload_start(r_[0], vbytes_));
  } else {
    NH_TRY(upload_start(R_, vbytes_));
  }

  // pass 1: eigenvalues.  The tridiagonal of one check point is analysed
  // (k_tri_windows, on a second stream) while the device runs the steps up to
  // the next one, and its results are looked at there, after that block of
  // steps has been queued.  Convergence is thus seen one block late; the steps of
  // that block are not used (the run ends at the converged check point).
  pin_cap_ = o->max_iter + 2;
  win_ = TriWindows{{o->erange_vb[0], o->erange_cb[0]},
                    {o->erange_vb[1], o->erange_cb[1]},
                    {o->num_eig_vb > 0 ? std::min(o->num_eig_vb, o->max_iter) + 24 : 0,
                     o->num_eig_cb > 0 ? std::min(o->num_eig_cb, o->max_iter) + 24 : 0}};
  const size_t tri = kTriHead + (size_t)(win_.want[0] + win_.want[1]) * kTriOut;
  NH_TRY(alloc((void **)&tri_out_, tri * sizeof(double)));
  NH_HIP(hipHostMalloc((void **)&pin_, (2 * (size_t)pin_cap_ + tri) * sizeof(double),
                       hipHostMallocDefault));
  if (!c->side) NH_HIP(hipStreamCreateWithFlags(&c->side, hipStreamNonBlocking));
  NH_HIP(hipEventCreateWithFlags(&fetch_ev_, hipEventDisableTiming));
  NH_HIP(hipEventCreateWithFlags(&check_ev_, hipEventDisableTiming));
  constexpr int kLook = 2, kLookAt = 8;  // steps queued before look() and its wait
  const bool looks = defer_ && vbytes_ == sizeof(double2) && (o->start == 2 || o->start == 3) &&
                     o->restore_len <= 0 && o->max_iter > kLookAt + 3;
  if (looks) NH_HIP(hipEventCreateWithFlags(&look_ev_, hipEventDisableTiming));
  int m = 0, skip = 0, pending = -1;
  bool done = false;
  Progress prog;
  if (o->restore_len > 0) {
    // restart from the tridiagonal of an earlier run (restoreState,
    // lanczos.c:1905-1960): no eigenvalue pass
    NH_CHECK(o->restore_alpha && o->restore_beta && o->restore_len <= o->max_iter,
             NH_ERR_ARG, "Lanczos restart: tridiagonal missing or longer than max_iter");
    m = o->restore_len;
    NH_HIP(hipMemcpyAsync(alpha_, o->restore_alpha, (size_t)m * sizeof(double),
                          hipMemcpyHostToDevice, c->stream));
    NH_HIP(hipMemcpyAsync(beta_, o->restore_beta, (size_t)m * sizeof(double),
                          hipMemcpyHostToDevice, c->stream));
    NH_TRY(fetch(m));
    // the analyses of the original run, at the same check points (which
    // converged values were recorded depends on where they were seen)
    int mm = 0, sk = 0;
    while (mm < m) {
      ++mm;
      ++sk;
      if (o->conv_check_start < mm && o->conv_check_skip <= sk) {
        sk = 0;
        NH_TRY(analyse(mm, o));
        done = window_done(0, o->num_eig_vb, o->stop_rule) &&
               window_done(1, o->num_eig_cb, o->stop_rule);
        if (done) break;
      }
    }
    if (!done) {
      NH_TRY(analyse(m, o));
      done = window_done(0, o->num_eig_vb, o->stop_rule) &&
             window_done(1, o->num_eig_cb, o->stop_rule);
    } else {
      m = mm;
    }
    pending = m;
  }
  while (o->restore_len <= 0 && m + 1 < o->max_iter) {
    NH_TRY(iterate(m, true));
    ++m;
    prog.tick("lanczos", m, (int)conv_.size());
    ++matvecs_;
    ++skip;
    if (looks && (m == kLook || m == kLookAt)) NH_TRY(look(m == kLookAt));
    if (o->conv_check_start < m && o->conv_check_skip <= skip) {
      skip = 0;
      if (pending > 0) {
        NH_TRY(analyse(pending, o));
        done = window_done(0, o->num_eig_vb, o->stop_rule) &&
               window_done(1, o->num_eig_cb, o->stop_rule);
        if (done) break;
      }
      NH_TRY(fetch(m));
      pending = m;
    }
  }
  if (done) {
    m = pending;
  } else if (o->restore_len <= 0) {
    // no check before and none beside steps: 23 us less than across streams
    alone_ = checked_ == 0;
    NH_TRY(fetch(m));
    NH_TRY(analyse(m, o));
    done = window_done(0, o->num_eig_vb, o->stop_rule) &&
           window_done(1, o->num_eig_cb, o->stop_rule);
  }
  if (res->tridiag_alpha && res->tridiag_beta) {
    const int cnt = std::min(m, res->tridiag_cap);
    std::copy(ha_.begin(), ha_.begin() + cnt, res->tridiag_alpha);
    std::copy(hb_.begin(), hb_.begin() + cnt, res->tridiag_beta);
  }

  // the converged eigenvalues nearest the gap in each window
  std::vector<Converged> pick;
  const int req[2] = {o->num_eig_vb, o->num_eig_cb};
  for (int w = 0; w < 2; ++w) {
    if (o->stop_rule == 0) {
      // every converged value of the window, nearest the gap first
      std::vector<Converged> in;
      for (const auto &x : conv_)
        if (x.window == w) in.push_back(x);
      std::sort(in.begin(), in.end(), [w](const Converged &a, const Converged &b) {
        return w == 0 ? a.value > b.value : a.value < b.value;
      });
      for (int t = 0; t < (int)in.size() && t < req[w]; ++t) pick.push_back(in[t]);
      continue;
    }
    const auto &r = lastRitz_[w];
    const auto &cv = lastConv_[w];
    int got = 0;
    for (int t = 0; t < (int)r.size() && got < req[w]; ++t) {
      const int idx = w == 0 ? (int)r.size() - 1 - t : t;
      // report only the converged prefix nearest the gap: an unconverged
      // Ritz value there may be a state that a farther converged one would
      // wrongly replace
      if (!cv[idx]) break;
      for (const auto &x : conv_)
        if (std::fabs(x.value - r[idx]) < 100.0 * o->conv_tolerance) {
          pick.push_back({r[idx], x.iter, w});
          break;
        }
      ++got;
    }
  }
  std::sort(pick.begin(), pick.end(),
            [](const Converged &a, const Converged &b) { return a.value < b.value; });
  const int ne = std::min((int)pick.size(), std::min(res->capacity, kMaxVec));
  res->n_found = ne;
  res->iterations = m;
  for (int e = 0; e < ne; ++e) {
    res->eigenvalues[e] = pick[e].value;
    if (res->residuals) res->residuals[e] = -1.0;
  }

  if (o->want_vectors && ne > 0) {
    // pass 2: rebuild the Lanczos vectors from r0 and accumulate
    int mmax = 0;
    for (int e = 0; e < ne; ++e) mmax = std::max(mmax, pick[e].iter);
    std::vector<std::vector<double>> z(ne);
    for (int e = 0; e < ne; ++e)
      tri_eigvec(ha_, hb_, pick[e].iter, pick[e].value, z[e]);
    // the deferred step's vectors of the eigenvalue pass are done with
    if (defer_)
      for (char *p : {r_[0], r_[1], u_[0], u_[1]}) release(p);
    double2 *V = nullptr;
    double *dZ = nullptr;
    NH_TRY(alloc((void **)&V, (size_t)ne * n_ * sizeof(double2)));
    NH_TRY(alloc((void **)&dZ, (size_t)kMaxVec * kRingMax * sizeof(double)));
    NH_HIP(hipMemsetAsync(V, 0, (size_t)ne * n_ * sizeof(double2), c->stream));
    // ring: K = 128 steps per flush when the ring takes at most half the
    // free memory (the run's buffers are released before any later stage
    // allocates), else 32, 16 or 8 (each flush reads and writes the
    // eigenvectors once)
    const bool rring = sk_like(c);
    {
      size_t fr = 0, tot = 0;
      NH_HIP(hipMemGetInfo(&fr, &tot));
      fr += pool_free_bytes(c);
      const size_t slot = (rring ? 2 : 1) * n_ * vbytes_;
      ring_k_ = kRingMax;
      while (ring_k_ > 8 && (size_t)ring_k_ * slot > fr / 2) ring_k_ /= 2;
      if (c->ring_steps > 0) ring_k_ = std::min(ring_k_, c->ring_steps);
    }
    if (rring) {
      NH_CHECK(n_ % 2 == 0, NH_ERR_STATE, "Lanczos: the ring needs an even N");
      NH_TRY(alloc((void **)&ringr_, (size_t)2 * ring_k_ * n_ * vbytes_));
      NH_TRY(upload_start(ringr_, vbytes_));
      if (defer_) Y_ = R0_;  // the start vector is in the ring: free for H v
    } else {
      NH_TRY(alloc((void **)&ring_, (size_t)ring_k_ * n_ * sizeof(double2)));
      NH_TRY(upload_start(R_, sizeof(double2)));
    }
    std::vector<double> hz((size_t)kMaxVec * kRingMax);
    const int rk = ring_k_;
    for (int k = 0; k < mmax; ++k) {
      NH_TRY(iterate(k, false));
      ++matvecs_;
      prog.tick("lanczos eigenvectors", k + 1, mmax);
      if ((k + 1) % rk == 0 || k + 1 == mmax) {
        const int k0 = k + 1 - ((k % rk) + 1);
        const int K = k + 1 - k0;
        for (int e = 0; e < ne; ++e)
          for (int t = 0; t < K; ++t) {
            const int j = k0 + t;
            // q_j = r_j / beta_{j-1} for the ring of r
            const double sc = ringr_ && j > 0 ? 1.0 / hb_[j - 1] : 1.0;
            hz[e * K + t] = j < pick[e].iter ? z[e][j] * sc : 0.0;
          }
        NH_HIP(hipMemcpyAsync(dZ, hz.data(), (size_t)ne * K * sizeof(double),
                              hipMemcpyHostToDevice, c->stream));
        int64_t g = (n_ + 255) / 256;
        if (g > 8192) g = 8192;
        // ring slots k0..k hold q_k0..q_k in order since k0 % K == 0 (ring of
        // r: slots k0 % (2 K) + t hold r_k0+t)
        if (ringr_ && vbytes_ == sizeof(float2))
          hipLaunchKernelGGL(k_lz_accum32, dim3((int)g), dim3(256), 0,
                             c->stream, n_, ne, K, dZ,
                             reinterpret_cast<const float2 *>(slot(k0)), n_, V, n_);
        else
          hipLaunchKernelGGL((k_lz_accum<double2>), dim3((int)g), dim3(256), 0,
                             c->stream, n_, ne, K, dZ,
                             ringr_ ? reinterpret_cast<const double2 *>(slot(k0)) : ring_, n_,
                             V, n_);
        NH_HIP(hipGetLastError());
        // the host array hz is reused next chunk: wait for the copy
        NH_HIP(hipStreamSynchronize(c->stream));
      }
    }
    // normalise, Rayleigh quotient and residual in FP64
    for (int e = 0; e < ne; ++e) {
      const nh_cplx *v = reinterpret_cast<const nh_cplx *>(V + (int64_t)e * n_);
      double nrm2;
      NH_TRY(reduce_nrm2sq(c, n_, v, &nrm2));
      int64_t g = (n_ + 255) / 256;
      if (g > 8192) g = 8192;
      hipLaunchKernelGGL(k_scale, dim3((int)g), dim3(256), 0, c->stream, n_,
                         V + (int64_t)e * n_, 1.0 / std::sqrt(nrm2));
      NH_TRY(launch_hv(c, 0.0, v, reinterpret_cast<nh_cplx *>(Y_), 1, n_));
      ++matvecs_;
      double rq[2];
      NH_TRY(reduce_dot(c, n_, v, reinterpret_cast<nh_cplx *>(Y_), rq));
      const nh_cplx a = {-rq[0], 0.0}, b = {1.0, 0.0};
      NH_TRY(launch_axpby(c, n_, a, v, b, reinterpret_cast<nh_cplx *>(Y_)));
      double r2;
      NH_TRY(reduce_nrm2sq(c, n_, reinterpret_cast<nh_cplx *>(Y_), &r2));
      res->eigenvalues[e] = rq[0];
      if (res->residuals) res->residuals[e] = std::sqrt(r2);
      // A tridiagonal of another recurrence (an older version's order of the
      // step, another precision or setting of the vectors) is not retraced:
      // its vectors drift from this recurrence's as far as rounding grows, and
      // what they add up to is no eigenvector.  A retraced one's residual is
      // beta times the last component, or the rounding of the vectors.
      if (o->restore_len > 0) {
        const int it = pick[e].iter;
        double tn = 0.0;
        for (int i = 0; i < it; ++i) tn = std::max(tn, std::fabs(ha_[i]) + 2.0 * std::fabs(hb_[i]));
        const double eps = c->precision == NH_PREC_FP64 ? 1e-16 : 1e-8;
        const double tail = std::fabs(hb_[it - 1] * z[e][it - 1]);
        if (!(std::sqrt(r2) <= 100.0 * tail + std::sqrt(eps) * tn)) {
          stale_ = true;
          return NH_ERR_STATE;
        }
      }
      if (res->eigenvectors)
        NH_HIP(hipMemcpy(res->eigenvectors + (int64_t)e * n_, v,
                         n_ * sizeof(nh_cplx), hipMemcpyDefault));  // host or device
    }
  }
  NH_HIP(hipStreamSynchronize(c->stream));
  res->matvecs = matvecs_;
  NH_TRY(collect_timing());
  res->hv_ms = hv_ms(0);
  res->hv_timed = hv_timed(0);
  res->hv_ms_vec = hv_ms(1);
  res->hv_timed_vec = hv_timed(1);
  res->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return done ? NH_OK : NH_ERR_NOCONV;
}

}  // namespace
}  // namespace nh

extern "C" nh_status nh_eigensolve_lanczos(nh_context *ctx,
                                           const nh_lanczos_opts *opts,
                                           nh_eig_result *res) {
  NH_CHECK(ctx && opts && res && res->eigenvalues && res->capacity > 0,
           NH_ERR_ARG, "nh_eigensolve_lanczos: bad arguments");
  (void)hipGetLastError();
  NH_HIP(hipSetDevice(ctx->device));
  const auto t0 = std::chrono::steady_clock::now();
  nh_lanczos_opts o = *opts;
  int before = 0;
  for (bool classic = false;;) {
    nh::LanczosRun run(ctx, classic);
    const nh_status st = run.run(&o, res);
    if (run.small_beta()) {
      classic = true;
    } else if (run.stale()) {
      // the eigenvalue pass after all
      o.restore_len = 0;
      classic = false;
    } else {
      if (st != NH_OK && st != NH_ERR_NOCONV) return st;
      res->matvecs += before;
      if (before > 0)
        res->seconds =
            std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
      return st;
    }
    before += run.matvecs();
  }
}
