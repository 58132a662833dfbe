// Keating valence-force-field relaxation on the GPU.
//
// Energy (calc_estrain, NEMO_3D/nemo3d/src/base/strain3d.c:1739-1890), per
// atom i over its present neighbours n, p:
//   E_i = sum_n  a_in / (2 d0_in^2) (|r_in|^2 - d0_in^2)^2
//       + sum_{n<p} sqrt(b_in b_ip) / (|d0_in| |d0_ip|) (r_in.r_ip - d0_in.d0_ip)^2
// with r_in the strained bond vector, d0_in the ideal bond vector of the
// pair's material (unstrained lattice constant), a, b the Keating constants
// of the pair (StrainParam).  The total is sum_i E_i, so each bond term
// enters from both of its atoms.
//
// The gradient is the reference's (strain3d.c:1806-1830 and 1889-2050): an
// atom receives the derivative of its own copy of each bond term only
// (-4 a/(2 d0^2) dl r_in), half the derivative of E, and the full
// derivative of the angle terms.  The relaxation follows that gradient, so
// its stationary point is that of E with each bond term counted once; E
// itself is reported as the reference prints it.
//
// StrainModel = VFF_keating_strained replaces a and sqrt(b_in b_ip) by the
// strain-scaled constants of StrainParam::alpha_eff / beta_eff
// (StrainParam.c:60-214): per bond a (1 - A (|r|^2 / d0^2 - 1)), per angle
// b_in (1 - B (cos + 1/3)) (1 - C (|r_in| |r_ip| / (|d0_in| |d0_ip|) - 1))
// with B, C the geometric means of the two bonds' constants and both
// factors truncated near their extrema; the reference's b_in is the
// constant of the lower-slot leg n.  As in calc_estrain (strain3d.c:
// 1687-1700, 1835-1860) the scaled constants are taken as fixed when the
// gradient is formed, so the "gradient" of this model is that of the
// harmonic form at the current constants.
//
// The gradient on atom i is gathered per atom (no atomics): its own bond
// and angle terms plus the angle terms centred on each neighbour j in which
// i is a leg.  Keating = FixSurfaceAll holds atoms with fewer than four
// neighbours fixed; AllFree moves every atom.  Minimisation: Polak-Ribiere+
// nonlinear conjugate gradients with a secant line search on the
// directional derivative (the reference uses MacKay's macopt CG,
// eigen/src/macopt.c, whose line search also uses only gradients).  The
// descent runs on the device: a gradient kernel (with the sums the line search
// needs) and a kernel that takes the next step of it, in turn; the host queues
// them in batches and looks whether it is over.
#include <chrono>
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "nh_internal.h"
#include "nh_vector.h"

namespace nh {

struct VffArgs {
  int A, S;
  const int32_t *species, *nbr, *bond_q;
  const double *alpha, *beta, *a0;  // [S][S]
  double lx, ly, lz;
  const double *aa, *ba, *ca;  // [S][S], NH_VFF_KEATING_STRAINED only
  int model;
  int fix_surface;
};

// StrainParam::alpha_eff with anh = 1 (StrainParam.c:60-100); the
// reference's how_close_to_maximum_of_distorsion_energy is 0.001
constexpr double kVffNearMax = 0.001;

__device__ __forceinline__ double alpha_eff(double al0, double A, double r2,
                                            double d2) {
  const double delt = 1.0 - kVffNearMax;
  if (r2 < d2 * (1.0 + delt * 2.0 / (3.0 * A)))
    return al0 * (1.0 - A * (r2 / d2 - 1.0));
  return al0 * (1.0 - delt / 1.5);
}

// StrainParam::beta_eff with anh = 1 (StrainParam.c:118-214): be0 the
// constant of the first leg, d1/d2 the ideal and r1/r2 the strained legs
__device__ __forceinline__ double beta_eff(double be0, double B, double C,
                                           const double d1[3],
                                           const double d2[3],
                                           const double r1[3],
                                           const double r2[3]) {
  const double d10 = sqrt(d1[0] * d1[0] + d1[1] * d1[1] + d1[2] * d1[2]);
  const double d20 = sqrt(d2[0] * d2[0] + d2[1] * d2[1] + d2[2] * d2[2]);
  const double rr = r1[0] * r2[0] + r1[1] * r2[1] + r1[2] * r2[2];
  const double r10 = sqrt(r1[0] * r1[0] + r1[1] * r1[1] + r1[2] * r1[2]);
  const double r20 = sqrt(r2[0] * r2[0] + r2[1] * r2[1] + r2[2] * r2[2]);
  const double rd = r10 * r20 / (d10 * d20);
  const double tt = rr / (r10 * r20);
  const double delt = 1.0 + kVffNearMax, delh = 1.0 - kVffNearMax;
  double beta = be0;
  bool flag = true;
  if (tt > delt / 3.0 * (2.0 * (1.0 / B - 1.0 / 3.0) - 1.0 / (3.0 * rd))) {
    beta = be0 * ((1.0 - 2.0 * delt / 3.0) +
                  B / 3.0 * (delt / 3.0 * (1.0 / rd + 2.0) - 1.0)) *
           (1.0 - C * (rd - 1.0));
    flag = false;
  }
  if (rd > 1.0 + delh * 2.0 / (3.0 * C)) {
    const double be = be0 * (1.0 - B * (tt + 1.0 / 3.0)) * (1.0 - delh * 2.0 / 3.0);
    if (flag || be > beta) beta = be;
    flag = false;
  }
  if (flag) beta = be0 * (1.0 - B * (tt + 1.0 / 3.0)) * (1.0 - C * (rd - 1.0));
  return beta;
}

// bond vector of slot n of atom i from its position a to b, q its ideal vector
// in units of a0 / 4
__device__ __forceinline__ void bond_vec(const VffArgs &g, const int32_t q[3], int ti, int tj,
                                         const double4 &a, const double4 &b, double r[3],
                                         double d0[3]) {
  const double lat[3] = {g.lx, g.ly, g.lz};
  const double u[3] = {b.x - a.x, b.y - a.y, b.z - a.z};
  const double a0 = g.a0[ti * g.S + tj];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double f = 0.25 * q[k];
    r[k] = lat[k] * f + u[k];
    d0[k] = a0 * f;
  }
}

__device__ __forceinline__ double dot3(const double a[3], const double b[3]) {
  return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

// A leg of an angle: strained and ideal bond vector from the centre, and
// beta / |d0|^2 of the (centre, leg) pair
struct Leg {
  double r[3], d0[3], w;
  int type;
};
// The angle term of legs 1, 2 (1 in the lower slot of the centre, of type tc):
// K (t - t0)^2 with K = constant / (|d0_1| |d0_2|); c = t - t0 = r1.r2 -
// d0_1.d0_2
template <int MODEL>
__device__ __forceinline__ void angle_term(const VffArgs &g, int tc, const Leg &a, const Leg &b,
                                           double &K, double &c) {
  c = dot3(a.r, b.r) - dot3(a.d0, b.d0);
  if constexpr (MODEL == NH_VFF_KEATING) {
    K = sqrt(a.w * b.w);
  } else {
    const double b1 = g.beta[tc * g.S + a.type];
    const double B = sqrt(g.ba[tc * g.S + a.type] * g.ba[tc * g.S + b.type]);
    const double C = sqrt(g.ca[tc * g.S + a.type] * g.ca[tc * g.S + b.type]);
    K = beta_eff(sqrt(b1 * b1), B, C, a.d0, b.d0, a.r, b.r) /
        sqrt(dot3(a.d0, a.d0) * dot3(b.d0, b.d0));
  }
}

template <int CTRL>
__device__ __forceinline__ double quad_move(double v) {
  const int64_t b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
  return __longlong_as_double((int64_t)(uint32_t)lo | (int64_t)hi << 32);
}
__device__ __forceinline__ double quad_sum(double v) {
  v += quad_move<0xB1>(v);  // 1 0 3 2
  v += quad_move<0x4E>(v);  // 2 3 0 1
  return v;
}
// Partial sums of a gradient, per workgroup: E, |grad|^2, grad.dir, grad.old
constexpr int kVffSums = 4;
// The sums over a workgroup of kRedThreads, in a fixed order, in every thread;
// s: kVffSums * kRedThreads / 64 doubles.  Each sum has its own part of s, so
// one barrier does for all of them (sums taken one after another through the
// same part would need a second one between a sum's read and the next's write)
__device__ __forceinline__ void vff_block_sums(double (&v)[kVffSums], double *s) {
  constexpr int kWaves = kRedThreads / 64;
#pragma unroll
  for (int k = 0; k < kVffSums; ++k) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off, 64);
    if ((threadIdx.x & 63) == 0) s[k * kWaves + (threadIdx.x >> 6)] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kVffSums; ++k) {
    v[k] = s[k * kWaves];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) v[k] += s[k * kWaves + w];
  }
}
// Gradient of E at pos (x, y, z, and the species in w) with the sums over it;
// dir, old: null for 0; st: the descent's state (null: none), nothing is done
// when it is over.  Bound by the latency of dependent gathers (neighbours,
// then their neighbours): a quad of lanes per atom, a lane per bond with the
// angles at both its ends, keeps four times the loads in flight (104,976
// atoms: 34 -> 17 us).  A descent of 40 steps there took 120 gradients, 199 dot
// products and as many waits of the host, 8.5 ms; now 80 gradients and steps,
// 2.1 ms (the gradient at an accepted point is the next one's start).
struct VffState {
  double t0, f0, t1, dg0, gg, step, e0, g0;
  int it, ls, par, done;  // par: which gradient buffer holds the current one
};
template <int MODEL>
__global__ __launch_bounds__(kRedThreads) void k_vff_grad(
    VffArgs g, const double4 *__restrict__ pos, double *__restrict__ grad0,
    double *__restrict__ grad1, const double *__restrict__ dir,
    const VffState *__restrict__ st, double *__restrict__ part) {
  double *grad = grad1;
  const double *old = nullptr;
  if (st) {
    if (st->done) return;
    grad = st->par ? grad0 : grad1;
    old = st->par ? grad1 : grad0;
  }
  const int slot = threadIdx.x & 3;
  double sum[kVffSums] = {0.0, 0.0, 0.0, 0.0};
  for (int64_t t = blockIdx.x * (int64_t)kRedThreads + threadIdx.x; t < (int64_t)g.A * 4;
       t += (int64_t)gridDim.x * kRedThreads) {
    const int i = (int)(t >> 2);
    const int j = g.nbr[t];
    const bool here = j >= 0;
    const double4 pi = pos[i], pj = pos[here ? j : i];
    const int ti = (int)pi.w, tj = (int)pj.w;
    Leg me{};
    me.type = here ? tj : -1;
    double gr[3], e = 0.0, f = 0.0;
    if (here) {
      const int32_t q[3] = {g.bond_q[t * 3], g.bond_q[t * 3 + 1], g.bond_q[t * 3 + 2]};
      bond_vec(g, q, ti, tj, pi, pj, me.r, me.d0);
      const double d0sq = dot3(me.d0, me.d0), rsq = dot3(me.r, me.r);
      const double al = MODEL == NH_VFF_KEATING
                            ? g.alpha[ti * g.S + tj]
                            : alpha_eff(g.alpha[ti * g.S + tj], g.aa[ti * g.S + tj], rsq, d0sq);
      const double dl = rsq - d0sq;
      me.w = g.beta[ti * g.S + tj] / d0sq;
      e = 0.5 * al / d0sq * dl * dl;
      // the derivative of this atom's copy of the bond term: d/du_i of
      // (a/2d0^2) dl^2 = -(2 a/d0^2) dl r_in (the neighbour's copy is
      // not differentiated here, as in the reference)
      f = -2.0 * al / d0sq * dl;
    }
    // the angles at i between this bond and the other three: both lanes of a
    // pair evaluate it (the lower slot's constants first) and take the part
    // along their own bond
    auto own = [&](auto X) {
      constexpr int x = X;
      constexpr int ctrl = x == 1 ? 0xB1 : x == 2 ? 0x4E : 0x1B;  // lane slot ^ x
      Leg o;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        o.r[k] = quad_move<ctrl>(me.r[k]);
        o.d0[k] = quad_move<ctrl>(me.d0[k]);
      }
      o.w = quad_move<ctrl>(me.w);
      o.type = __builtin_amdgcn_mov_dpp(me.type, ctrl, 0xF, 0xF, true);
      if (!here || o.type < 0) return;
      double K, c;
      if (MODEL == NH_VFF_KEATING || slot < (slot ^ x)) angle_term<MODEL>(g, ti, me, o, K, c);
      else angle_term<MODEL>(g, ti, o, me, K, c);
      e += 0.5 * K * c * c;
      f -= 2.0 * K * c;
    };
    own(std::integral_constant<int, 1>{});
    own(std::integral_constant<int, 2>{});
    own(std::integral_constant<int, 3>{});
#pragma unroll
    for (int k = 0; k < 3; ++k) gr[k] = f * me.r[k];
    // the angles at j in which this bond is a leg
    if (here) {
      const int4 nj = reinterpret_cast<const int4 *>(g.nbr)[j];
      const int nb[4] = {nj.x, nj.y, nj.z, nj.w};
      const int4 *qj = reinterpret_cast<const int4 *>(g.bond_q) + (int64_t)j * 3;
      const int4 q0 = qj[0], q1 = qj[1], q2 = qj[2];
      const int32_t q[12] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w,
                             q2.x, q2.y, q2.z, q2.w};
      double4 pk[4];
      // slot of i in j's list and the bond vector j -> i
      int si = -1;
      int32_t qi[3] = {0, 0, 0};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (nb[s] == i) {
          si = s;
          qi[0] = q[3 * s], qi[1] = q[3 * s + 1], qi[2] = q[3 * s + 2];
        }
        pk[s] = pos[nb[s] >= 0 ? nb[s] : j];
      }
      Leg back;
      bond_vec(g, qi, tj, ti, pj, pi, back.r, back.d0);
      back.type = ti;
      back.w = g.beta[tj * g.S + ti] / dot3(back.d0, back.d0);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s == si || nb[s] < 0) continue;
        const int32_t qs[3] = {q[3 * s], q[3 * s + 1], q[3 * s + 2]};
        Leg o;
        o.type = (int)pk[s].w;
        bond_vec(g, qs, tj, o.type, pj, pk[s], o.r, o.d0);
        o.w = g.beta[tj * g.S + o.type] / dot3(o.d0, o.d0);
        double K, c;
        // the angle's legs in j's slot order
        if (MODEL == NH_VFF_KEATING || si < s) angle_term<MODEL>(g, tj, back, o, K, c);
        else angle_term<MODEL>(g, tj, o, back, K, c);
#pragma unroll
        for (int k = 0; k < 3; ++k) gr[k] += 2.0 * K * c * o.r[k];
      }
    }
    const double present = quad_sum(here ? 1.0 : 0.0);
#pragma unroll
    for (int k = 0; k < 3; ++k) gr[k] = quad_sum(gr[k]);
    if (g.fix_surface && present < 4.0) gr[0] = gr[1] = gr[2] = 0.0;
    sum[0] += e;
    if (slot < 3) {
      const int64_t o = (int64_t)i * 3 + slot;
      const double v = slot == 0 ? gr[0] : slot == 1 ? gr[1] : gr[2];
      grad[o] = v;
      sum[1] += v * v;
      if (dir) sum[2] += v * dir[o];
      if (old) sum[3] += v * old[o];
    }
  }
  __shared__ double scratch[kVffSums * kRedThreads / 64];
  vff_block_sums(sum, scratch);
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < kVffSums; ++k) part[kVffSums * blockIdx.x + k] = sum[k];
}

namespace {

// sums of the workgroups' partials, in a fixed order, in every thread of a
// workgroup of kRedThreads; s as in vff_block_sums
__device__ __forceinline__ void vff_sums(int nparts, const double *__restrict__ part, double *s,
                                         double (&v)[kVffSums]) {
#pragma unroll
  for (int k = 0; k < kVffSums; ++k) v[k] = 0.0;
  for (int p = threadIdx.x; p < nparts; p += kRedThreads)
#pragma unroll
    for (int k = 0; k < kVffSums; ++k) v[k] += part[kVffSums * p + k];
  vff_block_sums(v, s);
}

// positions of displacements u (atoms' species in w)
__global__ void k_vff_pos(int A, const double *__restrict__ u,
                          const int32_t *__restrict__ species, double4 *__restrict__ pos) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < A) pos[i] = make_double4(u[3 * i], u[3 * i + 1], u[3 * i + 2], (double)species[i]);
}
__global__ __launch_bounds__(kRedThreads) void k_vff_total(int nparts,
                                                           const double *__restrict__ part,
                                                           double *__restrict__ out) {
  __shared__ double s[kVffSums * kRedThreads / 64];
  double v[kVffSums];
  vff_sums(nparts, part, s, v);
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < kVffSums; ++k) out[k] = v[k];
}

// The descent between two gradients: sums the last one's partials (every
// workgroup, the same bits), and either takes the line search's next point or
// accepts the point and takes the next direction (Polak-Ribiere+); writes the
// positions of the next gradient.  The state is read from s0 and left in s1
// (all workgroups read it).
__global__ __launch_bounds__(kRedThreads) void k_vff_step(
    int A, int nparts, const double *__restrict__ part, const VffState *__restrict__ s0,
    VffState *__restrict__ s1, int first, int max_iter, double gtol, double *__restrict__ u,
    double *__restrict__ d, const double *__restrict__ grad0, const double *__restrict__ grad1,
    double4 *__restrict__ pos) {
  __shared__ double scratch[kVffSums * kRedThreads / 64];
  VffState st{};
  if (!first) st = *s0;
  if (!first && st.done) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *s1 = st;
    return;
  }
  double v[kVffSums];
  vff_sums(nparts, part, scratch, v);
  const double gg = v[1], f1 = v[2], go = v[3];
  bool accept = true;
  double t = 0.0, bet = 0.0;  // u += t d, d = -grad + bet d
  if (first) {
    st.e0 = v[0];
    st.g0 = sqrt(gg);
    st.step = 1e-4;
  } else if (st.ls < 8 && !(fabs(f1) <= 1e-3 * fabs(st.dg0))) {
    // secant search for phi'(t) = grad(u + t d) . d = 0; the point after the
    // eighth is taken as it is
    double tn;
    if (f1 < 0.0 && f1 <= st.f0) tn = 2.0 * st.t1;  // still descending: expand
    else tn = st.t1 - f1 * (st.t1 - st.t0) / (f1 - st.f0);
    if (!(tn > 0.0) || !isfinite(tn)) tn = 0.5 * st.t1;
    st.t0 = st.t1;
    st.f0 = f1;
    st.t1 = tn;
    ++st.ls;
    accept = false;
  }
  if (accept) {
    if (!first) {
      st.step = t = st.t1;
      bet = (gg - go) / st.gg;
      if (bet < 0.0) bet = 0.0;
      ++st.it;
    }
    // slope along the new direction; not a descent direction: along -grad
    st.dg0 = bet == 0.0 ? -gg : bet * f1 - gg;
    if (st.dg0 >= 0.0) {
      bet = 0.0;
      st.dg0 = -gg;
    }
    st.gg = gg;
    st.par ^= 1;
    st.ls = 0;
    st.t0 = 0.0;
    st.f0 = st.dg0;
    st.t1 = st.step;
    st.done = !(st.it < max_iter && sqrt(gg) > gtol);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) *s1 = st;
  const double *grad = st.par ? grad1 : grad0;
  const double tp = st.done ? 0.0 : st.t1;
  for (int i = blockIdx.x * kRedThreads + threadIdx.x; i < A; i += gridDim.x * kRedThreads) {
    double p[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int64_t o = (int64_t)i * 3 + k;
      double x = u[o], y = first ? 0.0 : d[o];
      if (accept) {
        if (!first) u[o] = x = __builtin_fma(t, y, x);
        // bet = 0 drops d altogether (0 * NaN is NaN)
        d[o] = y = bet == 0.0 ? -grad[o] : __builtin_fma(bet, y, -grad[o]);
      }
      p[k] = st.done ? x : __builtin_fma(tp, y, x);
    }
    double4 *q = pos + i;
    q->x = p[0];
    q->y = p[1];
    q->z = p[2];
  }
}

void launch_grad(hipStream_t s, int blocks, const VffArgs &g, const double4 *pos, double *g0,
                 double *g1, const double *dir, const VffState *st, double *part) {
  if (g.model == NH_VFF_KEATING)
    hipLaunchKernelGGL(k_vff_grad<NH_VFF_KEATING>, dim3(blocks), dim3(kRedThreads), 0, s, g, pos,
                       g0, g1, dir, st, part);
  else
    hipLaunchKernelGGL(k_vff_grad<NH_VFF_KEATING_STRAINED>, dim3(blocks), dim3(kRedThreads), 0, s,
                       g, pos, g0, g1, dir, st, part);
}
// workgroups of a gradient: four a compute unit (its registers), whose sums
// the step reads in every workgroup (104,976 atoms: 820, 1024 and 1640
// workgroups 17.7, 16.7 and 17.8 us)
int vff_grid(int A) {
  return std::min((int)(((int64_t)A * 4 + kRedThreads - 1) / kRedThreads), 1024);
}

class Vff {
 public:
  Vff(nh_context *c, VffArgs a) : c_(c), g_(a) {}
  ~Vff() {
    for (void *p : mem_) pool_release(c_, p);
  }
  nh_status run(int max_iter, double gtol, double *out_disp, double *info);

 private:
  nh_status alloc(void **p, size_t bytes) {
    NH_TRY(pool_alloc(c_, p, bytes));
    mem_.push_back(*p);
    return NH_OK;
  }

  nh_context *c_;
  VffArgs g_;
  std::vector<void *> mem_;
};

nh_status Vff::run(int max_iter, double gtol, double *out_disp, double *info) {
  const int A = g_.A;
  const size_t n3 = (size_t)A * 3;
  NH_TRY(ensure_reduce(c_, 1));
  const int gb = vff_grid(A), sb = std::min((A + kRedThreads - 1) / kRedThreads, 512);
  double *u, *d, *gr[2], *part;
  double4 *pos;
  VffState *st;
  NH_TRY(alloc((void **)&u, n3 * sizeof(double)));
  NH_TRY(alloc((void **)&d, n3 * sizeof(double)));
  for (double *&q : gr) NH_TRY(alloc((void **)&q, n3 * sizeof(double)));
  NH_TRY(alloc((void **)&pos, (size_t)A * sizeof(double4)));
  NH_TRY(alloc((void **)&part, ((size_t)gb + 1) * kVffSums * sizeof(double)));
  NH_TRY(alloc((void **)&st, 2 * sizeof(VffState)));
  hipStream_t s = c_->stream;
  NH_HIP(hipMemcpyAsync(u, c_->disp, n3 * sizeof(double), hipMemcpyDeviceToDevice, s));
  hipLaunchKernelGGL(k_vff_pos, dim3((A + 255) / 256), dim3(256), 0, s, A, u, g_.species, pos);
  launch_grad(s, gb, g_, pos, gr[0], gr[1], nullptr, nullptr, part);
  int cur = 0;  // which of st[] holds the state
  auto step = [&](int first) {
    hipLaunchKernelGGL(k_vff_step, dim3(sb), dim3(kRedThreads), 0, s, A, gb, part, st + cur,
                       st + (cur ^ 1), first, max_iter, gtol, u, d, gr[0], gr[1], pos);
    cur ^= 1;
  };
  step(1);
  NH_HIP(hipGetLastError());
  // batches of points; the host looks at one batch's state while the next
  // runs (what is queued beyond the end does nothing)
  constexpr int kBatch = 8;
  static_assert(2 * sizeof(VffState) <= 64 * sizeof(double), "pinned buffer");
  VffState *seen = reinterpret_cast<VffState *>(c_->hred);
  struct Events {
    hipEvent_t e[2] = {nullptr, nullptr};
    ~Events() {
      for (hipEvent_t q : e)
        if (q) (void)hipEventDestroy(q);
    }
  } ev;
  for (hipEvent_t &e : ev.e) NH_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  int last = 0;
  for (int b = 0;; ++b) {
    NH_HIP(hipMemcpyAsync(seen + (b & 1), st + cur, sizeof(VffState), hipMemcpyDeviceToHost, s));
    NH_HIP(hipEventRecord(ev.e[b & 1], s));
    if (b > 0) {
      last = (b - 1) & 1;
      NH_HIP(hipEventSynchronize(ev.e[last]));
      if (seen[last].done) break;
    }
    for (int k = 0; k < kBatch; ++k) {
      launch_grad(s, gb, g_, pos, gr[0], gr[1], d, st + cur, part);
      step(0);
    }
    NH_HIP(hipGetLastError());
  }
  // the energy at the end; the gradient buffer is free by now
  double *total = part + (size_t)gb * kVffSums;
  launch_grad(s, gb, g_, pos, gr[0], gr[1], nullptr, nullptr, part);
  hipLaunchKernelGGL(k_vff_total, dim3(1), dim3(kRedThreads), 0, s, gb, part, total);
  NH_HIP(hipGetLastError());
  double e = 0.0;
  NH_HIP(hipMemcpyAsync(&e, total, sizeof(double), hipMemcpyDeviceToHost, s));
  NH_HIP(hipMemcpyAsync(c_->disp, u, n3 * sizeof(double), hipMemcpyDeviceToDevice, s));
  if (out_disp)
    NH_HIP(hipMemcpyAsync(out_disp, u, n3 * sizeof(double), hipMemcpyDeviceToHost, s));
  NH_HIP(hipStreamSynchronize(s));
  info[0] = seen[last].it;
  info[1] = seen[last].e0;
  info[2] = e;
  info[3] = seen[last].g0;
  info[4] = std::sqrt(seen[last].gg);
  return NH_OK;
}

}  // namespace
}  // namespace nh

namespace nh {
namespace {

// The parameter tables of a model on the device (six [S][S] tables in one
// allocation), freed with the object.
class VffTables {
 public:
  ~VffTables() { (void)hipFree(mem_); }
  nh_status upload(nh_context *c, const nh_vff_params *p) {
    NH_CHECK(p && p->alpha && p->beta && p->a0 &&
                 (p->model == NH_VFF_KEATING ||
                  (p->model == NH_VFF_KEATING_STRAINED && p->aa && p->ba && p->ca)) &&
                 (p->fix_surface == 0 || p->fix_surface == 1),
             NH_ERR_ARG, "VFF: bad parameters (model %d, fix_surface %d)",
             p ? p->model : -1, p ? p->fix_surface : -1);
    const size_t ss = (size_t)c->n_species * c->n_species;
    NH_TRY(device_malloc(c, (void **)&mem_, 6 * ss * sizeof(double)));
    const double *src[6] = {p->alpha, p->beta, p->a0, p->aa, p->ba, p->ca};
    for (int k = 0; k < 6; ++k)
      if (src[k])
        NH_HIP(hipMemcpy(mem_ + k * ss, src[k], ss * sizeof(double),
                         hipMemcpyHostToDevice));
    args = VffArgs{c->n_atoms, c->n_species, c->species, c->nbr, c->bond_q,
                   mem_, mem_ + ss, mem_ + 2 * ss, c->lattice[0], c->lattice[1],
                   c->lattice[2], mem_ + 3 * ss, mem_ + 4 * ss, mem_ + 5 * ss,
                   p->model, p->fix_surface};
    return NH_OK;
  }
  VffArgs args{};

 private:
  double *mem_ = nullptr;
};

nh_status energy_grad(nh_context *ctx, const nh_vff_params *p,
                      const double *disp, double *grad_out, double *energy) {
  NH_CHECK(ctx && disp && grad_out && energy, NH_ERR_ARG,
           "nh_vff_energy_grad: bad arguments");
  (void)hipGetLastError();
  NH_HIP(hipSetDevice(ctx->device));
  VffTables t;
  NH_TRY(t.upload(ctx, p));
  const int A = ctx->n_atoms;
  const int gb = vff_grid(A);
  // displacements, gradient, positions, partial sums
  void *m[4] = {nullptr, nullptr, nullptr, nullptr};
  const size_t sz[4] = {(size_t)A * 3 * sizeof(double), (size_t)A * 3 * sizeof(double),
                        (size_t)A * sizeof(double4),
                        ((size_t)gb + 1) * kVffSums * sizeof(double)};
  nh_status st = NH_OK;
  for (int k = 0; k < 4 && st == NH_OK; ++k) st = device_malloc(ctx, &m[k], sz[k]);
  hipError_t e = hipSuccess;
  double res[2] = {0, 0};
  if (st == NH_OK) {
    double *u = (double *)m[0], *gr = (double *)m[1], *part = (double *)m[3];
    double *total = part + (size_t)gb * kVffSums;
    double4 *pos = (double4 *)m[2];
    e = hipMemcpy(u, disp, sz[0], hipMemcpyHostToDevice);
    if (e == hipSuccess) {
      hipLaunchKernelGGL(k_vff_pos, dim3((A + 255) / 256), dim3(256), 0, ctx->stream, A, u,
                         t.args.species, pos);
      launch_grad(ctx->stream, gb, t.args, pos, nullptr, gr, nullptr, nullptr, part);
      hipLaunchKernelGGL(k_vff_total, dim3(1), dim3(kRedThreads), 0, ctx->stream, gb, part,
                         total);
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(grad_out, gr, sz[1], hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(res, total, sizeof(double), hipMemcpyDeviceToHost);
  }
  for (void *q : m) (void)hipFree(q);
  NH_TRY(st);
  NH_CHECK(e == hipSuccess, NH_ERR_HIP, "nh_vff_energy_grad: %s", hipGetErrorString(e));
  *energy = res[0];
  return NH_OK;
}

nh_status relax(nh_context *ctx, const nh_vff_params *p, int max_iter,
                double gtol, double *disp_out, double *info) {
  NH_CHECK(ctx && info && max_iter >= 0 && gtol >= 0, NH_ERR_ARG,
           "nh_vff_relax: bad arguments");
  (void)hipGetLastError();
  NH_HIP(hipSetDevice(ctx->device));
  VffTables t;
  NH_TRY(t.upload(ctx, p));
  Vff v(ctx, t.args);
  return v.run(max_iter, gtol, disp_out, info);
}

nh_vff_params keating(const double *alpha, const double *beta, const double *a0) {
  return nh_vff_params{alpha, beta, a0, nullptr, nullptr, nullptr,
                       NH_VFF_KEATING, 1};
}

}  // namespace
}  // namespace nh

extern "C" nh_status nh_vff_energy_grad(nh_context *ctx, const double *alpha,
                                        const double *beta, const double *a0,
                                        const double *disp, double *grad_out,
                                        double *energy) {
  const nh_vff_params p = nh::keating(alpha, beta, a0);
  return nh::energy_grad(ctx, &p, disp, grad_out, energy);
}

extern "C" nh_status nh_vff_relax(nh_context *ctx, const double *alpha,
                                  const double *beta, const double *a0,
                                  int max_iter, double gtol, double *disp_out,
                                  double *info) {
  const nh_vff_params p = nh::keating(alpha, beta, a0);
  return nh::relax(ctx, &p, max_iter, gtol, disp_out, info);
}

extern "C" nh_status nh_vff_energy_grad_model(nh_context *ctx,
                                              const nh_vff_params *p,
                                              const double *disp,
                                              double *grad_out, double *energy) {
  return nh::energy_grad(ctx, p, disp, grad_out, energy);
}

extern "C" nh_status nh_vff_relax_model(nh_context *ctx, const nh_vff_params *p,
                                        int max_iter, double gtol,
                                        double *disp_out, double *info) {
  return nh::relax(ctx, p, max_iter, gtol, disp_out, info);
}
