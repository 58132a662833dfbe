// On-device assembly of the sp3d5s* Hamiltonian.
//
// k_assemble: a quad of lanes per atom, a lane per neighbour slot.  A lane
// evaluates its bond in the cation's frame (so both rows of a bond get the
// same bits), writes what the layout stores of it (its own row's 10x10 block,
// or, the cation's lane, the SK record) and the Boykin diagonal corrections
// of its own atom (H_DiagStrainCorr_OffDiag_Wrapper + h3d_offdiag_diag_corr,
// h_cvectr_mult.c:1007-1126, mb_ham_spds_micro.c:597-1451); the quad adds
// them up and builds the onsite record: neighbour-averaged parameters, strain
// reference shift, dangling-bond passivation, potential and corrections
// (H_Diag_Wrapper, h_cvectr_mult.c:841-1005; h3d_diag,
// mb_ham_spds_micro.c:1453-1505; h3d_diag_dangling_bond_shift_zincblende,
// mb_ham_spds_micro.c:1910-2152).
// Each bond is evaluated from both ends: that costs 15 exponentials and about
// 300 operations a bond and saves a pass over 320 B an atom of corrections.
// The corrections are sums of squares of a row of the block less those of the
// unstrained block; the squares of a shell pair add up to its integrals'
// squares weighted by the row's angular functions, so neither block is formed
// (two tables of 100 numbers in scratch, a division per entry and 21 powers a
// bond took 0.86 ms for 395,136 atoms, the onsite records 0.07 and the fills
// 0.04; this 0.19 ms, 0.21 GB written; bound by the FP64 operations and the
// parameters' loads at two wavefronts a SIMD).
#include <utility>

#include "nh_internal.h"
#include "nh_hv_sk.h"

namespace nh {
namespace {

// Strained bond seen from the cation: nnv, nnv0 point anion -> cation
// (getRelativePosVec, geo_struct.c:2278-2294, with the cation-row sign
// flip of h_cvectr_mult.c:1073-1090).
__device__ __forceinline__ void cation_bond_vectors(
    const int32_t *bond_q, const double *disp, const double *lat, int i,
    int slot, int j, double a0, double nnv[3], double nnv0[3]) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double nrm = 0.25 * bond_q[(i * 4 + slot) * 3 + k];
    nnv0[k] = -(a0 * nrm);
    nnv[k] = -(lat[k] * nrm + disp[j * 3 + k] - disp[i * 3 + k]);
  }
}

// Integrals (index in parameters 10..30) of a shell of the anion with a shell
// of the cation: sigma, then pi, delta (-1: none)
__host__ __device__ constexpr int pair_integral(int sa, int sc, int part) {
  constexpr int s[16] = {1, 2, 6, 10, 3, 0, 4, 8, 7, 5, 12, 14, 11, 9, 15, 18};
  return part == 0 ? s[sa * 4 + sc]
         : sa == 2 && sc == 2 ? (part == 1 ? 13 : -1)
         : sa == 2 && sc == 3 ? (part == 1 ? 16 : -1)
         : sa == 3 && sc == 2 ? (part == 1 ? 17 : -1)
         : sa == 3 && sc == 3 ? 18 + part : -1;
}
// Weights of the squared sigma, pi and delta integrals in the sum of squares
// over a row of a shell pair, for the true sqrt 3; then what the reference's
// literal s changes of it (1e-12 relative): its first four d functions in s-d
// and p-d and its z2 entries of p-d pi and d-d are s / sqrt 3 times as large, so that
// a sum over the other shell's d functions gains k = s^2 / 3 - 1 times the
// squares of those entries (the products of sigma and pi still add up to 0).
struct RowWeights {
  static constexpr double k = kSqrt3Ref * kSqrt3Ref / 3.0 - 1.0;
  double p[3], ds[5], dp[5], dd[5], z;
  __device__ __forceinline__ RowWeights(double l, double m, double n) {
    const double l2 = l * l, m2 = m * m, n2 = n * n, dl = l2 - m2, lpm = l2 + m2;
    z = n2 - 0.5 * lpm;
    p[0] = l2, p[1] = m2, p[2] = n2;
    ds[0] = 3.0 * l2 * m2, ds[1] = 3.0 * m2 * n2, ds[2] = 3.0 * n2 * l2;
    ds[3] = 0.75 * dl * dl, ds[4] = z * z;
    dp[0] = lpm - 4.0 * l2 * m2, dp[1] = m2 + n2 - 4.0 * m2 * n2;
    dp[2] = n2 + l2 - 4.0 * n2 * l2, dp[3] = lpm - dl * dl, dp[4] = 3.0 * n2 * lpm;
    dd[0] = n2 + l2 * m2, dd[1] = l2 + m2 * n2, dd[2] = m2 + n2 * l2;
    dd[3] = n2 + 0.25 * dl * dl, dd[4] = 0.75 * lpm * lpm;
  }
  // sum over the row of orbital O (0..9) with shell X, q the squares of the
  // pair's integrals
  template <int O, int X>
  __device__ __forceinline__ double row(const double (&q)[3]) const {
    const double s3 = X == 3 ? 1.0 + k * (1.0 - ds[4]) : 1.0;
    if constexpr (O < 2) {
      return s3 * q[0];
    } else if constexpr (O < 5) {
      const double a = p[O - 2], w = O < 4 ? p[2] : 1.0 - p[2];
      return (a * s3) * q[0] + (1.0 - a + (X == 3 ? 3.0 * k * a * w * w : 0.0)) * q[1];
    } else if constexpr (X == 3) {
      return ds[O - 5] * q[0] + dp[O - 5] * q[1] + dd[O - 5] * q[2];
    } else {
      return (O < 9 ? 1.0 + k : 1.0) * ds[O - 5] * q[0] +
             (O == 9 ? 1.0 + k : 1.0) * dp[O - 5] * q[1];
    }
  }
  // the literal's part of the d-d rows
  __device__ __forceinline__ void add_dd(double dds, double ddp, double ddd,
                                         double (&r)[5]) const {
    const double y = z * dds - 2.0 * p[2] * ddp + 0.5 * (1.0 + p[2]) * ddd;
    const double w = z * dds + (1.0 - 2.0 * p[2]) * ddp - 0.5 * (1.0 - p[2]) * ddd;
    const double y2 = k * y * y, w2 = k * w * w;
    const double e[4] = {ds[0] * y2, ds[1] * w2, ds[2] * w2, ds[3] * y2};
#pragma unroll
    for (int c = 0; c < 4; ++c) r[c] += e[c];
    r[4] += (e[0] + e[1]) + (e[2] + e[3]);
  }
};

template <int N, typename F, int... I>
__device__ __forceinline__ void static_for_(F &f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F f) {
  static_for_<N>(f, std::make_integer_sequence<int, N>{});
}

// s + the quad's four x in slot order, in every lane
__device__ __forceinline__ double quad_add(double s, double x) {
  s += dpp_f64<0x00>(x);
  s += dpp_f64<0x55>(x);
  s += dpp_f64<0xAA>(x);
  return s + dpp_f64<0xFF>(x);
}

struct AssembleArgs {
  int A, S, passivate;
  const int32_t *species, *is_cation, *nbr, *rev_slot, *bond_q, *bond_of;
  const double *disp, *parmat, *strnmat, *phi;
  double lx, ly, lz, db_shift;
  double *onsite, *blocks, *sk;
};

enum { kOnsiteOnly = 0, kStoreBlocks = 1, kStoreSk = 2 };
constexpr int kAsmThreads = 128, kAsmAtoms = kAsmThreads / 4;
template <int STORE>
__global__ __launch_bounds__(kAsmThreads) void k_assemble(AssembleArgs g) {
  // onsite and bond records on their way out (24 doubles a bond, padded
  // against bank conflicts)
  constexpr int kRow = kSkStride + 1;
  __shared__ double lds[kAsmAtoms * kOnsiteStride];
  __shared__ double recs[STORE == kStoreSk ? kAsmThreads * kRow : 1];
  __shared__ int32_t rec_of[kAsmAtoms];
  const int slot = threadIdx.x & 3, la = threadIdx.x >> 2;
  const int i = blockIdx.x * kAsmAtoms + la;
  const bool in = i < g.A;
  const int j = in ? g.nbr[i * 4 + slot] : -1;
  const bool here = j >= 0;
  const bool cat = in && g.is_cation[i] != 0;
  double corr[10], e[10], strain_shift = 0.0;
#pragma unroll
  for (int k = 0; k < 10; ++k) corr[k] = e[k] = 0.0;
  if (STORE == kStoreSk && !here)
#pragma unroll
    for (int k = 0; k < kSkStride; ++k) recs[threadIdx.x * kRow + k] = 0.0;
  if (STORE == kStoreBlocks && in && !here) {
    double *B = g.blocks + ((size_t)i * 4 + slot) * 100;
    for (int k = 0; k < 100; ++k) B[k] = 0.0;
  }
  if (here) {
    const int ti = g.species[i], tj = g.species[j];
    const int c = cat ? ti : tj, a = cat ? tj : ti;
    const double *par = g.parmat + ((size_t)c * g.S + a) * 35;
    const double *strn = g.strnmat + ((size_t)c * g.S + a) * 33;
    const double lat[3] = {g.lx, g.ly, g.lz};
    const int back = g.rev_slot[i * 4 + slot];
    double nnv[3], nnv0[3];
    if (cat) cation_bond_vectors(g.bond_q, g.disp, lat, i, slot, j, par[P_A0], nnv, nnv0);
    else cation_bond_vectors(g.bond_q, g.disp, lat, j, back, i, par[P_A0], nnv, nnv0);
    const BondGeom b = bond_geom(nnv, nnv0, par[P_A0]);
    double v[21];
    scale_integrals(par, strn, b.brat, v);
    if constexpr (STORE == kStoreBlocks) {
      double T[100];
      sk_table(b.l, b.m, b.n, v, T);
      double *B = g.blocks + ((size_t)i * 4 + slot) * 100;
#pragma unroll
      for (int r = 0; r < 10; ++r)
#pragma unroll
        for (int q = 0; q < 10; ++q) {
          const double x = T[r * 10 + q], y = T[q * 10 + r];
          B[r * 10 + q] = cat ? y : x;
        }
    }
    if constexpr (STORE == kStoreSk)
      if (cat) {
        double rec[kSkStride];
        sk_record(b.l, b.m, b.n, v, rec);
#pragma unroll
        for (int k = 0; k < kSkStride; ++k) recs[threadIdx.x * kRow + k] = rec[k];
      }
    // Boykin terms ((V0^2 - V^2) c_strain / (E_a + E_c)) * c_pair
    // (mb_ham_spds_VoffdEdiag_constructors.h; the pVpE_* macros are not
    // parenthesised, so the pair coefficient multiplies the quotient).
    const RowWeights w(b.l, b.m, b.n), w0(b.l0, b.m0, b.n0);
    const double cs = strn[S_CONST];
    auto pair = [&](auto SO, auto SX) {
      constexpr int so = SO, sx = SX;  // shells of this atom, of the other
      const double ea = par[cat ? e_anion(sx) : e_anion(so)];
      const double ec = par[cat ? e_cation(so) : e_cation(sx)];
      const double f = cs / (ea + ec) * strn[cat ? cpair_index(sx, so) : cpair_index(so, sx)];
      double q[3], q0[3];
#pragma unroll
      for (int part = 0; part < 3; ++part) {
        q[part] = q0[part] = 0.0;
        if (pair_integral(so, sx, part) < 0) continue;
        const int ia = pair_integral(so, sx, part), ic = pair_integral(sx, so, part);
        const double x = cat ? v[ic] : v[ia], x0 = par[10 + (cat ? ic : ia)];
        q[part] = x * x;
        q0[part] = x0 * x0;
      }
      double lit[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
      if constexpr (so == 3 && sx == 3) {
        double less[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        w0.add_dd(par[P_DDS], par[P_DDP], par[P_DDD], lit);
        w.add_dd(v[18], v[19], v[20], less);
#pragma unroll
        for (int c = 0; c < 5; ++c) lit[c] -= less[c];
      }
      auto add = [&](auto O) {
        constexpr int o = O;
        if constexpr (shell_of(o) == so) {
          double dif = w0.template row<o, sx>(q0) - w.template row<o, sx>(q);
          if constexpr (so == 3 && sx == 3) dif += lit[o - 5];
          corr[o] += dif * f;
        }
      };
      static_for<10>(add);
    };
    static_for<4>([&](auto SO) { static_for<4>([&](auto SX) { pair(SO, SX); }); });
    // of the averaged parameters only the onsite energies and the spin-orbit
    // constants are used
#pragma unroll
    for (int k = 0; k < 10; ++k) e[k] = par[k];
    strain_shift = strn[cat ? S_CAT_SHIFT : S_AN_SHIFT];
  }
  const int cnt = (int)quad_add(0.0, here ? 1.0 : 0.0);
  strain_shift = quad_add(0.0, strain_shift) / cnt;
#pragma unroll
  for (int k = 0; k < 10; ++k) e[k] = quad_add(0.0, e[k]) / cnt;
  double hd[10];
#pragma unroll
  for (int o = 0; o < 10; ++o) {
    const double ec = e[e_cation(shell_of(o))], ea = e[e_anion(shell_of(o))];
    hd[o] = cat ? ec : ea;
  }
  double sp[6] = {0, 0, 0, 0, 0, 0};
  if (g.passivate && in && cnt < 4) {
    // sp3 hybrid directions of the dangling-bond projector
    const double hyb[4][3] = {{0.25, 0.25, 0.25},
                              {-0.25, -0.25, 0.25},
                              {0.25, -0.25, -0.25},
                              {-0.25, 0.25, -0.25}};
    double v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = 0.25 * g.db_shift;
    double cosv = 0.0;
    for (int n = 0; n < 4; ++n) {
      double d[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) d[k] = 0.25 * g.bond_q[(i * 4 + n) * 3 + k];
      int ib = 0;
      cosv = d[0] * hyb[0][0] + d[1] * hyb[0][1] + d[2] * hyb[0][2];
      while (fabs(cosv) < 0.15 && ib < 3) {
        ++ib;
        cosv = d[0] * hyb[ib][0] + d[1] * hyb[ib][1] + d[2] * hyb[ib][2];
      }
      if (g.nbr[i * 4 + n] >= 0) v[ib] = 0.0;
    }
    const double s = cosv > 0 ? 1.0 : -1.0;
    const double dsp = v[0] + v[1] + v[2] + v[3];
    sp[0] = s * (v[0] - v[1] + v[2] - v[3]);
    sp[1] = s * (v[0] - v[1] - v[2] + v[3]);
    sp[2] = s * (v[0] + v[1] - v[2] - v[3]);
    sp[3] = v[0] + v[1] - v[2] - v[3];
    sp[4] = v[0] - v[1] - v[2] + v[3];
    sp[5] = v[0] - v[1] + v[2] - v[3];
#pragma unroll
    for (int k = 1; k < 5; ++k) hd[k] += dsp;
  }
  const double ph = in && g.phi ? g.phi[i] : 0.0;
#pragma unroll
  for (int k = 0; k < 10; ++k) hd[k] = quad_add(hd[k] + strain_shift - ph, corr[k]);
  // through LDS, so that consecutive lanes write consecutive numbers
  const int a0 = blockIdx.x * kAsmAtoms, na = min(kAsmAtoms, g.A - a0);
  if (slot == 0) {
    double *os = lds + la * kOnsiteStride;
#pragma unroll
    for (int k = 0; k < 10; ++k) os[k] = hd[k];
#pragma unroll
    for (int k = 0; k < 6; ++k) os[10 + k] = sp[k];
    os[16] = cat ? e[P_LC] : e[P_LA];
    os[17] = 0.0;
  }
  if constexpr (STORE == kStoreSk) {
    // a cation's four records follow one another (bond number 4 c + slot)
    if (here && cat) rec_of[la] = g.bond_of[i * 4 + slot] - slot;
    else if (slot == 0 && !cat) rec_of[la] = -1;
  }
  __syncthreads();
  for (int t = threadIdx.x; t < na * kOnsiteStride; t += kAsmThreads)
    g.onsite[(size_t)a0 * kOnsiteStride + t] = lds[t];
  if constexpr (STORE == kStoreSk) {
    for (int t = threadIdx.x; t < na * 4 * kSkStride; t += kAsmThreads) {
      const int r = t / kSkStride, k = t % kSkStride, rr = rec_of[r >> 2];
      if (rr >= 0) g.sk[((size_t)rr + (r & 3)) * kSkStride + k] = recs[r * kRow + k];
    }
  }
}

// Matrix-free layout tables: per atom its displacement and species, per
// slot the ideal bond vector seen from the bond's cation (cation rows keep
// their own vector, anion rows negate theirs), packed as 3 x int8.
__global__ void k_mf_geo(int A, const int32_t *__restrict__ species,
                         const int32_t *__restrict__ is_cation,
                         const int32_t *__restrict__ bond_q,
                         const double *__restrict__ disp,
                         double4 *__restrict__ geo, int32_t *__restrict__ q) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= A) return;
  geo[i] = make_double4(disp[i * 3], disp[i * 3 + 1], disp[i * 3 + 2],
                        (double)species[i]);
  const int sg = is_cation[i] ? 1 : -1;
  for (int n = 0; n < 4; ++n) {
    int packed = 0;
    for (int k = 0; k < 3; ++k)
      packed |= ((sg * bond_q[(i * 4 + n) * 3 + k]) & 0xff) << (8 * k);
    q[i * 4 + n] = packed;
  }
}

// The two atoms of every bond of the products' blocks: 4 cation atom + slot,
// anion atom (-1 pads).
__global__ void k_mf_ends(int n, const int32_t *__restrict__ bonds,
                          const int32_t *__restrict__ cations,
                          const int32_t *__restrict__ nbr, int2 *__restrict__ ends) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int b = bonds[k];
  const int e = b >= 0 ? cations[b >> 2] * 4 + (b & 3) : -1;
  ends[k] = make_int2(e, e >= 0 ? nbr[e] : -1);
}

// Per (cation, anion) species pair: integrals 10..30, strain exponents
// 0..14, lattice constant (the parameters k_assemble reads).
__global__ void k_mf_pair(int S, const double *__restrict__ parmat,
                          const double *__restrict__ strnmat,
                          double *__restrict__ pair) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= S * S) return;
  const double *par = parmat + (size_t)p * 35;
  const double *strn = strnmat + (size_t)p * 33;
  double *o = pair + (size_t)p * kMfPair;
  for (int k = 0; k < 21; ++k) o[k] = par[10 + k];
  for (int e = 0; e < 15; ++e) o[kMfEta + e] = strn[e];
  o[kMfA0] = par[P_A0];
  for (int k = kMfA0 + 1; k < kMfPair; ++k) o[k] = 0.0;
}

template <typename T>
__global__ void k_convert(int64_t n, const double *__restrict__ src,
                          T *__restrict__ dst) {
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * blockDim.x)
    dst[k] = T(src[k]);
}

// FP32 SK records (sk_round), a record a thread
__global__ __launch_bounds__(256) void k_sk32(int64_t n, const double4 *__restrict__ src,
                                              float4 *__restrict__ dst) {
  const int64_t b = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (b >= n) return;
  double d[kSkStride];
  float k[kSkStride];
#pragma unroll
  for (int i = 0; i < kSkStride / 4; ++i) {
    const double4 v = src[b * (kSkStride / 4) + i];
    d[4 * i] = v.x, d[4 * i + 1] = v.y, d[4 * i + 2] = v.z, d[4 * i + 3] = v.w;
  }
  sk_round(d, k);
#pragma unroll
  for (int i = 0; i < kSkStride / 4; ++i)
    dst[b * (kSkStride / 4) + i] = make_float4(k[4 * i], k[4 * i + 1], k[4 * i + 2], k[4 * i + 3]);
}

inline int grid_for(int64_t n, int block) {
  int64_t g = (n + block - 1) / block;
  return (int)(g < 1 ? 1 : g);
}

}  // namespace

// What a rebuild does not use of the last build is freed; the rest is written
// again (its sizes depend on the context alone).  Freeing and allocating all
// of it took most of a rebuild (786,520 atoms: 2 GB).
static void free_ham(nh_context *c, int layout) {
  auto drop = [](auto *&p) {
    (void)hipFree(p);
    p = nullptr;
  };
  if (layout != NH_LAYOUT_BLOCKS) drop(c->blocks64);
  // FP32 copies are derived anew (select_precision)
  drop(c->blocks32);
  drop(c->sk32);
  if (layout != NH_LAYOUT_SK) drop(c->sk64);
  if (layout != NH_LAYOUT_MATRIX_FREE) {
    drop(c->mf_geo);
    drop(c->mf_q);
    drop(c->mf_pair);
    drop(c->mf_ends);
  }
  c->layout = c->precision = -1;
}

nh_status assemble(nh_context *c, int layout, int precision) {
  NH_CHECK(layout == NH_LAYOUT_BLOCKS || layout == NH_LAYOUT_SK ||
               layout == NH_LAYOUT_MATRIX_FREE,
           NH_ERR_ARG, "layout %d not available", layout);
  NH_CHECK(precision == NH_PREC_FP64 || precision == NH_PREC_FP32, NH_ERR_ARG,
           "precision %d not available", precision);
  NH_HIP(hipStreamSynchronize(c->stream));
  free_ham(c, layout);
  if (layout != NH_LAYOUT_BLOCKS) NH_TRY(ensure_blocks(c));
  auto need = [c](auto **p, size_t bytes) {
    return *p ? NH_OK : device_malloc(c, (void **)p, bytes);
  };
  const int A = c->n_atoms;
  const size_t nblk = (size_t)A * 4 * 100;
  NH_TRY(need(&c->onsite, (size_t)A * kOnsiteStride * sizeof(double)));
  if (layout == NH_LAYOUT_BLOCKS) NH_TRY(need(&c->blocks64, nblk * sizeof(double)));
  if (layout == NH_LAYOUT_SK)
    NH_TRY(need(&c->sk64, (size_t)c->n_cations * 4 * kSkStride * sizeof(double)));
  const int S = c->n_species;
  if (layout == NH_LAYOUT_MATRIX_FREE) {
    NH_TRY(need(&c->mf_geo, (size_t)A * sizeof(double4)));
    NH_TRY(need(&c->mf_q, (size_t)A * 4 * sizeof(int32_t)));
    NH_TRY(need(&c->mf_pair, (size_t)S * S * kMfPair * sizeof(double)));
    hipLaunchKernelGGL(k_mf_geo, dim3(grid_for(A, 128)), dim3(128), 0, c->stream,
                       A, c->species, c->is_cation, c->bond_q, c->disp,
                       c->mf_geo, c->mf_q);
    const int ne = c->n_blocks * kSkBondPad;
    NH_TRY(need(&c->mf_ends, (size_t)ne * sizeof(int2)));
    hipLaunchKernelGGL(k_mf_ends, dim3(grid_for(ne, 256)), dim3(256), 0, c->stream, ne,
                       c->blk_bonds, c->cations, c->nbr, c->mf_ends);
    hipLaunchKernelGGL(k_mf_pair, dim3(1), dim3(64 * ((S * S + 63) / 64)), 0,
                       c->stream, S, c->parmat, c->strnmat, c->mf_pair);
    NH_HIP(hipGetLastError());
  }
  const AssembleArgs g{A, S, c->passivate, c->species, c->is_cation, c->nbr, c->rev_slot,
                       c->bond_q, c->bond_of, c->disp, c->parmat, c->strnmat, c->phi,
                       c->lattice[0], c->lattice[1], c->lattice[2], c->db_shift, c->onsite,
                       c->blocks64, c->sk64};
  const dim3 grid(grid_for(A, kAsmAtoms)), block(kAsmThreads);
  if (layout == NH_LAYOUT_BLOCKS)
    hipLaunchKernelGGL(k_assemble<kStoreBlocks>, grid, block, 0, c->stream, g);
  else if (layout == NH_LAYOUT_SK)
    hipLaunchKernelGGL(k_assemble<kStoreSk>, grid, block, 0, c->stream, g);
  else
    hipLaunchKernelGGL(k_assemble<kOnsiteOnly>, grid, block, 0, c->stream, g);
  NH_HIP(hipGetLastError());
  NH_HIP(hipStreamSynchronize(c->stream));
  c->layout = layout;
  c->precision = NH_PREC_FP64;
  return select_precision(c, precision);
}

nh_status select_precision(nh_context *c, int precision) {
  NH_CHECK(c->layout == NH_LAYOUT_BLOCKS || sk_like(c), NH_ERR_STATE,
           "build the Hamiltonian first");
  NH_CHECK(precision == NH_PREC_FP64 || precision == NH_PREC_FP32, NH_ERR_ARG,
           "precision %d not available", precision);
  const int A = c->n_atoms;
  if (precision == NH_PREC_FP32) {
    // the FP64 values are always kept: derive the FP32 blocks or records once
    // (the matrix-free layout needs none; onsite terms are FP64 always)
    if (c->layout == NH_LAYOUT_BLOCKS && !c->blocks32) {
      const size_t nblk = (size_t)A * 4 * 100;
      NH_TRY(device_malloc(c, (void **)&c->blocks32, nblk * sizeof(float)));
      hipLaunchKernelGGL(k_convert<float>, dim3(4096), dim3(256), 0, c->stream,
                         (int64_t)nblk, c->blocks64, c->blocks32);
    }
    if (c->layout == NH_LAYOUT_SK && !c->sk32) {
      const int64_t nr = (int64_t)c->n_cations * 4;
      NH_TRY(device_malloc(c, (void **)&c->sk32, nr * kSkStride * sizeof(float)));
      hipLaunchKernelGGL(k_sk32, dim3(grid_for(nr, 256)), dim3(256), 0, c->stream, nr,
                         reinterpret_cast<const double4 *>(c->sk64),
                         reinterpret_cast<float4 *>(c->sk32));
    }
    NH_HIP(hipGetLastError());
    NH_HIP(hipStreamSynchronize(c->stream));
  }
  c->precision = precision;
  return NH_OK;
}

}  // namespace nh
