// H·v in the SK-compressed and matrix-free layouts: per bond only a record
// of 24 numbers (direction and combinations of the strain-scaled two-centre
// integrals, nh_sk_apply.h) is needed, stored once per bond (cation-owned) or
// recomputed from the atoms' displacements (MfSrc); the 10x10 block is never
// formed.  The onsite record (diagonal with Boykin corrections, surface
// couplings, spin-orbit) is stored per atom as in the block layout.
//
// Mapping: a workgroup of 256 threads takes a block of up to 32 cations and
// 32 anions from a cube of cells (2 x 2 x 2 cells in the bulk).  It stages
// the vector entries of its own atoms and of their other neighbours (the
// halo: 46 atoms on average) and the records of their bonds (154) in LDS,
// each once, a quad of lanes (64 bytes a load) per item, all loads in flight
// together; then a quad per atom computes, its lanes owning the four real
// component vectors of a 20-band atom (re and im of both spins): each lane
// applies the atom's four bonds to its component from LDS and adds them up in
// its own FP64 accumulators, so no sums cross lanes.  (10-band atoms have two
// components: the quad's halves take two bonds each and are added.)
// What bounds it: the traffic between L2 and the CUs.  Gathering each atom's
// four neighbours and both rows' records separately moved 2.55 GB through L2
// per FP64 product of a 786,520-atom dot (atom entries five times, records
// twice) and kept the texture addresser busy 76% of 255 us whatever the order
// of the atoms; the block moves the entries 1.7 times and the records 1.2
// times: 786,520 atoms FP64 0.312 -> 0.238 ms (SK), 8 columns of 395,136
// atoms 1.25 -> 0.65 ms (matrix-free); what is left is FP64 VALU (93 operations
// a bond, component and row) and LDS reads about evenly, behind 0.94 GB of HBM.
// The role (cation or anion) is uniform in a wavefront, so whether T or its
// transpose is applied is a scalar branch.
#pragma once

#include <type_traits>

#include "nh_internal.h"
#include "nh_sk_apply.h"

namespace nh {

// ---- blocks of atoms ---------------------------------------------------------

// Blocks (built by the first SK or matrix-free build, ensure_blocks): capacity
// 32 cations and 32 anions of its own, 64 more neighbours (the halo), 176
// bonds; -1 pads the tables.
constexpr int kSkOwn = 64, kSkHalo = 64, kSkBonds = 176, kSkBondPad = 192;
constexpr int kSkThreads = 256;

struct SkTable {
  const int32_t *own;   // [blocks][64] atoms (0-31 cations, 32-63 anions)
  const int32_t *halo;  // [blocks][64] atoms
  const uint2 *local;   // [blocks][64] a byte per slot: x: neighbour's place
                        // (own slot or 64 + halo place), y: bond's place; 255
  int n;                // blocks
  int per;              // blocks of an XCD, ceil(n / 8)
};
inline SkTable sk_table_of(const nh_context *c) {
  return SkTable{c->blk_own, c->blk_halo, c->blk_local,
                 c->n_blocks, (c->n_blocks + 7) / 8};
}
// Workgroups: as many as run at a time (`groups` a CU, 32 CUs an XCD), each
// taking block after block.  Consecutive workgroups go to different XCDs
// (round robin over 8): workgroup g runs on XCD g % 8 and takes the blocks
// (g % 8) per + g / 8, + grid / 8, ... < (g % 8 + 1) per, so each XCD works
// on a compact region of the crystal whose vector entries and records are
// shared in its L2.
inline int sk_grid(const nh_context *c, int groups) {
  const int per = (c->n_blocks + 7) / 8;
  return 8 * (per / 32 < groups ? per : 32 * groups);
}
struct SkWalk {
  int b, step, end;
  __device__ __forceinline__ explicit SkWalk(const SkTable &t) {
    const int x = blockIdx.x & 7;
    b = x * t.per + (int)(blockIdx.x >> 3);
    step = (int)(gridDim.x >> 3);
    end = min(t.n, (x + 1) * t.per);
  }
};

// Complex entries of the FP64 vector, or of an FP32 one widened on load
__device__ __forceinline__ double2 widen2(double2 v) { return v; }
__device__ __forceinline__ double2 widen2(float2 v) { return make_double2(v.x, v.y); }

// Staged items, in 16-byte chunks.  20 bands: the chunks of the two spins
// alternate, so the four components of an orbital that a quad's lanes read
// together lie in 32 bytes, and the stride is an odd number of 32 bytes: quads
// reading places that differ modulo 8 (see the places of a block) meet
// different banks.  10 bands: an odd number of chunks.
template <int NSP, typename XT>
struct SkX {  // the entries of an atom
  static constexpr int kChunks = NSP * 10 * (int)sizeof(XT) / 16;  // 20/10, 10/5
  static constexpr int kLoads = (kChunks + 3) / 4;                 // per lane of a quad
  // a place also holds an onsite record (9) or ten FP64 entries
  static constexpr int kStride =
      NSP == 2 ? (kChunks / 2 | 1) * 2 : (kChunks < 10 ? 10 : kChunks) | 1;
  // where chunk i lies
  __device__ __forceinline__ static int at(int i) {
    return NSP == 1 ? i : i < kChunks / 2 ? 2 * i : 2 * i - kChunks + 1;
  }
};
template <typename R>
struct SkRec {  // a bond record (24 numbers)
  static constexpr int kChunks = 24 * (int)sizeof(R) / 16;  // 12 / 6
  static constexpr int kLoads = (kChunks + 3) / 4;
  static constexpr int kStride = kChunks + 1;
};
constexpr int kOsChunks = kOnsiteStride / 2;

template <int NSP, typename R, typename XT>
struct SkLds {
  uint4 x[(kSkOwn + kSkHalo) * SkX<NSP, XT>::kStride];
  uint4 rec[kSkBonds * SkRec<R>::kStride];
};

// Exchange of a double between lanes through DPP moves
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)b, CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), CTRL, 0xF, 0xF, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) |
                                          (unsigned)lo));
}
constexpr int kQuadXor1 = 0xB1;  // quad_perm [1, 0, 3, 2]
constexpr int kQuadXor2 = 0x4E;  // quad_perm [2, 3, 0, 1]
constexpr int kQuadXor3 = 0x1B;  // quad_perm [3, 2, 1, 0]

// ---- FP32 / deferred Lanczos vectors ---------------------------------------

// Lanczos vectors in Paige's order: r_k = u_{k-1} - a r_{k-1}, a =
// alpha_{k-1} / beta_{k-1} (so that a r_{k-1} = alpha_{k-1} q_{k-1}),
// formed by the product as it reads u_{k-1} and r_{k-1}.
// FP32 vectors: a is split into two FP32 parts (a = hi + lo to 2^-48
// relative): two fmas, rounding entry by entry.  The coefficient must not be
// rounded to FP32 alone: its error is the same for every entry, i.e. an
// error along q_{k-1} in every step, which cost a 786,520-atom dot 10,251
// steps instead of 7,901 (and a level, from another start); with the split
// it takes the same 7,826 steps as one FP64 fma per entry.
// FP64 vectors: one fma.  Every kernel that forms r_k (the products that
// read u_{k-1} and r_{k-1}, the eigenvector pass that writes r_k) evaluates
// these expressions on the same operands, so they agree bit for bit.
template <typename XT>
struct LzCoef;
template <>
struct LzCoef<float2> {
  float hi, lo;
};
template <>
struct LzCoef<double2> {
  double a;
};
template <typename XT>
__device__ __forceinline__ LzCoef<XT> lz_defer_coef(double al, double inv) {
  const double a = al * inv;
  if constexpr (sizeof(XT) == 8) {
    const float hi = (float)a;
    return LzCoef<XT>{hi, (float)(a - (double)hi)};
  } else {
    return LzCoef<XT>{a};
  }
}
__device__ __forceinline__ float lz_defer1(float u, float rp, LzCoef<float2> a) {
  // the cancellation u - hi rp happens inside the first fma (one rounding
  // of the exact difference), then the small correction: about one ulp of
  // r in all (the other order adds half an ulp of u, which can be larger)
  return __builtin_fmaf(-a.lo, rp, __builtin_fmaf(-a.hi, rp, u));
}
__device__ __forceinline__ double lz_defer1(double u, double rp, LzCoef<double2> a) {
  return __builtin_fma(-a.a, rp, u);
}
// a 16-byte chunk of r_k: two FP32 entries or one FP64 entry
template <typename XT>
__device__ __forceinline__ uint4 lz_defer_chunk(uint4 u, uint4 rp, LzCoef<XT> a) {
  uint4 o;
  if constexpr (sizeof(XT) == 8) {
    o.x = __float_as_uint(lz_defer1(__uint_as_float(u.x), __uint_as_float(rp.x), a));
    o.y = __float_as_uint(lz_defer1(__uint_as_float(u.y), __uint_as_float(rp.y), a));
    o.z = __float_as_uint(lz_defer1(__uint_as_float(u.z), __uint_as_float(rp.z), a));
    o.w = __float_as_uint(lz_defer1(__uint_as_float(u.w), __uint_as_float(rp.w), a));
  } else {
    const double2 du = *reinterpret_cast<const double2 *>(&u);
    const double2 dr = *reinterpret_cast<const double2 *>(&rp);
    double2 r;
    r.x = lz_defer1(du.x, dr.x, a);
    r.y = lz_defer1(du.y, dr.y, a);
    o = *reinterpret_cast<const uint4 *>(&r);
  }
  return o;
}

// ---- bond records ------------------------------------------------------------

// A source of bond records: index() reads which records a block needs,
// load() requests what they are made of, stage() writes them to LDS.
//
// SkSrc: the stored SK layout, 24 numbers per bond (each bond once); the
// block's records are loaded by quads, one record a quad and round.
template <typename R>
struct SkSrc {
  const R *__restrict__ sk;
  const int32_t *__restrict__ bonds;

  static constexpr int kRounds = kSkBondPad / 64;
  struct Index {
    int b[kRounds];
  };
  struct Data {
    uint4 r[kRounds][SkRec<R>::kLoads];
  };
  __device__ __forceinline__ void index(int blk, Index &i) const {
#pragma unroll
    for (int k = 0; k < kRounds; ++k)
      i.b[k] = bonds[blk * kSkBondPad + 64 * k + (int)(threadIdx.x >> 2)];
  }
  __device__ __forceinline__ void load(const Index &i, Data &d) const {
    const int c = threadIdx.x & 3;
#pragma unroll
    for (int k = 0; k < kRounds; ++k)
#pragma unroll
      for (int q = 0; q < SkRec<R>::kLoads; ++q) {
        d.r[k][q] = make_uint4(0, 0, 0, 0);
        if (i.b[k] >= 0 && 4 * q + c < SkRec<R>::kChunks)
          d.r[k][q] = reinterpret_cast<const uint4 *>(sk + (size_t)i.b[k] * kSkStride)[4 * q + c];
      }
  }
  __device__ __forceinline__ void stage(const Data &d, uint4 *rec) const {
    const int Q = threadIdx.x >> 2, c = threadIdx.x & 3;
#pragma unroll
    for (int k = 0; k < kRounds; ++k)
#pragma unroll
      for (int q = 0; q < SkRec<R>::kLoads; ++q)
        if (64 * k + Q < kSkBonds && 4 * q + c < SkRec<R>::kChunks)
          rec[(64 * k + Q) * SkRec<R>::kStride + 4 * q + c] = d.r[k][q];
  }
};

// MfSrc: the matrix-free layout (the reference's HamCompute = Recompute,
// Hmult_spds_col, NEMO_3D/nemo3d/src/base/h_cvectr_mult.c:1134-1886): the
// record is recomputed on every product from the two atoms' displacements
// and species and the slot's ideal bond vector, as the assembly computes it
// (strain_corr_prep, mb_ham_spds_micro.c:2848-2978): direction cosines of
// the strained bond and the 21 integrals scaled by (d0/d)^eta, with
// (d0/d)^eta = exp(eta log(d0/d)) (one log and 15 exp per bond and block, a
// lane per bond).  Both rows of a bond get
// bit-identical records (the bond vector is formed in the cation's frame), so
// H stays exactly Hermitian.  With R = float the integrals are scaled in
// FP32 (geometry and the log in FP64).
template <typename R>
struct MfSrc {
  const int2 *__restrict__ ends;    // [blocks][192] 4 cation atom + slot, anion
  const double4 *__restrict__ geo;  // [A] displacement x, y, z (nm), species
  const int32_t *__restrict__ q;    // [A][4] packed int8 ideal bond vector,
                                    // cation frame
  const double *__restrict__ pair;  // [S][S][kMfPair]
  int S;
  double lx, ly, lz;

  __device__ __forceinline__ static void scale(const double *__restrict__ P,
                                               double lb, R *__restrict__ v) {
    R f[15];
#pragma unroll
    for (int e = 0; e < 15; ++e) {
      if constexpr (sizeof(R) == 8) f[e] = exp(P[kMfEta + e] * lb);
      else f[e] = __expf((float)(P[kMfEta + e] * lb));
    }
#pragma unroll
    for (int k = 0; k < 21; ++k) v[k] = R(P[k]) * f[eta_index(k)];
  }

  // the record of a bond from its two atoms and its ideal vector
  __device__ __forceinline__ void make(const double4 &gc, const double4 &ga, int qp,
                                       R (&rec)[24]) const {
    const double qx = (double)(int8_t)(qp & 0xff);
    const double qy = (double)(int8_t)((qp >> 8) & 0xff);
    const double qz = (double)(int8_t)((qp >> 16) & 0xff);
    // anion -> cation (getRelativePosVec, geo_struct.c:2278-2294, with the
    // cation-row sign of h_cvectr_mult.c:1073-1090)
    const double nx = -(lx * (0.25 * qx) + ga.x - gc.x);
    const double ny = -(ly * (0.25 * qy) + ga.y - gc.y);
    const double nz = -(lz * (0.25 * qz) + ga.z - gc.z);
    const double den = sqrt(nx * nx + ny * ny + nz * nz);
    R v[21];
    const int p = (int)gc.w * S + (int)ga.w;
    // the common case, one species pair across the wavefront, reads the
    // pair constants through the scalar cache
    const int pu = __builtin_amdgcn_readfirstlane(p);
    if (__all(p == pu)) {
      const double *P = pair + pu * kMfPair;
      scale(P, log((0.25 * kSqrt3Ref * P[kMfA0]) / den), v);
    } else {
      const double *P = pair + p * kMfPair;
      scale(P, log((0.25 * kSqrt3Ref * P[kMfA0]) / den), v);
    }
    if constexpr (sizeof(R) == 8) {
      sk_record(nx / den, ny / den, nz / den, v, rec);
    } else {
      double w[21], k[24];
#pragma unroll
      for (int i = 0; i < 21; ++i) w[i] = v[i];
      sk_record(nx / den, ny / den, nz / den, w, k);
      sk_round(k, rec);
    }
  }


  struct Index {
    int2 e;
  };
  struct Data {
    double4 gc, ga;
    int q;
  };
  __device__ __forceinline__ void index(int blk, Index &i) const {
    i.e = make_int2(-1, -1);
    if (threadIdx.x < kSkBonds) i.e = ends[blk * kSkBondPad + (int)threadIdx.x];
  }
  __device__ __forceinline__ void load(const Index &i, Data &d) const {
    d.q = -1;
    if (i.e.x >= 0) {
      d.gc = geo[i.e.x >> 2];
      d.ga = geo[i.e.y];
      d.q = q[i.e.x] & 0xffffff;
    }
  }
  __device__ __forceinline__ void stage(const Data &d, uint4 *rec) const {
    if (d.q >= 0) {
      R k[24];
      make(d.gc, d.ga, d.q, k);
      const uint4 *r = reinterpret_cast<const uint4 *>(k);
#pragma unroll
      for (int i = 0; i < SkRec<R>::kChunks; ++i)
        rec[threadIdx.x * SkRec<R>::kStride + i] = r[i];
    }
  }
};

template <typename R>
inline MfSrc<R> mf_src(const nh_context *c) {
  return MfSrc<R>{c->mf_ends, c->mf_geo, c->mf_q, c->mf_pair, c->n_species,
                  c->lattice[0], c->lattice[1], c->lattice[2]};
}

// ---- one block ------------------------------------------------------------------

// What a thread is: quad Q of lanes, its atom's slot in the block; lane c of
// the quad: chunks c, c + 4, ... when the quad moves an item, component re /
// im (comp) of spin h (20 bands) or of bond half h (10 bands) when it computes.
struct SkThread {
  int Q, c, comp, h;
  __device__ __forceinline__ SkThread() {
    Q = threadIdx.x >> 2;
    c = threadIdx.x & 3;
    comp = c & 1;
    h = c >> 1;
  }
};

// The thread's part of a block's tables: the two atoms whose entries its quad
// stages (its own and one of the halo), the neighbours' and records' places,
// the records.
template <typename SRC>
struct SkIndex {
  int own, halo;
  uint2 local;
  typename SRC::Index rec;
  __device__ __forceinline__ void read(const SkTable &tab, const SRC &src, int blk, int Q) {
    own = tab.own[blk * kSkOwn + Q];
    halo = tab.halo[blk * kSkHalo + Q];
    local = tab.local[blk * kSkOwn + Q];
    src.index(blk, rec);
  }
};

// whether some own atom of the wavefront lacks a neighbour (a byte of all ones)
__device__ __forceinline__ bool sk_surface(int own, uint2 local) {
  const unsigned z = ~local.x;
  return __any(own >= 0 && ((z - 0x01010101u) & ~z & 0x80808080u) != 0);
}

// The entries of an atom, chunks c, c + 4, ... by lane c
template <int NSP, typename XT>
__device__ __forceinline__ void sk_load_x(int atom, int c, const XT *__restrict__ x,
                                          uint4 (&X)[SkX<NSP, XT>::kLoads]) {
  const uint4 *p = reinterpret_cast<const uint4 *>(x) + (int64_t)atom * SkX<NSP, XT>::kChunks;
#pragma unroll
  for (int i = 0; i < SkX<NSP, XT>::kLoads; ++i) {
    X[i] = make_uint4(0, 0, 0, 0);
    if (atom >= 0 && 4 * i + c < SkX<NSP, XT>::kChunks) X[i] = p[4 * i + c];
  }
}
template <int NSP, typename XT>
__device__ __forceinline__ void sk_stage_x(uint4 *place, int c,
                                           const uint4 (&X)[SkX<NSP, XT>::kLoads]) {
#pragma unroll
  for (int i = 0; i < SkX<NSP, XT>::kLoads; ++i)
    if (4 * i + c < SkX<NSP, XT>::kChunks) place[SkX<NSP, XT>::at(4 * i + c)] = X[i];
}
// r_k from the chunks of u_{k-1} and r_{k-1}
template <typename XT, int K>
__device__ __forceinline__ void sk_defer(uint4 (&X)[K], const uint4 (&P)[K], LzCoef<XT> a) {
#pragma unroll
  for (int i = 0; i < K; ++i) X[i] = lz_defer_chunk<XT>(X[i], P[i], a);
}

// The thread's component (of its spin) of the item at `place`
template <int NSP, typename R, typename XT>
__device__ __forceinline__ void sk_read_x(const uint4 *place, const SkThread &t, R (&x)[10]) {
  using E = typename std::conditional<sizeof(XT) == 16, double, float>::type;
  constexpr int kPer = 16 / (int)sizeof(XT);  // entries of a chunk
  const E *p = reinterpret_cast<const E *>(place) + (NSP == 2 ? 2 * kPer * t.h : 0) + t.comp;
#pragma unroll
  for (int o = 0; o < 10; ++o) x[o] = R(p[2 * (NSP * kPer * (o / kPer) + o % kPer)]);
}

// acc = the thread's component of sum_n T_n x_n from the staged block; R
// inside a bond, FP64 over the bonds.  20 bands: the lane applies the atom's
// four bonds; 10 bands: the two lanes of a component two each.
template <int NSP, typename R, bool CATION, typename XT>
__device__ __forceinline__ void sk_bonds(const SkThread &t, uint2 local,
                                         const SkLds<NSP, R, XT> &L, double (&acc)[10]) {
#pragma unroll
  for (int o = 0; o < 10; ++o) acc[o] = 0.0;
#pragma unroll
  for (int n = 0; n < 2 * NSP; ++n) {
    const int sh = NSP == 2 ? 8 * n : 8 * n + 16 * t.h;
    const int lx = (local.x >> sh) & 0xff, lb = (local.y >> sh) & 0xff;
    if (lx != 0xff) {
      R k[24], x[10];
#pragma unroll
      for (int i = 0; i < SkRec<R>::kChunks; ++i)
        *reinterpret_cast<uint4 *>(&k[i * (16 / (int)sizeof(R))]) =
            L.rec[lb * SkRec<R>::kStride + i];
      sk_read_x<NSP, R, XT>(L.x + lx * SkX<NSP, XT>::kStride, t, x);
      if constexpr (sizeof(R) == 8) {
        sk_apply<CATION, double>(k, x, acc);
      } else {
        float y[10];
#pragma unroll
        for (int o = 0; o < 10; ++o) y[o] = 0.0f;
        sk_apply<CATION, float>(k, x, y);
#pragma unroll
        for (int o = 0; o < 10; ++o) acc[o] += (double)y[o];
      }
    }
  }
  if constexpr (NSP == 1) {
#pragma unroll
    for (int o = 0; o < 10; ++o) acc[o] += dpp_f64<kQuadXor2>(acc[o]);
  }
}

// y += the onsite terms of the thread's component x: diagonal - shift, surface
// s-p couplings (surface: some atom of the wavefront has them), spin-orbit.
template <int NSP>
__device__ __forceinline__ void sk_onsite(const SkThread &t, const double (&x)[10],
                                          const uint4 *place, double shift, bool surface,
                                          double (&y)[10]) {
  const double *os = reinterpret_cast<const double *>(place);
#pragma unroll
  for (int o = 0; o < 10; ++o) y[o] = __builtin_fma(os[o] - shift, x[o], y[o]);
  if (surface) {
    // couplings (1,2) (1,3) (1,4) (2,3) (2,4) (3,4)
    const double s0 = os[10], s1 = os[11], s2 = os[12], s3 = os[13], s4 = os[14], s5 = os[15];
    y[1] = __builtin_fma(s2, x[4], __builtin_fma(s1, x[3], __builtin_fma(s0, x[2], y[1])));
    y[2] = __builtin_fma(s4, x[4], __builtin_fma(s3, x[3], __builtin_fma(s0, x[1], y[2])));
    y[3] = __builtin_fma(s5, x[4], __builtin_fma(s3, x[2], __builtin_fma(s1, x[1], y[3])));
    y[4] = __builtin_fma(s5, x[3], __builtin_fma(s4, x[2], __builtin_fma(s2, x[1], y[4])));
  }
  if constexpr (NSP == 2) {
    // lambda L.S on the p orbitals; lanes 0..3: up re, up im, down re, down im
    const double lam = os[16];
    const double a1 = t.comp != t.h ? -lam : lam;  // + - - +
    const double a2 = t.h ? -lam : lam;            // + + - -
    const double a3 = t.comp ? -lam : lam;         // + - + -
    const double x2_1 = dpp_f64<kQuadXor1>(x[2]), x3_1 = dpp_f64<kQuadXor1>(x[3]);
    const double x4_2 = dpp_f64<kQuadXor2>(x[4]), x2_2 = dpp_f64<kQuadXor2>(x[2]);
    const double x4_3 = dpp_f64<kQuadXor3>(x[4]), x3_3 = dpp_f64<kQuadXor3>(x[3]);
    y[2] = __builtin_fma(a2, x4_2, __builtin_fma(a1, x3_1, y[2]));
    y[3] = __builtin_fma(a3, x4_3, __builtin_fma(-a1, x2_1, y[3]));
    y[4] = __builtin_fma(-a3, x3_3, __builtin_fma(-a2, x2_2, y[4]));
  }
}

// The rest of a product once its bonds are summed: acc += the onsite terms
// (own entries from LDS, onsite record os in the quad's chunks).  The barrier:
// every wavefront has read the staged block; from then on each quad works on
// its own two places only, of which the halo one is free for reuse.
template <int NSP, typename R, typename XT>
__device__ __forceinline__ void sk_finish(const SkThread &t, SkLds<NSP, R, XT> &L,
                                          const uint4 (&os)[3], double shift, bool surface,
                                          double (&acc)[10]) {
  const uint4 *own = L.x + t.Q * SkX<NSP, XT>::kStride;
  uint4 *halo = L.x + (kSkOwn + t.Q) * SkX<NSP, XT>::kStride;
  double xo[10];
  sk_read_x<NSP, double, XT>(own, t, xo);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (4 * i + t.c < kOsChunks) halo[4 * i + t.c] = os[i];
  wave_sync();
  sk_onsite<NSP>(t, xo, halo, shift, surface, acc);
  wave_sync();
}
// components -> entries (FP64) at `place`, from entry `first` on
__device__ __forceinline__ void sk_entries(uint4 *place, int comp, int first,
                                           const double (&y)[10]) {
  double *p = reinterpret_cast<double *>(place + first) + comp;
#pragma unroll
  for (int o = 0; o < 10; ++o) p[2 * o] = y[o];
}
// the quad's chunks of the atom's onsite record
__device__ __forceinline__ void sk_load_onsite(int atom, int c, const double *__restrict__ onsite,
                                               uint4 (&os)[3]) {
  const uint4 *p = reinterpret_cast<const uint4 *>(onsite) + (int64_t)atom * kOsChunks;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    os[i] = make_uint4(0, 0, 0, 0);
    if (atom >= 0 && 4 * i + c < kOsChunks) os[i] = p[4 * i + c];
  }
}

}  // namespace nh
