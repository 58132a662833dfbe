// Rows of the stored-block H·v, shared by the plain operator kernel and the
// fused Lanczos kernel (the library is built without relocatable device code,
// so every kernel's translation unit includes this).
//
// Row-owner mapping: 10 lanes per atom, six atoms a wavefront; lane o of an
// atom owns spatial orbital o of both spins, so the spin-shared 10x10 real
// neighbour blocks (HamZincBlende::Hu, spin-diagonal and spin-independent) are
// read once per row and applied to both spin components (Hv_stored_20_Hzb,
// Hmult_stored.c:176-607, which applies Hu to rows i and i+10).
//
// The blocks are the traffic (3,200 B an atom in FP64).  Each wavefront loads
// the six 800-byte blocks of a slot as consecutive 16-byte chunks, all four
// slots in flight together, and hands them to the rows through its part of
// LDS, as it does with the neighbours' entries.  A lane that loads its own
// 80-byte row touches every cache line of the wavefront's 5 KB with each of
// its five loads; with the lines of all wavefronts larger than the L1 that
// fetched them several times from L2: 104,976 atoms, FP64, 146 -> 103 us (419
// MB, 4.1 TB/s; a copy moves 4.7).
//
// FP32 storage: each block product is formed in FP32 (values and the FP32
// image of x) and added to an FP64 row accumulator.
#pragma once

#include "nh_internal.h"

namespace nh {

constexpr int kRowAtoms = 6;  // of a wavefront (60 lanes)
constexpr int kThreads = 256;
constexpr int kAtomsPerBlock = kThreads / 64 * kRowAtoms;

// Surface s-p coupling partner list for lane o in {1,2,3,4}: partner
// orbital and index into the 6 stored couplings (1,2),(1,3),(1,4),(2,3),
// (2,4),(3,4).
__device__ __forceinline__ void sp_partners(int o, int p[3], int k[3]) {
  switch (o) {
    case 1: p[0] = 2; k[0] = 0; p[1] = 3; k[1] = 1; p[2] = 4; k[2] = 2; break;
    case 2: p[0] = 1; k[0] = 0; p[1] = 3; k[1] = 3; p[2] = 4; k[2] = 4; break;
    case 3: p[0] = 1; k[0] = 1; p[1] = 2; k[1] = 3; p[2] = 4; k[2] = 5; break;
    default: p[0] = 1; k[0] = 2; p[1] = 2; k[1] = 4; p[2] = 3; k[2] = 5; break;
  }
}

// Onsite part of row (atom, spin s, orbital o): (diagonal - shift) x,
// dangling-bond s-p couplings and spin-orbit.  Initialises acc.
template <int NSP>
__device__ __forceinline__ void hv_onsite(int atom, int o,
                                          const double *__restrict__ onsite,
                                          double shift,
                                          const double2 *__restrict__ xc,
                                          double acc_re[NSP], double acc_im[NSP],
                                          double2 xi[NSP]) {
  constexpr int NB = NSP * 10;
  const int64_t base = (int64_t)atom * NB;
  const double *os = onsite + (size_t)atom * kOnsiteStride;
  const double d = os[o] - shift;
#pragma unroll
  for (int s = 0; s < NSP; ++s) {
    xi[s] = xc[base + s * 10 + o];
    acc_re[s] = d * xi[s].x;
    acc_im[s] = d * xi[s].y;
  }
  // dangling-bond s-p couplings (zero away from the surface)
  if (o >= 1 && o <= 4) {
    int p[3], k[3];
    sp_partners(o, p, k);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const double h = os[10 + k[q]];
      if (h != 0.0) {
#pragma unroll
        for (int s = 0; s < NSP; ++s) {
          const double2 xp = xc[base + s * 10 + p[q]];
          acc_re[s] += h * xp.x;
          acc_im[s] += h * xp.y;
        }
      }
    }
  }
  // spin-orbit (h3d_diag + mb_ham_spds_so.h; pairs HamZincBlende.c:170-183)
  if (NSP == 2 && o >= 2 && o <= 4) {
    const double lam = os[16];
    const double2 *xa = xc + base;
    // up row o and down row 10+o
    if (o == 2) {        // (2,3) = -i lam, (2,14) = lam ; (12,13) = i lam, (12,4) = -lam
      acc_re[0] += lam * xa[3].y + lam * xa[14].x;
      acc_im[0] += -lam * xa[3].x + lam * xa[14].y;
      acc_re[NSP - 1] += -lam * xa[13].y - lam * xa[4].x;
      acc_im[NSP - 1] += lam * xa[13].x - lam * xa[4].y;
    } else if (o == 3) { // (3,2) = i lam, (3,14) = -i lam ; (13,12) = -i lam, (13,4) = -i lam
      acc_re[0] += -lam * xa[2].y + lam * xa[14].y;
      acc_im[0] += lam * xa[2].x - lam * xa[14].x;
      acc_re[NSP - 1] += lam * xa[12].y + lam * xa[4].y;
      acc_im[NSP - 1] += -lam * xa[12].x - lam * xa[4].x;
    } else {             // (4,12) = -lam, (4,13) = i lam ; (14,2) = lam, (14,3) = i lam
      acc_re[0] += -lam * xa[12].x - lam * xa[13].y;
      acc_im[0] += -lam * xa[12].y + lam * xa[13].x;
      acc_re[NSP - 1] += lam * xa[2].x - lam * xa[3].y;
      acc_im[NSP - 1] += lam * xa[2].y + lam * xa[3].x;
    }
  }
}

// One neighbour block row applied to both spins: acc += B[o][:] x_j.
template <int NSP, typename TB, typename TA>
__device__ __forceinline__ void hv_block(const TB *__restrict__ B,
                                         const double2 *xj, double acc_re[NSP],
                                         double acc_im[NSP]) {
  TA br[NSP], bi[NSP];
#pragma unroll
  for (int s = 0; s < NSP; ++s) br[s] = bi[s] = TA(0);
#pragma unroll
  for (int k = 0; k < 10; ++k) {
    const TA b = TA(B[k]);
#pragma unroll
    for (int s = 0; s < NSP; ++s) {
      const double2 v = xj[s * 10 + k];
      br[s] += b * TA(v.x);
      bi[s] += b * TA(v.y);
    }
  }
#pragma unroll
  for (int s = 0; s < NSP; ++s) {
    acc_re[s] += double(br[s]);
    acc_im[s] += double(bi[s]);
  }
}

// A wavefront's staging: the blocks of one slot and the neighbours' entries
template <int NSP, typename TB>
struct RowLds {
  static constexpr int kSeg = 100 * (int)sizeof(TB) / 16;  // chunks of a block
  static constexpr int kNx = NSP * 10;                     // chunks of an atom's entries
  uint4 b[kRowAtoms * kSeg], x[kRowAtoms * kNx];
};

// What a wavefront holds of its six atoms (the first is a0): its share of the
// 24 blocks' chunks, all requested together, the neighbours of the atoms whose
// entries it stages and of the lane's own atom (-1: no row, the lane only
// takes part in the loads).
template <int NSP, typename TB>
struct Rows {
  using S = RowLds<NSP, TB>;
  static constexpr int kB = (kRowAtoms * S::kSeg + 63) / 64, kX = (kRowAtoms * S::kNx + 63) / 64;
  uint4 bl[4][kB];
  int4 nx[kX], own;
  int atom, o;

  __device__ __forceinline__ Rows(int a0, int A, const TB *__restrict__ blocks,
                                  const int32_t *__restrict__ nbr) {
    const int lane = threadIdx.x & 63, na = min(kRowAtoms, A - a0);
    const int4 *nb4 = reinterpret_cast<const int4 *>(nbr);
    o = lane % 10;
    atom = lane / 10 < na ? a0 + lane / 10 : -1;
#pragma unroll
    for (int i = 0; i < kX; ++i) {
      const int seg = (lane + 64 * i) / S::kNx;
      nx[i] = seg < na ? nb4[a0 + seg] : make_int4(-1, -1, -1, -1);
    }
    own = atom >= 0 ? nb4[atom] : make_int4(-1, -1, -1, -1);
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int i = 0; i < kB; ++i) {
        const int c = lane + 64 * i, seg = c / S::kSeg;
        bl[n][i] = make_uint4(0, 0, 0, 0);
        if (seg < na)
          bl[n][i] = reinterpret_cast<const uint4 *>(
              blocks)[((int64_t)(a0 + seg) * 4 + n) * S::kSeg + c % S::kSeg];
      }
  }

  // acc[s] = ((H - shift I) x) at row (atom, spin s, orbital o)
  template <typename TA>
  __device__ __forceinline__ void apply(const double *__restrict__ onsite, double shift,
                                        const double2 *__restrict__ xc, S &L, double acc_re[NSP],
                                        double acc_im[NSP], double2 xi[NSP]) const {
    const int lane = threadIdx.x & 63, la = lane / 10;
    auto slot = [](const int4 &v, int n) { return n == 0 ? v.x : n == 1 ? v.y : n == 2 ? v.z : v.w; };
    uint4 xl[4][kX];
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int i = 0; i < kX; ++i) {
        const int j = slot(nx[i], n);
        xl[n][i] = make_uint4(0, 0, 0, 0);
        if (j >= 0)
          xl[n][i] =
              reinterpret_cast<const uint4 *>(xc)[(int64_t)j * S::kNx + (lane + 64 * i) % S::kNx];
      }
    if (atom >= 0) hv_onsite<NSP>(atom, o, onsite, shift, xc, acc_re, acc_im, xi);
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      wave_sync();
#pragma unroll
      for (int i = 0; i < kB; ++i)
        if (lane + 64 * i < kRowAtoms * S::kSeg) L.b[lane + 64 * i] = bl[n][i];
#pragma unroll
      for (int i = 0; i < kX; ++i)
        if (lane + 64 * i < kRowAtoms * S::kNx) L.x[lane + 64 * i] = xl[n][i];
      wave_sync();
      if (slot(own, n) >= 0)
        hv_block<NSP, TB, TA>(reinterpret_cast<const TB *>(L.b + la * S::kSeg) + o * 10,
                              reinterpret_cast<const double2 *>(L.x + la * S::kNx), acc_re,
                              acc_im);
    }
  }
};

}  // namespace nh
