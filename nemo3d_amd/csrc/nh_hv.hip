// Sparse H·v and block H·V for the stored-block layout (row computation
// in nh_hv_row.h).
#include <algorithm>

#include "nh_hv_row.h"
#include "nh_hv_sk.h"

namespace nh {
namespace {

// SK-compressed and matrix-free layouts (see nh_hv_sk.h; SRC = SkSrc or
// MfSrc): each workgroup takes block after block.  COLS: `per` columns of a
// block one after another (its records, tables and onsite terms read once for
// them; Hmatmult_spds_col_stored, Hmult_stored.c:2359-2474, re-reads H for
// every column), the next column's entries requested while the current one is
// computed; a group of columns per grid row.
template <bool COLS, int NSP, typename R, typename SRC>
__global__ __launch_bounds__(kSkThreads, 2) void k_hv_sk(
    SkTable tab, const double *__restrict__ onsite, const SRC src, double shift,
    const double2 *__restrict__ X, double2 *__restrict__ Y, int64_t ld, int ncol, int per) {
  __shared__ SkLds<NSP, R, double2> L;
  using S = SkX<NSP, double2>;
  const SkThread t;
  SkWalk w(tab);
  if (w.b >= w.end) return;
  const int c0 = COLS ? blockIdx.y * per : blockIdx.y, nc = COLS ? min(per, ncol - c0) : 1;
  const double2 *x0 = X + (int64_t)c0 * ld;
  double2 *y0 = Y + (int64_t)c0 * ld;
  // the role is uniform across the wavefront; read as a scalar, the role
  // branches below are scalar branches (one per wave)
  const bool cat = __builtin_amdgcn_readfirstlane(t.Q) < kSkOwn / 2;
  uint4 *own = L.x + t.Q * S::kStride, *halo = L.x + (kSkOwn + t.Q) * S::kStride;
  SkIndex<SRC> ix;
  ix.read(tab, src, w.b, t.Q);
  while (w.b < w.end) {
    typename SRC::Data rec;
    uint4 xo[S::kLoads], xh[S::kLoads], os[3];
    const int atom = ix.own, hatom = ix.halo;
    sk_load_x<NSP>(atom, t.c, x0, xo);
    sk_load_x<NSP>(hatom, t.c, x0, xh);
    src.load(ix.rec, rec);
    sk_load_onsite(atom, t.c, onsite, os);
    const uint2 local = ix.local;
    const bool surface = sk_surface(atom, local);
    w.b += w.step;
    if (w.b < w.end) ix.read(tab, src, w.b, t.Q);
    src.stage(rec, L.rec);
    for (int col = 0; col < nc; ++col) {
      sk_stage_x<NSP, double2>(own, t.c, xo);
      sk_stage_x<NSP, double2>(halo, t.c, xh);
      __syncthreads();
      if (COLS && col + 1 < nc) {
        sk_load_x<NSP>(atom, t.c, x0 + (int64_t)(col + 1) * ld, xo);
        sk_load_x<NSP>(hatom, t.c, x0 + (int64_t)(col + 1) * ld, xh);
      }
      double acc[10];
      if (cat) sk_bonds<NSP, R, true, double2>(t, local, L, acc);
      else sk_bonds<NSP, R, false, double2>(t, local, L, acc);
      sk_finish<NSP, R, double2>(t, L, os, shift, surface, acc);
      if (NSP == 2 || t.h == 0) sk_entries(own, t.comp, NSP == 2 ? 10 * t.h : 0, acc);
      wave_sync();
      if (atom >= 0) {
        uint4 *y = reinterpret_cast<uint4 *>(y0 + (int64_t)col * ld) + (int64_t)atom * S::kChunks;
#pragma unroll
        for (int i = 0; i < S::kLoads; ++i)
          if (4 * i + t.c < S::kChunks) y[4 * i + t.c] = own[4 * i + t.c];
      }
      wave_sync();
    }
  }
}

// A column per grid row, or (COLS) `per`: the blocks are read once for all of
// them and stay in registers (104,976 atoms, 8 columns, FP64: 424 us, a column
// per grid row 720).
template <bool COLS, int NSP, typename TB, typename TA>
__global__ __launch_bounds__(kThreads, COLS ? 2 : 3) void k_hv_blocks(
    int A, const double *__restrict__ onsite, const TB *__restrict__ blocks,
    const int32_t *__restrict__ nbr, double shift,
    const double2 *__restrict__ x, double2 *__restrict__ y, int64_t ld, int ncol, int per) {
  constexpr int NB = NSP * 10;
  __shared__ RowLds<NSP, TB> L[kThreads / 64];
  const int wave = threadIdx.x >> 6;
  const int a0 = (blockIdx.x * (kThreads / 64) + wave) * kRowAtoms;
  if (a0 >= A) return;
  const Rows<NSP, TB> rows(a0, A, blocks, nbr);
  const int64_t c0 = COLS ? blockIdx.y * (int64_t)per : blockIdx.y;
  const int nc = COLS ? min(per, (int)(ncol - c0)) : 1;
  for (int c = 0; c < nc; ++c) {
    double acc_re[NSP], acc_im[NSP];
    double2 xi[NSP];
    rows.template apply<TA>(onsite, shift, x + (c0 + c) * ld, L[wave], acc_re, acc_im, xi);
    if (rows.atom >= 0) {
      double2 *yr = y + (c0 + c) * ld + (int64_t)rows.atom * NB + rows.o;
#pragma unroll
      for (int s = 0; s < NSP; ++s) yr[s * 10] = make_double2(acc_re[s], acc_im[s]);
    }
  }
}

// Columns of a workgroup (mode: NH_SET_BLOCK_HV).  All of them, H read once,
// where the `groups` workgroups of one column fill the chip (`slots` run at a
// time); fewer where they do not: each further column costs a workgroup about
// 3 us, one beside it nothing while the chip has room (SK, FP64, 8 columns:
// 1,000 atoms 39.5 us all / 17.9 one, 11,520 atoms 42.3 / 36.7, 24,576 atoms
// 56 / 58, 108,160 atoms 180 / 220; stored blocks 39 / 20, 56 / 77, 95 / 152,
// 417 / 722).
int hv_columns(int mode, int groups, int slots, int ncol) {
  if (ncol == 1 || mode == 0) return 1;
  if (mode > 0) return ncol;
  const int rows = std::min(ncol, std::max(1, slots / groups));
  return (ncol + rows - 1) / rows;
}

}  // namespace

nh_status launch_hv(nh_context *c, double shift, const nh_cplx *x, nh_cplx *y,
                    int ncol, int64_t ld) {
  NH_CHECK(c->layout == NH_LAYOUT_BLOCKS || sk_like(c), NH_ERR_STATE,
           "H·v: Hamiltonian not built in a supported layout");
  NH_CHECK(ncol >= 1 && ncol <= 65535 && ld >= c->n, NH_ERR_ARG,
           "H·V: bad ncol %d / ld %lld", ncol, (long long)ld);
  // block products: several columns of a workgroup with H read once (SK and
  // matrix-free, 395,136 atoms, 8 columns, FP64: 0.65 ms against 0.83 / 1.06
  // with a column per grid row; stored blocks, 104,976 atoms, 8 columns: 424 us
  // FP64, 331 FP32 against 720 and 416; FP32 matrix instructions, a wavefront
  // per atom and 8 columns: 519)
  const int mode = c->block_hv;
  if (sk_like(c)) {
    const SkTable tab = sk_table_of(c);
    const double2 *xd = reinterpret_cast<const double2 *>(x);
    double2 *yd = reinterpret_cast<double2 *>(y);
    const int per = hv_columns(mode, std::max(1, c->n_blocks), 512, ncol);
    const bool cols = per > 1;
    // one block per workgroup; the matrix-free product of one vector is
    // faster with as many workgroups as run at a time, their next tables read
    // ahead (786,520 atoms, FP64: 0.273 against 0.292 ms; SK 0.243 / 0.232)
    const bool walk = c->layout == NH_LAYOUT_MATRIX_FREE && !cols;
    const dim3 g(walk ? sk_grid(c, 2) : sk_grid(c, 1 << 20), (ncol + per - 1) / per);
#define SKL(NSP, R, SRC)                                                       \
  do {                                                                         \
    if (cols)                                                                  \
      hipLaunchKernelGGL((k_hv_sk<true, NSP, R, decltype(SRC)>), g,            \
                         dim3(kSkThreads), 0, c->stream, tab, c->onsite, SRC,  \
                         shift, xd, yd, ld, ncol, per);                        \
    else                                                                       \
      hipLaunchKernelGGL((k_hv_sk<false, NSP, R, decltype(SRC)>), g,           \
                         dim3(kSkThreads), 0, c->stream, tab, c->onsite, SRC,  \
                         shift, xd, yd, ld, ncol, 1);                          \
  } while (0)
#define SKP(R, SRC)                                                          \
  do {                                                                       \
    if (c->nb == 20) SKL(2, R, SRC);                                         \
    else SKL(1, R, SRC);                                                     \
  } while (0)
    if (c->layout == NH_LAYOUT_MATRIX_FREE) {
      if (c->precision == NH_PREC_FP64) SKP(double, mf_src<double>(c));
      else SKP(float, mf_src<float>(c));
    } else if (c->precision == NH_PREC_FP64) {
      SKP(double, (SkSrc<double>{c->sk64, c->blk_bonds}));
    } else {
      SKP(float, (SkSrc<float>{c->sk32, c->blk_bonds}));
    }
#undef SKP
#undef SKL
    NH_HIP(hipGetLastError());
    return NH_OK;
  }
  const int groups = (c->n_atoms + kAtomsPerBlock - 1) / kAtomsPerBlock;
  const int per = hv_columns(mode, groups, 768, ncol);
  const bool cols = per > 1;
  const dim3 grid(groups, (ncol + per - 1) / per);
  const double2 *xd = reinterpret_cast<const double2 *>(x);
  double2 *yd = reinterpret_cast<double2 *>(y);
#define HVB(NSP, TB, TA, BLK)                                                  \
  do {                                                                       \
    if (cols)                                                                \
      hipLaunchKernelGGL((k_hv_blocks<true, NSP, TB, TA>), grid,             \
                         dim3(kThreads), 0, c->stream, c->n_atoms, c->onsite, \
                         BLK, c->nbr, shift, xd, yd, ld, ncol, per);         \
    else                                                                     \
      hipLaunchKernelGGL((k_hv_blocks<false, NSP, TB, TA>), grid,            \
                         dim3(kThreads), 0, c->stream, c->n_atoms, c->onsite, \
                         BLK, c->nbr, shift, xd, yd, ld, ncol, 1);           \
  } while (0)
  if (c->precision == NH_PREC_FP64) {
    if (c->nb == 20) HVB(2, double, double, c->blocks64);
    else HVB(1, double, double, c->blocks64);
  } else {
    if (c->nb == 20) HVB(2, float, float, c->blocks32);
    else HVB(1, float, float, c->blocks32);
  }
#undef HVB
  NH_HIP(hipGetLastError());
  return NH_OK;
}

}  // namespace nh
