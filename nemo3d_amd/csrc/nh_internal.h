// Internal state of libnemohip (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>
#include <utility>
#include <mutex>
#include <vector>

#include "../../include/nemohip.h"

namespace nh {

void set_error(const char *fmt, ...);

#define NH_HIP(call)                                                       \
  do {                                                                     \
    const hipError_t nh_hip_status_ = (call);                              \
    if (nh_hip_status_ != hipSuccess) {                                    \
      ::nh::set_error("%s:%d %s: %s", __FILE__, __LINE__, #call,          \
                      hipGetErrorString(nh_hip_status_));                  \
      return NH_ERR_HIP;                                                   \
    }                                                                      \
  } while (0)

#define NH_CHECK(cond, code, ...)                                          \
  do {                                                                     \
    if (!(cond)) {                                                         \
      ::nh::set_error(__VA_ARGS__);                                        \
      return code;                                                         \
    }                                                                      \
  } while (0)

// (the local's name must not collide with any identifier used in `expr`,
// e.g. a member s_, which it would shadow inside its own initialiser)
#define NH_TRY(expr)                                                       \
  do {                                                                     \
    const nh_status nh_try_status_ = (expr);                               \
    if (nh_try_status_ != NH_OK) return nh_try_status_;                    \
  } while (0)

// Onsite record per atom: 10 diagonal energies, 6 surface s-p couplings,
// spin-orbit lambda (17 doubles, padded to 18 for 16-byte alignment).
constexpr int kOnsiteStride = 18;
// Per-bond SK record: l, m, n and 21 combinations of the scaled integrals
// (sk_record, nh_sk_apply.h).
constexpr int kSkStride = 24;
// Matrix-free layout, per (cation species, anion species) pair: the 21
// unscaled two-centre integrals (parameters 10..30), the 15 strain
// exponents (strain parameters 0..14) and the unstrained lattice constant.
constexpr int kMfPair = 40;
constexpr int kMfEta = 21, kMfA0 = 36;

// LDS accesses of one wavefront execute in order; this keeps the compiler
// from moving them across (lanes read what other lanes of the wavefront
// wrote).  No instruction is emitted.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace nh

struct nh_context {
  int device = 0;
  int nb = 0;        // 10 or 20
  int n_atoms = 0;
  int n_species = 0;
  int n_cations = 0;
  int64_t n = 0;     // n_atoms * nb
  double lattice[3] = {0, 0, 0};
  int passivate = 0;
  double db_shift = 0;
  hipStream_t stream = nullptr;
  hipStream_t side = nullptr;  // convergence checks beside the steps (on first use)

  // model (device)
  double *parmat = nullptr;     // [S][S][35]
  double *strnmat = nullptr;    // [S][S][33]
  int32_t *species = nullptr;   // [A]
  int32_t *is_cation = nullptr; // [A]
  int32_t *nbr = nullptr;       // [A][4]
  int32_t *bond_q = nullptr;    // [A][4][3]
  double *disp = nullptr;       // [A][3]
  double *phi = nullptr;        // [A] or null
  int32_t *cations = nullptr;   // [Nc] atom index of each cation
  int32_t *bond_of = nullptr;   // [A][4] cation-owned bond id (ci*4+slot)
  int32_t *rev_slot = nullptr;  // [A][4] slot of this atom in the nbr's list
  // blocks of atoms of the SK / matrix-free products (SkTable, nh_hv_sk.h)
  int n_blocks = 0;
  int32_t *blk_own = nullptr, *blk_halo = nullptr, *blk_bonds = nullptr;
  uint2 *blk_local = nullptr;

  // settings (nh_context_set)
  int hv_staged = -1;  // NH_SET_HV_STAGED (0: no FP32 Lanczos vectors)
  int ring_steps = 0;  // NH_SET_RING_STEPS (0: by free memory)
  int block_hv = -1;   // NH_SET_BLOCK_HV (-1: by size, hv_columns)
  int lz_vectors = -1; // NH_SET_LZ_VECTORS (-1: default, lz_fp32_vectors)

  // assembled Hamiltonian
  int layout = -1;
  int precision = -1;
  double *onsite = nullptr;     // [A][kOnsiteStride]
  double *blocks64 = nullptr;   // [A][4][100] (NH_LAYOUT_BLOCKS, FP64)
  float *blocks32 = nullptr;    // [A][4][100] (NH_LAYOUT_BLOCKS, FP32)
  double *sk64 = nullptr;       // [Nc*4][kSkStride] (NH_LAYOUT_SK)
  float *sk32 = nullptr;
  double4 *mf_geo = nullptr;    // [A] displacement (nm) x, y, z; species
  int32_t *mf_q = nullptr;      // [A][4] ideal bond vector of the slot seen
                                // from its cation, units a/4, 3 x int8
  double *mf_pair = nullptr;    // [S][S][kMfPair] (cation, anion) constants
  int2 *mf_ends = nullptr;      // [blocks][192] atoms of the blocks' bonds

  // work buffers
  double *red = nullptr;        // reduction partials
  int red_cap = 0;
  double *hred = nullptr;       // pinned host mirror of reductions
  nh_cplx *xbuf = nullptr;      // host-pointer staging
  nh_cplx *ybuf = nullptr;
  int64_t buf_cap = 0;          // complex elements in xbuf/ybuf
  // solver workspace kept across solves: blocks a solver releases stay
  // allocated for the next request (a hipFree of tens of GB can stall for
  // a second or more); freed with the context
  struct PoolBlock {
    void *p;
    size_t bytes;
    bool used;
  };
  std::vector<PoolBlock> pool;
  // blocks of nh_device_alloc that were freed, for its next requests of the
  // same size (device_keep); several threads may allocate on one context
  std::vector<PoolBlock> kept;
  std::mutex kept_mu;
};

namespace nh {
// Layouts applied bond by bond from records (nh_hv_sk.h): the stored SK records
// and the matrix-free one.
inline bool sk_like(const nh_context *c) {
  return c->layout == NH_LAYOUT_SK || c->layout == NH_LAYOUT_MATRIX_FREE;
}
// Lanczos vectors stored in FP32 (FP32 SK or matrix-free products).  Default on
// (786,520-atom dot, mixed solve: 3.87 s and 7,976 FP32 steps, 5.88 s and 8,001
// with FP64 vectors, to the same eigenvalues)
inline bool lz_fp32_vectors(const nh_context *c) {
  return sk_like(c) && c->precision == NH_PREC_FP32 && c->hv_staged != 0 &&
         c->lz_vectors != 0;
}
}  // namespace nh


namespace nh {
// Sampled kernel timing with HIP events on the launching stream: begin()/
// end() around a launch; collect() after a synchronisation folds the
// elapsed times into the mean.
struct KernelTimer {
  std::vector<std::pair<hipEvent_t, hipEvent_t>> ev;
  double sum_ms = 0.0;
  int count = 0;
  hipEvent_t pending = nullptr;
  ~KernelTimer() { release(); }
  void release() {
    for (auto &e : ev) {
      (void)hipEventDestroy(e.first);
      (void)hipEventDestroy(e.second);
    }
    ev.clear();
    if (pending) (void)hipEventDestroy(pending);
    pending = nullptr;
  }
  nh_status begin(hipStream_t s) {
    NH_HIP(hipEventCreate(&pending));
    NH_HIP(hipEventRecord(pending, s));
    return NH_OK;
  }
  nh_status end(hipStream_t s) {
    hipEvent_t e;
    NH_HIP(hipEventCreate(&e));
    NH_HIP(hipEventRecord(e, s));
    ev.push_back({pending, e});
    pending = nullptr;
    return NH_OK;
  }
  nh_status collect(hipStream_t s) {
    NH_HIP(hipStreamSynchronize(s));
    for (auto &e : ev) {
      float ms = 0.f;
      NH_HIP(hipEventElapsedTime(&ms, e.first, e.second));
      sum_ms += ms;
      ++count;
    }
    release();
    return NH_OK;
  }
  double mean_ms() const { return count ? sum_ms / count : 0.0; }
};

// Progress lines on stderr for long solves (NEMOHIP_PROGRESS=1): at most
// one every 15 s, so that a caller's log shows the solve is alive.
struct Progress {
  bool on = false;
  double last = 0.0;
  Progress();
  void tick(const char *what, int iter, int extra);
};

// kernels / launchers (nh_assemble.hip, nh_hv.hip, nh_vector.hip)
nh_status assemble(nh_context *c, int layout, int precision);
nh_status select_precision(nh_context *c, int precision);
nh_status launch_hv(nh_context *c, double shift, const nh_cplx *x,
                    nh_cplx *y, int ncol, int64_t ld);
nh_status reduce_dot(nh_context *c, int64_t n, const nh_cplx *x,
                     const nh_cplx *y, double *out2 /* host re,im */);
nh_status reduce_nrm2sq(nh_context *c, int64_t n, const nh_cplx *x,
                        double *out);
// nh_dot_noalloc (nh_vector.hip): file-scope scratch per device, its address
// resolved once per device at context creation
nh_status init_noalloc_scratch(int device);
nh_status reduce_dot_noalloc(nh_context *c, int64_t n, const nh_cplx *x,
                             const nh_cplx *y, double *out2);
nh_status launch_axpby(nh_context *c, int64_t n, nh_cplx a, const nh_cplx *x,
                       nh_cplx b, nh_cplx *y);
nh_status ensure_reduce(nh_context *c, int blocks);
// the block tables of the SK and matrix-free products (cations, bond_of,
// blk_*), made by the first build that needs them: the relaxation, the stored
// blocks and the learned start do without
nh_status ensure_blocks(nh_context *c);
// hipMalloc that, when the device is full, frees the idle workspace blocks
// of every context on the device and tries once more (NH_ERR_NOMEM after
// that); every device allocation of the library goes through it
nh_status device_malloc(nh_context *c, void **p, size_t bytes);
template <typename T>
inline nh_status device_alloc(nh_context *c, T **p, size_t count) {
  return device_malloc(c, reinterpret_cast<void **>(p), count * sizeof(T));
}
// The reference's random starts on the host (nh_random.hip): glibc's
// rand() after srand(seed), LAPACK's dlaruv / zlarnv(idist = 1), and the
// Lanczos Random start (rand() / RAND_MAX, 0) built from them.
class GlibcRand {
 public:
  explicit GlibcRand(uint32_t seed);
  int32_t next() { return (int32_t)(step() >> 1); }

 private:
  uint32_t step();
  uint32_t r_[34];
  int k_ = 0;
};
void dlaruv(int32_t iseed[4], int n, double *x);
void zlarnv_uniform(int32_t iseed[4], int64_t n, nh_cplx *x);
void rand_start(uint32_t seed, int64_t n, nh_cplx *x);
// device memory from the context's workspace pool: the smallest free block
// of at least `bytes` and at most twice that, else a new allocation (after
// returning the free blocks to the device if it is full); pool_release
// hands a block back (work queued on the context's stream that uses it may
// still be running: the next user is ordered after it on that stream)
nh_status pool_alloc(nh_context *c, void **p, size_t bytes);
void pool_release(nh_context *c, void *p);
// bytes in the idle blocks of every context on c's device
size_t pool_free_bytes(const nh_context *c);
nh_status ensure_buffers(nh_context *c, int64_t elems);
}  // namespace nh
