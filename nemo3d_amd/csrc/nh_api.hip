// C-ABI entry points of libnemohip (declared in include/nemohip.h).
#include <algorithm>
#include <chrono>
#include <climits>
#include <cstdarg>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <vector>

#include "nh_internal.h"

namespace nh {

static thread_local char g_err[1024] = "";

// Every live context, so that an allocation that fails on a device can take
// back the idle workspace blocks of all contexts on that device, and ring
// sizing can count them as available.
static std::mutex g_ctx_mu;
static std::vector<nh_context *> g_ctxs;

Progress::Progress() {
  const char *e = std::getenv("NEMOHIP_PROGRESS");
  on = e && e[0] == '1';
  last = std::chrono::duration<double>(
             std::chrono::steady_clock::now().time_since_epoch()).count();
}

void Progress::tick(const char *what, int iter, int extra) {
  if (!on) return;
  const double now = std::chrono::duration<double>(
                         std::chrono::steady_clock::now().time_since_epoch()).count();
  if (now - last < 15.0) return;
  last = now;
  std::fprintf(stderr, "# %s: iteration %d (%d)\n", what, iter, extra);
  std::fflush(stderr);
}

void set_error(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

// Frees the idle workspace blocks of one context (after its queued work).
static nh_status pool_trim(nh_context *c) {
  NH_HIP(hipStreamSynchronize(c->stream));
  std::vector<nh_context::PoolBlock> keep;
  for (auto &b : c->pool) {
    if (b.used) keep.push_back(b);
    else NH_HIP(hipFree(b.p));
  }
  c->pool.swap(keep);
  std::lock_guard<std::mutex> g(c->kept_mu);
  for (auto &b : c->kept) NH_HIP(hipFree(b.p));
  c->kept.clear();
  return NH_OK;
}

// Blocks of nh_device_alloc freed by the caller stay with the context, at
// most kKeepBlocks of them and, over all contexts, one part in kKeepShare of
// the device's memory, and serve its next requests of the same size.  A program that asks for its vectors
// anew on every call otherwise runs at the speed at which the driver clears
// freed memory: products of 2 GB a call, each freed when the next one is
// there, took 55 ms a call once the device had been gone through once
// (37 GB/s), the call itself 3.5 ms.
constexpr int kKeepBlocks = 8;
constexpr size_t kKeepShare = 32;

// true: *p is a kept block of exactly `bytes`
static bool device_take(nh_context *c, void **p, size_t bytes) {
  std::lock_guard<std::mutex> g(c->kept_mu);
  for (size_t i = 0; i < c->kept.size(); ++i)
    if (c->kept[i].bytes == bytes) {
      *p = c->kept[i].p;
      c->kept.erase(c->kept.begin() + i);
      return true;
    }
  return false;
}
// keep p, or else free it (p that is not the start of a device allocation:
// hipFree's error)
static nh_status device_keep(nh_context *c, void *p) {
  hipDeviceptr_t base = nullptr;
  size_t bytes = 0, fr = 0, total = 0;
  hipPointerAttribute_t at{};
  const bool ours = hipPointerGetAttributes(&at, p) == hipSuccess &&
                    at.type == hipMemoryTypeDevice && at.device == c->device &&
                    hipMemGetAddressRange(&base, &bytes, p) == hipSuccess && base == p &&
                    hipMemGetInfo(&fr, &total) == hipSuccess;
  (void)hipGetLastError();
  if (!ours || bytes > total / kKeepShare) {
    NH_HIP(hipFree(p));
    return NH_OK;
  }
  // as hipFree does: whatever stream used the memory is done with it
  NH_HIP(hipDeviceSynchronize());
  std::lock_guard<std::mutex> all(g_ctx_mu);
  size_t sum = bytes;  // with the other contexts' blocks
  for (nh_context *o : g_ctxs) {
    if (o->device != c->device) continue;
    std::lock_guard<std::mutex> k(o->kept_mu);
    for (const auto &b : o->kept) {
      NH_CHECK(b.p != p, NH_ERR_ARG, "nh_device_free: freed twice");
      sum += b.bytes;
    }
  }
  std::lock_guard<std::mutex> g(c->kept_mu);
  c->kept.push_back({p, bytes, false});
  while (!c->kept.empty() &&
         (sum > total / kKeepShare || c->kept.size() > (size_t)kKeepBlocks)) {
    // the oldest one goes
    sum -= c->kept.front().bytes;
    NH_HIP(hipFree(c->kept.front().p));
    c->kept.erase(c->kept.begin());
  }
  return NH_OK;
}

nh_status device_malloc(nh_context *c, void **p, size_t bytes) {
  bytes = bytes > 0 ? bytes : 16;
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) {
    // give the idle workspace of every context on this device back and
    // try once more
    (void)hipGetLastError();
    std::vector<nh_context *> same;
    {
      std::lock_guard<std::mutex> g(g_ctx_mu);
      for (nh_context *o : g_ctxs)
        if (o->device == c->device) same.push_back(o);
    }
    for (nh_context *o : same) NH_TRY(pool_trim(o));
    e = hipMalloc(p, bytes);
  }
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
    set_error("hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
    return NH_ERR_NOMEM;
  }
  return NH_OK;
}

nh_status pool_alloc(nh_context *c, void **p, size_t bytes) {
  bytes = bytes > 0 ? (bytes + 255) / 256 * 256 : 256;
  int best = -1;
  for (int i = 0; i < (int)c->pool.size(); ++i) {
    const auto &b = c->pool[i];
    if (!b.used && b.bytes >= bytes && b.bytes <= 2 * bytes &&
        (best < 0 || b.bytes < c->pool[best].bytes))
      best = i;
  }
  if (best >= 0) {
    c->pool[best].used = true;
    *p = c->pool[best].p;
    return NH_OK;
  }
  NH_TRY(device_malloc(c, p, bytes));
  c->pool.push_back({*p, bytes, true});
  return NH_OK;
}

void pool_release(nh_context *c, void *p) {
  for (auto &b : c->pool)
    if (b.p == p) {
      b.used = false;
      return;
    }
}

size_t pool_free_bytes(const nh_context *c) {
  std::lock_guard<std::mutex> g(g_ctx_mu);
  size_t s = 0;
  for (nh_context *o : g_ctxs)
    if (o->device == c->device) {
      for (const auto &b : o->pool)
        if (!b.used) s += b.bytes;
      std::lock_guard<std::mutex> k(o->kept_mu);
      for (const auto &b : o->kept) s += b.bytes;
    }
  return s;
}

nh_status ensure_buffers(nh_context *c, int64_t elems) {
  if (elems <= c->buf_cap) return NH_OK;
  NH_HIP(hipStreamSynchronize(c->stream));
  (void)hipFree(c->xbuf);
  (void)hipFree(c->ybuf);
  c->xbuf = c->ybuf = nullptr;
  c->buf_cap = 0;
  NH_TRY(device_malloc(c, (void **)&c->xbuf, elems * sizeof(nh_cplx)));
  NH_TRY(device_malloc(c, (void **)&c->ybuf, elems * sizeof(nh_cplx)));
  c->buf_cap = elems;
  return NH_OK;
}

template <typename T>
static nh_status upload(nh_context *c, T **dst, const T *src, size_t count) {
  (void)hipFree(*dst);  // of an attempt that failed later on
  *dst = nullptr;
  NH_TRY(device_malloc(c, (void **)dst, count * sizeof(T) + 16));
  NH_HIP(hipMemcpy(*dst, src, count * sizeof(T), hipMemcpyHostToDevice));
  return NH_OK;
}

static void destroy(nh_context *c) {
  if (!c) return;
  {
    std::lock_guard<std::mutex> g(g_ctx_mu);
    g_ctxs.erase(std::remove(g_ctxs.begin(), g_ctxs.end(), c), g_ctxs.end());
  }
  (void)hipSetDevice(c->device);
  void *ptrs[] = {c->parmat, c->strnmat, c->species, c->is_cation, c->nbr,
                  c->bond_q, c->disp, c->phi, c->cations, c->bond_of, c->blk_own,
                  c->blk_local, c->blk_halo, c->blk_bonds, c->mf_geo, c->mf_q,
                  c->mf_pair, c->mf_ends,
                  c->rev_slot, c->onsite, c->blocks64, c->blocks32,
                  c->sk64, c->sk32, c->red, c->xbuf, c->ybuf};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  (void)hipStreamSynchronize(c->stream);
  for (auto &b : c->pool) (void)hipFree(b.p);
  for (auto &b : c->kept) (void)hipFree(b.p);
  if (c->hred) (void)hipHostFree(c->hred);
  if (c->side) (void)hipStreamDestroy(c->side);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

// Blocks of atoms for the SK and matrix-free products (nh_hv_sk.h): the atoms
// are ordered by bricks of 16 cells and inside them by cubes of 2 x 2 x 2
// cells (ideal positions, from the ideal bond vectors by a walk over the bond
// graph), and cut into blocks within the kernels' capacities.  A cube starts a
// new block unless it fits into the open one whole, so the blocks of a
// crystal coincide with its cubes (64 atoms, at most 57 halo atoms and 170
// bonds) and only thin rests of cubes at the surface are put together.
// Inside a block every atom goes, where it can, to a place that is its color
// modulo 8, a linear function of its lattice position: eight atoms in
// consecutive places then have neighbours of eight different colors in any
// direction, and the quads that read them from LDS together meet eight
// different groups of banks.  A bond's color is its cation's.
// Bond numbers are 4 (number of the cation in `cations`) + slot, the cations
// in block order.
struct BlockTables {
  std::vector<int32_t> cations, bond_of;  // bond_of [A][4], -1 for none
  std::vector<int32_t> own, halo, bonds;  // [blocks][64], [64], [192]; -1 pads
  std::vector<uint8_t> local;  // [blocks][64][2][4]: place of x, of the record
  int n = 0;
};

static void cube_order(const nh_model *m, std::vector<int32_t> &order,
                       std::vector<int64_t> &cube, std::vector<uint8_t> &color) {
  const int A = m->n_atoms;
  std::vector<int32_t> pos((size_t)A * 3, 0);
  std::vector<char> seen(A, 0);
  std::vector<int32_t> stack;
  for (int s0 = 0; s0 < A; ++s0) {
    if (seen[s0]) continue;
    seen[s0] = 1;
    stack.push_back(s0);
    while (!stack.empty()) {
      const int i = stack.back();
      stack.pop_back();
      for (int n = 0; n < 4; ++n) {
        const int j = m->nbr[i * 4 + n];
        if (j < 0 || seen[j]) continue;
        seen[j] = 1;
        for (int d = 0; d < 3; ++d)
          pos[(size_t)j * 3 + d] = pos[(size_t)i * 3 + d] + m->bond_q[(i * 4 + n) * 3 + d];
        stack.push_back(j);
      }
    }
  }
  int32_t lo[3] = {INT32_MAX, INT32_MAX, INT32_MAX};
  for (int i = 0; i < A; ++i)
    for (int d = 0; d < 3; ++d) lo[d] = std::min(lo[d], pos[(size_t)i * 3 + d]);
  // units a/4: 8 a cube, 64 a brick (8 cubes): 17 + 3 bits a direction
  std::vector<std::pair<int64_t, int32_t>> key(A);
  for (int i = 0; i < A; ++i) {
    int64_t b = 0, c = 0;
    for (int d = 2; d >= 0; --d) b = b << 17 | (((pos[(size_t)i * 3 + d] - lo[d]) >> 6) & 0x1ffff);
    for (int d = 0; d < 3; ++d) c = c << 3 | (((pos[(size_t)i * 3 + d] - lo[d]) >> 3) & 7);
    key[i] = {b << 9 | c, i};
  }
  std::sort(key.begin(), key.end());
  order.resize(A);
  cube.resize(A);
  color.resize(A);
  for (int i = 0; i < A; ++i) {
    order[i] = key[i].second;
    cube[i] = key[i].first;
    // cations and anions in units of a/2: 4 x 2 of the 4 x 4 x 2 sites of a
    // role in a cube are told apart
    color[i] = (uint8_t)(((pos[(size_t)i * 3] >> 1) + 4 * (pos[(size_t)i * 3 + 1] >> 1)) & 7);
  }
}
// places base .. base + cap of the items, of their color modulo 8 where one is
// free; taken: places given so far
template <typename F>
static void color_places(const std::vector<int32_t> &items, int base, int cap, F color,
                         std::vector<int32_t> &taken, std::vector<int32_t> &place) {
  std::vector<int32_t> rest;
  for (int32_t a : items) {
    int p = color(a);
    while (p < cap && taken[base + p] >= 0) p += 8;
    if (p >= cap) {
      rest.push_back(a);
      continue;
    }
    taken[base + p] = a;
    place[a] = base + p;
  }
  int p = 0;
  for (int32_t a : rest) {
    while (taken[base + p] >= 0) ++p;
    taken[base + p] = a;
    place[a] = base + p;
  }
}

static void build_blocks(const nh_model *m, const std::vector<int32_t> &rev, BlockTables &T) {
  constexpr int kOwn = 64, kHalf = 32, kHalo = 64, kBonds = 176, kBondPad = 192;
  const int A = m->n_atoms;
  std::vector<int32_t> order;
  std::vector<int64_t> cube;
  std::vector<uint8_t> color;
  cube_order(m, order, cube, color);
  for (int i : order)
    if (m->is_cation[i]) T.cations.push_back(i);
  T.bond_of.assign((size_t)A * 4, -1);
  for (size_t ci = 0; ci < T.cations.size(); ++ci) {
    const int i = T.cations[ci];
    for (int n = 0; n < 4; ++n) {
      const int j = m->nbr[i * 4 + n];
      if (j < 0) continue;
      T.bond_of[(size_t)i * 4 + n] = (int32_t)(ci * 4 + n);
      T.bond_of[(size_t)j * 4 + rev[(size_t)i * 4 + n]] = (int32_t)(ci * 4 + n);
    }
  }
  // of the open block: an atom's place (own, or kOwn + halo), a bond's place
  std::vector<int32_t> place(A, -1), bplace(T.cations.size() * 4, -1);
  std::vector<int32_t> halo, bonds;   // members in order of arrival; a halo
  int32_t own[kOwn];                  // atom that became an own one leaves a -1
  int nc = 0, na = 0, nh = 0;
  std::fill(own, own + kOwn, -1);
  auto close = [&]() {
    if (nc + na == 0) return;
    // final places: cations, anions, halo, bonds
    const std::vector<int32_t> oc(own, own + nc), oa(own + kHalf, own + kHalf + na);
    halo.erase(std::remove(halo.begin(), halo.end(), -1), halo.end());
    std::vector<int32_t> at(kOwn + kHalo, -1), rec(kBondPad, -1);
    auto col = [&](int32_t i) { return (int)color[i]; };
    color_places(oc, 0, kHalf, col, at, place);
    color_places(oa, kHalf, kHalf, col, at, place);
    color_places(halo, kOwn, kHalo, col, at, place);
    // bond of slot n of an own cation in place p: 32 n + p; the others after
    // them and in the gaps
    std::vector<int32_t> others;
    for (int32_t q : bonds) {
      const int p = place[T.cations[q >> 2]];
      if (p < kHalf) {
        rec[kHalf * (q & 3) + p] = q;
        bplace[q] = kHalf * (q & 3) + p;
      } else {
        others.push_back(q);
      }
    }
    std::reverse(rec.begin(), rec.begin() + kBonds);  // the free end first
    for (int32_t q : others) bplace[q] = -1;
    color_places(others, 0, kBonds,
                 [&](int32_t q) { return 7 - (int)color[T.cations[q >> 2]]; }, rec, bplace);
    std::reverse(rec.begin(), rec.begin() + kBonds);
    for (int32_t q : others) bplace[q] = kBonds - 1 - bplace[q];
    T.own.insert(T.own.end(), at.begin(), at.begin() + kOwn);
    T.halo.insert(T.halo.end(), at.begin() + kOwn, at.end());
    T.bonds.insert(T.bonds.end(), rec.begin(), rec.end());
    const size_t l0 = T.local.size();
    T.local.resize(l0 + kOwn * 8, 255);
    for (int s = 0; s < kOwn; ++s) {
      if (at[s] < 0) continue;
      for (int n = 0; n < 4; ++n) {
        const int j = m->nbr[(size_t)at[s] * 4 + n];
        if (j < 0) continue;
        T.local[l0 + s * 8 + n] = (uint8_t)place[j];
        T.local[l0 + s * 8 + 4 + n] = (uint8_t)bplace[T.bond_of[(size_t)at[s] * 4 + n]];
      }
    }
    for (int32_t a : at)
      if (a >= 0) place[a] = -1;
    for (int32_t q : bonds) bplace[q] = -1;
    std::fill(own, own + kOwn, -1);
    halo.clear();
    bonds.clear();
    nc = na = nh = 0;
    ++T.n;
  };
  for (size_t k = 0; k < order.size(); ++k) {
    if (k == 0 || cube[k] != cube[k - 1]) {
      int gc = 0, ga = 0;
      for (size_t e = k; e < order.size() && cube[e] == cube[k]; ++e)
        ++(m->is_cation[order[e]] ? gc : ga);
      if (nc + gc > kHalf || na + ga > kHalf) close();
    }
    const int i = order[k];
    const bool cat = m->is_cation[i] != 0;
    int dh = 0, db = 0;
    auto count = [&]() {
      dh = place[i] >= kOwn ? -1 : 0;
      db = 0;
      for (int n = 0; n < 4; ++n) {
        const int j = m->nbr[(size_t)i * 4 + n];
        if (j < 0) continue;
        if (place[j] < 0) ++dh;
        if (bplace[T.bond_of[(size_t)i * 4 + n]] < 0) ++db;
      }
    };
    count();
    if ((cat ? nc : na) == kHalf || nh + dh > kHalo || (int)bonds.size() + db > kBonds) {
      close();
      count();
    }
    if (place[i] >= kOwn) halo[place[i] - kOwn] = -1;
    const int s = cat ? nc++ : kHalf + na++;
    own[s] = i;
    place[i] = s;
    for (int n = 0; n < 4; ++n) {
      const int j = m->nbr[(size_t)i * 4 + n];
      if (j < 0) continue;
      if (place[j] < 0) {
        place[j] = kOwn + (int32_t)halo.size();
        halo.push_back(j);
      }
      const int q = T.bond_of[(size_t)i * 4 + n];
      if (bplace[q] < 0) {
        bplace[q] = (int32_t)bonds.size();
        bonds.push_back(q);
      }
    }
    nh += dh;
  }
  close();
}

nh_status ensure_blocks(nh_context *c) {
  if (c->n_blocks > 0) return NH_OK;
  const size_t A = c->n_atoms;
  std::vector<int32_t> nbr(A * 4), bond_q(A * 12), is_cation(A), rev(A * 4);
  auto get = [](std::vector<int32_t> &v, const int32_t *d) {
    return hipMemcpy(v.data(), d, v.size() * sizeof(int32_t), hipMemcpyDeviceToHost);
  };
  NH_HIP(get(nbr, c->nbr));
  NH_HIP(get(bond_q, c->bond_q));
  NH_HIP(get(is_cation, c->is_cation));
  NH_HIP(get(rev, c->rev_slot));
  nh_model m{};
  m.n_atoms = c->n_atoms;
  m.nbr = nbr.data();
  m.bond_q = bond_q.data();
  m.is_cation = is_cation.data();
  BlockTables b;
  build_blocks(&m, rev, b);
  NH_TRY(upload(c, &c->cations, b.cations.data(), b.cations.size()));
  NH_TRY(upload(c, &c->bond_of, b.bond_of.data(), b.bond_of.size()));
  NH_TRY(upload(c, &c->blk_own, b.own.data(), b.own.size()));
  NH_TRY(upload(c, &c->blk_local, reinterpret_cast<const uint2 *>(b.local.data()),
                b.local.size() / 8));
  NH_TRY(upload(c, &c->blk_halo, b.halo.data(), b.halo.size()));
  NH_TRY(upload(c, &c->blk_bonds, b.bonds.data(), b.bonds.size()));
  c->n_blocks = b.n;
  return NH_OK;
}

static nh_status create(const nh_model *m, int device, nh_context **out) {
  NH_CHECK(m && out, NH_ERR_ARG, "null model or output pointer");
  NH_CHECK(m->nb == 10 || m->nb == 20, NH_ERR_ARG, "nb must be 10 or 20");
  NH_CHECK(m->n_atoms > 0 && m->n_species > 0, NH_ERR_ARG, "empty model");
  NH_CHECK(m->parmat && m->strnmat && m->species && m->is_cation && m->nbr &&
               m->bond_q && m->disp,
           NH_ERR_ARG, "missing model array");
  const int A = m->n_atoms, S = m->n_species;
  NH_CHECK((int64_t)A * m->nb < ((int64_t)1 << 40), NH_ERR_ARG, "too large");
  std::vector<int32_t> rev((size_t)A * 4, -1);
  int n_cations = 0;
  for (int i = 0; i < A; ++i) {
    NH_CHECK(m->species[i] >= 0 && m->species[i] < S, NH_ERR_ARG,
             "species[%d] out of range", i);
    int present = 0;
    for (int n = 0; n < 4; ++n) {
      const int j = m->nbr[i * 4 + n];
      NH_CHECK(j >= -1 && j < A && j != i, NH_ERR_ARG, "nbr[%d][%d] invalid",
               i, n);
      if (j < 0) continue;
      ++present;
      NH_CHECK((m->is_cation[i] != 0) != (m->is_cation[j] != 0), NH_ERR_ARG,
               "bond %d-%d does not join a cation and an anion", i, j);
      int r = -1;
      for (int q = 0; q < 4; ++q)
        if (m->nbr[j * 4 + q] == i) r = q;
      NH_CHECK(r >= 0, NH_ERR_ARG, "neighbour table not symmetric at %d-%d",
               i, j);
      rev[i * 4 + n] = r;
    }
    NH_CHECK(present > 0, NH_ERR_ARG, "atom %d has no neighbours", i);
  }
  for (int i = 0; i < A; ++i) n_cations += m->is_cation[i] != 0;
  NH_CHECK(n_cations > 0, NH_ERR_ARG, "no cation-role atoms");

  NH_HIP(hipSetDevice(device));
  NH_TRY(init_noalloc_scratch(device));
  nh_context *c = new nh_context();
  c->device = device;
  c->nb = m->nb;
  c->n_atoms = A;
  c->n_species = S;
  c->n_cations = n_cations;
  c->n = (int64_t)A * m->nb;
  for (int k = 0; k < 3; ++k) c->lattice[k] = m->lattice[k];
  c->passivate = m->passivate;
  c->db_shift = m->db_shift;
  nh_status st = NH_OK;
#define UP(dst, src, cnt)                              \
  if (st == NH_OK) st = upload(c, &c->dst, src, (size_t)(cnt));
  UP(parmat, m->parmat, (size_t)S * S * 35);
  UP(strnmat, m->strnmat, (size_t)S * S * 33);
  UP(species, m->species, A);
  UP(is_cation, m->is_cation, A);
  UP(nbr, m->nbr, (size_t)A * 4);
  UP(bond_q, m->bond_q, (size_t)A * 12);
  UP(disp, m->disp, (size_t)A * 3);
  if (m->phi) UP(phi, m->phi, A);
  UP(rev_slot, rev.data(), (size_t)A * 4);
#undef UP
  if (st == NH_OK) {
    hipError_t e = hipStreamCreate(&c->stream);
    if (e != hipSuccess) {
      set_error("hipStreamCreate: %s", hipGetErrorString(e));
      st = NH_ERR_HIP;
    }
  }
  if (st != NH_OK) {
    destroy(c);
    return st;
  }
  {
    std::lock_guard<std::mutex> g(g_ctx_mu);
    g_ctxs.push_back(c);
  }
  *out = c;
  return NH_OK;
}

static nh_status check_ctx(nh_context *c) {
  NH_CHECK(c, NH_ERR_ARG, "null context");
  (void)hipGetLastError();  // errors of earlier, already reported calls
  NH_HIP(hipSetDevice(c->device));
  return NH_OK;
}

}  // namespace nh

using namespace nh;

extern "C" {

nh_status nh_context_set(nh_context *ctx, int what, int value) {
  NH_CHECK(ctx, NH_ERR_ARG, "null context");
  switch (what) {
    case NH_SET_HV_STAGED:
      NH_CHECK(value >= -1 && value <= 1, NH_ERR_ARG,
               "NH_SET_HV_STAGED: value %d not in -1..1", value);
      ctx->hv_staged = value;
      return NH_OK;
    case NH_SET_SK_LANES:
      NH_CHECK(value == -1 || value == 4 || value == 8, NH_ERR_ARG,
               "NH_SET_SK_LANES: value %d not -1, 4 or 8", value);
      return NH_OK;
    case NH_SET_LZ_VECTORS:
      NH_CHECK(value >= -1 && value <= 1, NH_ERR_ARG,
               "NH_SET_LZ_VECTORS: value %d not in -1..1", value);
      ctx->lz_vectors = value;
      return NH_OK;
    case NH_SET_SK_ROLES:
      NH_CHECK(value >= -1 && value <= 1, NH_ERR_ARG,
               "NH_SET_SK_ROLES: value %d not in -1..1", value);
      return NH_OK;
    case NH_SET_BLOCK_HV:
      NH_CHECK(value >= -1 && value <= 2, NH_ERR_ARG,
               "NH_SET_BLOCK_HV: value %d not in -1..2", value);
      ctx->block_hv = value;
      return NH_OK;
    case NH_SET_RING_STEPS:
      NH_CHECK(value == 0 || value == 8 || value == 16 || value == 32 || value == 64 ||
                   value == 128,
               NH_ERR_ARG, "NH_SET_RING_STEPS: value %d not 0, 8, 16, 32, 64 or 128",
               value);
      ctx->ring_steps = value;
      return NH_OK;
    default:
      NH_CHECK(false, NH_ERR_ARG, "nh_context_set: unknown setting %d", what);
  }
}

const char *nh_last_error(void) { return g_err; }

nh_status nh_context_create(const nh_model *model, int device,
                            nh_context **out) {
  return create(model, device, out);
}

void nh_context_destroy(nh_context *ctx) { destroy(ctx); }

int64_t nh_context_dim(const nh_context *ctx) { return ctx ? ctx->n : 0; }

nh_status nh_ham_build(nh_context *ctx, int layout, int precision) {
  NH_TRY(check_ctx(ctx));
  return assemble(ctx, layout, precision);
}

nh_status nh_ham_set_precision(nh_context *ctx, int precision) {
  NH_TRY(check_ctx(ctx));
  NH_HIP(hipSetDevice(ctx->device));
  return select_precision(ctx, precision);
}

nh_status nh_hv(nh_context *ctx, double shift, const nh_cplx *x, nh_cplx *y,
                int ptr_kind) {
  return nh_hV(ctx, shift, x, y, 1, ctx ? ctx->n : 0, ptr_kind);
}

nh_status nh_hV(nh_context *ctx, double shift, const nh_cplx *X, nh_cplx *Y,
                int ncol, int64_t ld, int ptr_kind) {
  NH_TRY(check_ctx(ctx));
  NH_CHECK(X && Y && X != Y, NH_ERR_ARG, "H·v: x and y must be distinct");
  NH_CHECK(ncol >= 1 && ld >= ctx->n, NH_ERR_ARG, "H·V: bad ncol/ld");
  if (ptr_kind == NH_PTR_DEVICE) {
    NH_TRY(launch_hv(ctx, shift, X, Y, ncol, ld));
    NH_HIP(hipStreamSynchronize(ctx->stream));
    return NH_OK;
  }
  NH_CHECK(ptr_kind == NH_PTR_HOST, NH_ERR_ARG, "bad ptr_kind");
  const int64_t n = ctx->n;
  NH_TRY(ensure_buffers(ctx, n * ncol));
  for (int k = 0; k < ncol; ++k)
    NH_HIP(hipMemcpyAsync(ctx->xbuf + k * n, X + k * ld, n * sizeof(nh_cplx),
                          hipMemcpyHostToDevice, ctx->stream));
  NH_TRY(launch_hv(ctx, shift, ctx->xbuf, ctx->ybuf, ncol, n));
  for (int k = 0; k < ncol; ++k)
    NH_HIP(hipMemcpyAsync(Y + k * ld, ctx->ybuf + k * n, n * sizeof(nh_cplx),
                          hipMemcpyDeviceToHost, ctx->stream));
  NH_HIP(hipStreamSynchronize(ctx->stream));
  return NH_OK;
}

nh_status nh_ham_export(nh_context *ctx, double *onsite, double *blocks) {
  NH_TRY(check_ctx(ctx));
  NH_CHECK(ctx->layout == NH_LAYOUT_BLOCKS && ctx->onsite && ctx->blocks64, NH_ERR_STATE,
           "nh_ham_export: needs a build in NH_LAYOUT_BLOCKS");
  const int A = ctx->n_atoms;
  if (onsite) {
    std::vector<double> tmp((size_t)A * kOnsiteStride);
    NH_HIP(hipMemcpy(tmp.data(), ctx->onsite, tmp.size() * sizeof(double),
                     hipMemcpyDeviceToHost));
    for (int i = 0; i < A; ++i)
      memcpy(onsite + (size_t)i * 17, tmp.data() + (size_t)i * kOnsiteStride,
             17 * sizeof(double));
  }
  if (blocks)
    NH_HIP(hipMemcpy(blocks, ctx->blocks64, (size_t)A * 400 * sizeof(double),
                     hipMemcpyDeviceToHost));
  return NH_OK;
}

nh_status nh_context_mem_info(nh_context *ctx, int64_t *free_bytes,
                              int64_t *pool_idle_bytes) {
  NH_TRY(check_ctx(ctx));
  size_t fr = 0, tot = 0;
  NH_HIP(hipMemGetInfo(&fr, &tot));
  if (free_bytes) *free_bytes = (int64_t)fr;
  if (pool_idle_bytes) *pool_idle_bytes = (int64_t)pool_free_bytes(ctx);
  return NH_OK;
}

nh_status nh_device_alloc(nh_context *ctx, int64_t bytes, void **dptr) {
  NH_TRY(check_ctx(ctx));
  NH_CHECK(dptr && bytes >= 0, NH_ERR_ARG, "nh_device_alloc: bad arguments");
  if (device_take(ctx, dptr, (size_t)bytes)) return NH_OK;
  return device_malloc(ctx, dptr, (size_t)bytes);
}

nh_status nh_device_free(nh_context *ctx, void *dptr) {
  NH_TRY(check_ctx(ctx));
  NH_HIP(hipStreamSynchronize(ctx->stream));
  return dptr ? device_keep(ctx, dptr) : NH_OK;
}

nh_status nh_memcpy_h2d(nh_context *ctx, void *dst, const void *src,
                        int64_t bytes) {
  NH_TRY(check_ctx(ctx));
  NH_CHECK(dst && src && bytes >= 0, NH_ERR_ARG, "nh_memcpy_h2d: bad arguments");
  NH_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
  NH_HIP(hipStreamSynchronize(ctx->stream));
  return NH_OK;
}

nh_status nh_memcpy_d2h(nh_context *ctx, void *dst, const void *src,
                        int64_t bytes) {
  NH_TRY(check_ctx(ctx));
  NH_CHECK(dst && src && bytes >= 0, NH_ERR_ARG, "nh_memcpy_d2h: bad arguments");
  NH_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
  NH_HIP(hipStreamSynchronize(ctx->stream));
  return NH_OK;
}

nh_status nh_dot(nh_context *ctx, int64_t n, const nh_cplx *x,
                 const nh_cplx *y, nh_cplx *out) {
  NH_TRY(check_ctx(ctx));
  NH_CHECK(x && y && out && n >= 0, NH_ERR_ARG, "nh_dot: bad arguments");
  double r[2];
  NH_TRY(reduce_dot(ctx, n, x, y, r));
  out->re = r[0];
  out->im = r[1];
  return NH_OK;
}

nh_status nh_dot_noalloc(nh_context *ctx, int64_t n, const nh_cplx *x,
                         const nh_cplx *y, nh_cplx *out) {
  NH_TRY(check_ctx(ctx));
  NH_CHECK(x && y && out && n >= 0, NH_ERR_ARG, "nh_dot_noalloc: bad arguments");
  double r[2];
  NH_TRY(reduce_dot_noalloc(ctx, n, x, y, r));
  out->re = r[0];
  out->im = r[1];
  return NH_OK;
}

nh_status nh_nrm2(nh_context *ctx, int64_t n, const nh_cplx *x, double *out) {
  NH_TRY(check_ctx(ctx));
  NH_CHECK(x && out && n >= 0, NH_ERR_ARG, "nh_nrm2: bad arguments");
  double s;
  NH_TRY(reduce_nrm2sq(ctx, n, x, &s));
  *out = sqrt(s);
  return NH_OK;
}

nh_status nh_axpby(nh_context *ctx, int64_t n, nh_cplx a, const nh_cplx *x,
                   nh_cplx b, nh_cplx *y) {
  NH_TRY(check_ctx(ctx));
  NH_CHECK(x && y && n >= 0, NH_ERR_ARG, "nh_axpby: bad arguments");
  NH_TRY(launch_axpby(ctx, n, a, x, b, y));
  NH_HIP(hipStreamSynchronize(ctx->stream));
  return NH_OK;
}

}  // extern "C"
