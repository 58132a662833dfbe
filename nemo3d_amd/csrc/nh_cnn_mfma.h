// Kernels of the learned start's network on the matrix cores.
//
// Products with the BF16 weights: FP32 on the FP32 matrix units, which add the
// products of one output one after the other, each rounded once, as a chain of
// multiply-adds does (checked bit by bit against fmaf): summed in the order of
// offset and channel, the forward's outputs are those of a scalar loop.
// Writing an FP32 value exactly as three BF16 ones and taking three BF16
// products is 2.8 times faster for a layer, but the BF16 units' sums are less
// accurate (parameter gradients 3.6e-6 off against 0.8e-6).
// Gradients of the weights: sums of FP32 x FP32 products over every grid
// point, kept in FP64 on the FP64 matrix units.
//
// Operand layouts (64 lanes, l): v_mfma_f32_32x32x2_f32: A[m = l % 32]
// [k = l / 32], B[k][n = l % 32], D[m = 8 (i / 4) + 4 (l / 32) + i % 4][n];
// v_mfma_f64_16x16x4: A[m = l % 16][k = l / 16], B[k][n = l % 16],
// D[m = l / 16 + 4 i][n].
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "nh_internal.h"

namespace nh {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) double f64x4;

constexpr int kCnnW = 32;  // channels of the hidden layers

__device__ __forceinline__ float bf16_to_f(uint16_t h) {
  return __uint_as_float(((uint32_t)h) << 16);
}
// round to nearest even
__device__ __forceinline__ uint16_t f_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  const uint32_t lsb = (u >> 16) & 1u;
  u += 0x7FFFu + lsb;
  return (uint16_t)(u >> 16);
}

// C + A B over 16 products: the lane's eight weights (packed BF16) and the
// eight values of the same k
__device__ __forceinline__ f32x16 mfma_f32x16(const uint4 &w, const float4 &x0, const float4 &x1,
                                              f32x16 c) {
  const uint32_t u[4] = {w.x, w.y, w.z, w.w};
  const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
  for (int j = 0; j < 8; ++j)
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(
        __uint_as_float(j % 2 ? u[j / 2] & 0xffff0000u : u[j / 2] << 16), x[j], c, 0, 0, 0);
  return c;
}

// eight consecutive floats of a row, the entries from n on zero (vec: the row
// starts on 16 bytes and n is a multiple of 4)
__device__ __forceinline__ void load8(const float *p, int n, bool vec, float (&x)[8]) {
  if (vec) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float4 v = 4 * j < n ? *reinterpret_cast<const float4 *>(p + 4 * j)
                                 : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      x[4 * j] = v.x, x[4 * j + 1] = v.y, x[4 * j + 2] = v.z, x[4 * j + 3] = v.w;
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = j < n ? p[j] : 0.0f;
  }
}

// ---- weights in operand order -------------------------------------------------

// One packed operand array per layer and use, [frag][lane][8] BF16:
//  kPackConv   frag = offset k * ks + s: W[co = l % 32][ci = ci0 + 16 s + q][k]
//  kPackConvT  (backward, data) W[co = 16 s + q][ci = l % 32][26 - k]
//  kPackHead   frag = 2 t + s: W[co = 32 t + l % 32][ci = 16 s + q]
//  kPackHeadT  frag = s: W[co = 16 s + p][ci = l % 32]
// (q = 2 j + l / 32: the products in the order of the channels; p = 8 (l / 32)
// + j: each lane reads eight consecutive ones)
enum { kPackConv, kPackConvT, kPackHead, kPackHeadT };
struct PackSeg {
  int kind, ci_n, ci0, ks, co_n;
  int64_t src, dst, frags;  // offsets into the parameters / the packed array
};
constexpr int kMaxPack = 24;
struct PackList {
  int n;
  PackSeg s[kMaxPack];
};
__global__ __launch_bounds__(256) void k_pack_weights(PackList list,
                                                      const uint16_t *__restrict__ bf,
                                                      uint16_t *__restrict__ out) {
  const PackSeg g = list.s[blockIdx.y];
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < g.frags * 512;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int j = t % 8, l = (t / 8) % 64;
    const int f = t / 512, m = l % 32;
    const int kk = g.kind == kPackHeadT ? 8 * (l / 32) + j : 2 * j + l / 32;
    int64_t src = -1;
    if (g.kind == kPackConv) {
      const int ci = g.ci0 + 16 * (f % g.ks) + kk;
      if (ci < g.ci_n) src = ((int64_t)m * g.ci_n + ci) * 27 + f / g.ks;
    } else if (g.kind == kPackConvT) {
      const int co = 16 * (f % g.ks) + kk;
      src = ((int64_t)co * g.ci_n + m) * 27 + (26 - f / g.ks);
    } else if (g.kind == kPackHead) {
      const int co = 32 * (f / 2) + m, ci = 16 * (f % 2) + kk;
      if (co < g.co_n) src = (int64_t)co * g.ci_n + ci;
    } else {
      const int co = 16 * f + kk;
      if (co < g.co_n) src = (int64_t)co * g.ci_n + m;
    }
    out[g.dst + t] = src >= 0 ? bf[g.src + src] : (uint16_t)0;
  }
}

// ---- 3x3x3 convolution ----------------------------------------------------------

// 32 outputs of every point from KS * 16 input channels (from ci0 on):
//  forward   out = relu(bias + sum) (relu only with the last channels; first
//            channels: bias, later ones add to out)
//  BWD       out = sum where mask > 0, else 0 (gradient before the lower
//            layer's relu; mask: its output)
// A workgroup keeps up to 128 points of a (y, z) plane, a rectangle that suits
// the grid, and walks along x: it stages one plane of inputs at a time in LDS
// (the rectangle and the points around it, the next plane's loads in flight
// meanwhile) and adds each plane to the three output planes it touches, so
// every operand read from LDS feeds three matrix instructions; planes beyond
// its segment only to the one it needs.  Bound by the FP32 matrix rate; the
// weights lie in LDS (54 KB), so that two workgroups share a compute unit.
// One thread per point with the weights in LDS took 3.74 ms for a layer of
// 106 x 106 x 71 points (bound by 864 scalar multiply-adds and LDS reads per
// point and output block), this 0.46 ms (0.52 with rectangles of 8 x 16 only).
constexpr int kConvPos = 192;  // points of a staged plane at most
struct ConvTile {
  int ty, tz, seg;  // ty tz <= 128, (ty + 2) (tz + 2) <= kConvPos
};
template <int KS, bool BWD>
__global__ __launch_bounds__(256, 2) void k_conv(
    int gx, int gy, int gz, ConvTile tile, int ld, int ci0, const float *__restrict__ in,
    const uint4 *__restrict__ W, const uint16_t *__restrict__ bias, bool relu,
    const float *__restrict__ mask, float *out) {
  constexpr int kOct = 2 * KS;  // groups of 8 channels
  constexpr int kItems = kConvPos * kOct, kPer = (kItems + 255) / 256;
  __shared__ uint4 wlds[27 * KS * 64];
  // a plane's even, then its odd channels, four at a time
  __shared__ float4 lds[2 * kOct * kConvPos];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, h = lane >> 5, n = lane & 31;
  const int sz = tile.tz + 2, npos = (tile.ty + 2) * sz;  // the staged plane
  const int ntz = (gz + tile.tz - 1) / tile.tz;
  const int z0 = blockIdx.x % ntz * tile.tz, y0 = blockIdx.x / ntz * tile.ty;
  const int x0 = blockIdx.y * tile.seg, x1 = min(x0 + tile.seg, gx);
  // this lane's output point (column n of wavefront w); idle ones read point 0
  const bool in_tile = 32 * w + n < tile.ty * tile.tz;
  const int lp = in_tile ? 32 * w + n : 0, ly = lp / tile.tz, lz = lp % tile.tz;
  const bool mine = in_tile && y0 + ly < gy && z0 + lz < gz;
  const int64_t plane = (int64_t)gy * gz, pt = (int64_t)(y0 + ly) * gz + z0 + lz;

  for (int f = threadIdx.x; f < 27 * KS * 64; f += 256) wlds[f] = W[f];
  float b0[16];
#pragma unroll
  for (int i = 0; i < 16; ++i)
    b0[i] = !BWD && bias ? bf16_to_f(bias[8 * (i / 4) + 4 * h + i % 4]) : 0.0f;

  // staging: item = (point of the plane, group of 8 channels)
  int64_t off[kPer];
  int cnt[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int t = threadIdx.x + 256 * i, pos = t / kOct, q = t % kOct;
    const int y = y0 - 1 + pos / sz, z = z0 - 1 + pos % sz;
    const int c = ci0 + 8 * q;
    off[i] = ((int64_t)y * gz + z) * ld + c;
    cnt[i] = pos < npos && y >= 0 && y < gy && z >= 0 && z < gz ? ld - c : 0;
  }
  const bool vec = ld % 4 == 0;
  float nx[kPer][8];
  auto load = [&](int x) {
    const float *src = in + x * plane * ld;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      if (cnt[i] > 0) {
        load8(src + off[i], cnt[i], vec, nx[i]);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) nx[i][j] = 0.0f;
      }
    }
  };
  auto stage = [&] {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int t = threadIdx.x + 256 * i, pos = t / kOct, q = t % kOct;
      if (pos < npos)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          lds[(c * kOct + q) * kConvPos + pos] =
              make_float4(nx[i][c], nx[i][2 + c], nx[i][4 + c], nx[i][6 + c]);
    }
  };
  // what the sums of output plane x start from
  auto init = [&](int x) {
    f32x16 a;
    if (!BWD && !bias && mine && x < x1) {
      const float *o = out + (x * plane + pt) * kCnnW + 4 * h;
#pragma unroll
      for (int i = 0; i < 16; ++i) a[i] = o[8 * (i / 4) + i % 4];
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) a[i] = b0[i];
    }
    return a;
  };

  f32x16 acc[3];  // outputs of planes x - 1, x, x + 1
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[d][i] = 0.0f;
  acc[2] = init(x0);
  // add the staged plane to the output planes d0 .. d1 (x - 1 + d)
  const float4 *buf = lds + h * kOct * kConvPos + (ly + 1) * sz + lz + 1;
  auto apply = [&](auto d0, auto d1) {
#pragma unroll
    for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
      for (int dz = -1; dz <= 1; ++dz)
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const float4 *b = buf + dy * sz + dz + 2 * s * kConvPos;
          const float4 v0 = b[0], v1 = b[kConvPos];
          // output plane x - 1 + d sees this plane at offset 1 - d
          const int k0 = (dy + 1) * 3 + dz + 1;
#pragma unroll
          for (int d = d0; d <= d1; ++d)
            acc[d] = mfma_f32x16(wlds[(((2 - d) * 9 + k0) * KS + s) * 64 + lane], v0, v1, acc[d]);
        }
  };
  using std::integral_constant;
  load(max(x0 - 1, 0));
  stage();
  for (int x = x0 - 1; x <= x1; ++x) {
    if (x >= 0 && x < gx) {
      const bool more = x < x1 && x + 1 < gx;
      if (more) load(x + 1);
      __syncthreads();  // this plane is staged
      if (x < x0)
        apply(integral_constant<int, 2>{}, integral_constant<int, 2>{});
      else if (x == x1)
        apply(integral_constant<int, 0>{}, integral_constant<int, 0>{});
      else
        apply(integral_constant<int, 0>{}, integral_constant<int, 2>{});
      __syncthreads();  // .. and has been read
      if (more) stage();
    }
    if (x - 1 >= x0 && mine) {
      const int64_t o = ((x - 1) * plane + pt) * kCnnW + 4 * h;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float4 v = make_float4(acc[0][4 * q], acc[0][4 * q + 1], acc[0][4 * q + 2],
                               acc[0][4 * q + 3]);
        if constexpr (BWD) {
          const float4 m = *reinterpret_cast<const float4 *>(mask + o + 8 * q);
          v.x = m.x > 0.0f ? v.x : 0.0f;
          v.y = m.y > 0.0f ? v.y : 0.0f;
          v.z = m.z > 0.0f ? v.z : 0.0f;
          v.w = m.w > 0.0f ? v.w : 0.0f;
        } else if (relu) {
          v.x = v.x > 0.0f ? v.x : 0.0f;
          v.y = v.y > 0.0f ? v.y : 0.0f;
          v.z = v.z > 0.0f ? v.z : 0.0f;
          v.w = v.w > 0.0f ? v.w : 0.0f;
        }
        *reinterpret_cast<float4 *>(out + o + 8 * q) = v;
      }
    }
    acc[0] = acc[1];
    acc[1] = acc[2];
    acc[2] = init(x + 2);
  }
}
// The tile and the x planes of a workgroup: the split that takes the least
// time, 3 seg + 2 thirds of a plane (the two planes beyond its ends cost a
// third each), 12 a round of two workgroups on each compute unit, 7 if every
// workgroup has one for itself (85 x 85 x 57 points: 484 workgroups of 8
// planes 274 us, 748 of 5 320, 220 of 17 325; 106 x 106 x 71, tiles of 8 x 16
// / 16 x 8: 490 of 16 planes 516, 504 of 14 461, 252 of 27 509).  Equal ones:
// the tile with the fewest points around it.  No more than 65,535 parts of x
// (a grid's rows).
inline ConvTile conv_tile(int gx, int gy, int gz) {
  ConvTile best{8, 16, gx};
  int64_t cost = INT64_MAX;
  for (int tz = 4; tz <= 32; ++tz) {
    const int ty = std::min(128 / tz, kConvPos / (tz + 2) - 2);
    const int64_t tiles = (int64_t)((gy + ty - 1) / ty) * ((gz + tz - 1) / tz);
    for (int n = 1, seg; n <= gx; n = seg > 1 ? (gx + seg - 2) / (seg - 1) : gx + 1) {
      seg = (gx + n - 1) / n;
      if ((gx + seg - 1) / seg > 65535) break;
      const int64_t w = tiles * ((gx + seg - 1) / seg);
      const int64_t c = (w <= 256 ? 7 : (w + 511) / 512 * 12) * (3 * seg + 2);
      if (c < cost || (c == cost && ty + tz < best.ty + best.tz)) {
        cost = c;
        best = {ty, tz, seg};
      }
    }
  }
  return best;
}

// ---- head -------------------------------------------------------------------------

// the activations of a row as operands (lane: channels 2 i + l / 32)
struct HeadAct {
  float4 v[4];
};
__device__ __forceinline__ HeadAct load_act(const float *row, int h, bool ok) {
  HeadAct a;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    float x[8];
    load8(row + 8 * s, ok ? 8 : 0, true, x);
    a.v[s] = h ? make_float4(x[1], x[3], x[5], x[7]) : make_float4(x[0], x[2], x[4], x[6]);
  }
  return a;
}
// bias + W a of rows 32 t .. 32 t + 31
__device__ __forceinline__ f32x16 head_tile(const uint4 *__restrict__ W, int t, int lane,
                                            const HeadAct &b, f32x16 acc) {
#pragma unroll
  for (int s = 0; s < 2; ++s)
    acc = mfma_f32x16(W[(2 * t + s) * 64 + lane], b.v[2 * s], b.v[2 * s + 1], acc);
  return acc;
}
// bias of rows r .. r + 3 (r a multiple of 4)
__device__ __forceinline__ void head_bias(const uint16_t *__restrict__ b, int r, int co_n,
                                          float (&v)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = r + j < co_n ? bf16_to_f(b[r + j]) : 0.0f;
}

// out[p][co] = b[co] + sum_ci W[co][ci] a[p][ci]: a wavefront takes 32 points
// and streams the packed weights (L2); bound by writing out
__global__ __launch_bounds__(256) void k_head_fwd(
    int64_t P, int co_n, const float *__restrict__ a, const uint4 *__restrict__ W,
    const uint16_t *__restrict__ bias, float *__restrict__ out) {
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const int nt = (co_n + 31) / 32;
  for (int64_t g = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); g * 32 < P;
       g += (int64_t)gridDim.x * 4) {
    const int64_t p = g * 32 + (lane & 31);
    const HeadAct b = load_act(a + p * kCnnW, h, p < P);
    for (int t = 0; t < nt; ++t) {
      f32x16 acc;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v[4];
        head_bias(bias, 32 * t + 8 * q + 4 * h, co_n, v);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[4 * q + j] = v[j];
      }
      acc = head_tile(W, t, lane, b, acc);
      if (p < P) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = 32 * t + 8 * q + 4 * h;
          float *o = out + p * co_n + r;
          if (co_n % 4 == 0) {
            if (r < co_n)
              *reinterpret_cast<float4 *>(o) = make_float4(
                  acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (r + j < co_n) o[j] = acc[4 * q + j];
          }
        }
      }
    }
  }
}

// The head at the atoms only, straight to the start block: y_e[atom nb + o]
// (re, im) = channels 2 ((e 2 + slot) nb + o) and the next of the atom's
// point.  A wavefront takes 32 atoms, kMapRows channels at a time (whole
// states: 4 nb divides them), keeps each atom's slot in LDS and writes them
// out state by state.  Through the head's output of all points (as large as
// the start block) it took 5.25 + 0.56 ms for 786,520 atoms, this 0.50 ms
// (2.0 GB written, 0.43 ms at the rate of a copy; half its products are for
// the slot an atom is not in).  The bias goes through LDS and the places are
// stepped on instead of divided out: with 80 short loads of the bias a block
// and the divisions the vector units were as busy as the matrix units (0.74).
constexpr int kMapRows = 160;
__global__ __launch_bounds__(256) void k_head_map(
    int64_t A, int nb, int ne, int co_n, const int32_t *__restrict__ point,
    const int32_t *__restrict__ slot, const float *__restrict__ act,
    const uint4 *__restrict__ W, const uint16_t *__restrict__ bias, double2 *__restrict__ Y,
    int64_t ld) {
  // [wave][atom][kMapRows / 2], rows of an odd number of 16-byte chunks
  constexpr int kRow = kMapRows / 2 + 4;
  __shared__ float lds[4][32 * kRow];
  __shared__ float4 blds[4][kMapRows / 4];  // a block's bias
  const int lane = threadIdx.x & 63, h = lane >> 5, n = lane & 31;
  float *buf = lds[threadIdx.x >> 6];
  float4 *brow = blds[threadIdx.x >> 6];
  const int per = kMapRows / (4 * nb);  // states of a block
  const int da = 64 / nb, dq = 64 % nb;  // 64 entries on, in atoms and entries
  for (int64_t g = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); g * 32 < A;
       g += (int64_t)gridDim.x * 4) {
    const int64_t a0 = g * 32, at = a0 + n;
    const bool ok = at < A;
    const int sl = ok ? slot[at] : 0;
    const HeadAct b = load_act(act + (ok ? (int64_t)point[at] : 0) * kCnnW, h, ok);
    const int rows = (int)min((int64_t)32, A - a0) * nb;  // entries of a state
    for (int e0 = 0; e0 < ne; e0 += per) {
      const int t0 = e0 * 4 * nb / 32;
      if (lane < kMapRows / 4) {
        float v[4];
        head_bias(bias, 32 * t0 + 4 * lane, co_n, v);
        brow[lane] = make_float4(v[0], v[1], v[2], v[3]);
      }
      wave_sync();
      // rows r .. r + 3 belong to one state and slot (2 nb is a multiple of
      // 4): o = r % (4 nb) less the slot's rows, dst the state's place
      int o = 4 * h - (sl ? 2 * nb : 0);
      float *dst = buf + n * kRow;
#pragma unroll
      for (int t = 0; t < kMapRows / 32; ++t) {
        f32x16 acc;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4 v = brow[8 * t + 2 * q + h];
          acc[4 * q] = v.x, acc[4 * q + 1] = v.y, acc[4 * q + 2] = v.z, acc[4 * q + 3] = v.w;
        }
        acc = head_tile(W, t0 + t, lane, b, acc);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (o >= 0 && o < 2 * nb)
            *reinterpret_cast<float4 *>(dst + o) =
                make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
          o += 8;
          if (o >= (sl ? 2 * nb : 4 * nb)) {  // the next state
            o -= 4 * nb;
            dst += 2 * nb;
          }
        }
      }
      wave_sync();
      for (int e = 0; e < per && e0 + e < ne; ++e) {
        double2 *y = Y + (e0 + e) * ld + a0 * nb;
        int off = (lane / nb) * kRow + 2 * (lane % nb), q = lane % nb;
        for (int i = lane; i < rows; i += 64) {
          const float2 s = *reinterpret_cast<const float2 *>(buf + e * 2 * nb + off);
          y[i] = make_double2(s.x, s.y);
          off += da * kRow + 2 * dq;
          q += dq;
          if (q >= nb) {
            q -= nb;
            off += kRow - 2 * nb;
          }
        }
      }
      wave_sync();
    }
  }
}

// head backward, data: out[p][ci] = sum_co W[co][ci] dout[p][co] where the
// last layer's output act > 0, else 0; a wavefront takes 32 points, bound by
// reading dout (1.05 GB for 85 x 85 x 57 points and 640 channels: 0.33 ms, a
// wavefront per point 7.7 ms)
__global__ __launch_bounds__(256) void k_head_bwd_data(
    int64_t P, int co_n, const float *__restrict__ dout, const uint4 *__restrict__ W,
    const float *__restrict__ act, float *__restrict__ out) {
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const bool vec = co_n % 4 == 0;
  for (int64_t g = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); g * 32 < P;
       g += (int64_t)gridDim.x * 4) {
    const int64_t p = g * 32 + (lane & 31);
    const float *row = dout + p * co_n + 8 * h;
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll 4
    for (int k = 0; k < co_n; k += 16) {
      float x[8];
      load8(row + k, p < P ? co_n - k - 8 * h : 0, vec, x);
      acc = mfma_f32x16(W[(k / 16) * 64 + lane], make_float4(x[0], x[1], x[2], x[3]),
                        make_float4(x[4], x[5], x[6], x[7]), acc);
    }
    if (p < P) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t o = p * kCnnW + 8 * q + 4 * h;
        const float4 m = *reinterpret_cast<const float4 *>(act + o);
        *reinterpret_cast<float4 *>(out + o) =
            make_float4(m.x > 0.0f ? acc[4 * q] : 0.0f, m.y > 0.0f ? acc[4 * q + 1] : 0.0f,
                        m.z > 0.0f ? acc[4 * q + 2] : 0.0f, m.w > 0.0f ? acc[4 * q + 3] : 0.0f);
      }
    }
  }
}

// ---- weight gradients -----------------------------------------------------------

// Sums over points in FP64 on the matrix units, four points an instruction;
// a workgroup takes a chunk of the points (its wavefronts share it and add up
// in LDS) and leaves its sums in part[chunk]; k_grad_sum adds the chunks in
// order.

// add the four wavefronts' sums into wavefront 0's (N doubles a lane)
template <int N>
__device__ __forceinline__ void wave_sums(double (&v)[N], double *lds) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int k = 1; k < 4; ++k) {
    __syncthreads();
    if (w == k)
#pragma unroll
      for (int i = 0; i < N; ++i) lds[i * 64 + lane] = v[i];
    __syncthreads();
    if (w == 0)
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] += lds[i * 64 + lane];
  }
}

// conv layer: part[chunk][(k * 32 + co) * cp + ci] = sum_p d[p][co] in[p + d_k][ci]
// (cp = ci_n rounded up to 16; sums of channels from ci_n on are not read),
// then 32 sums of d (bias).  blockIdx.x: chunk and (dx, dy); blockIdx.y: 16 NT
// input channels.  A wavefront takes lines of z, each of an instruction's four
// points a quarter of the line: going along it, a point's inputs serve the
// next two points as well and are loaded and converted once.  One workgroup
// per (co, ci) with 27 sums a thread read both arrays 32 times and took 15.9 ms
// for 85 x 85 x 57 points; four neighbouring points an instruction, each input
// loaded for all three offsets, 0.51 ms; this 0.42 ms (0.31 ms at the FP64
// matrix rate; two workgroups a compute unit 0.44).
template <int NT>
__global__ __launch_bounds__(256, 3) void k_conv_bwd_w(
    int gx, int gy, int gz, int ci_n, int chunks, const float *__restrict__ d,
    const float *__restrict__ in, double *__restrict__ part, int64_t len) {
  __shared__ double lds[3 * 2 * NT * 4 * 64];
  const int lane = threadIdx.x & 63, m = lane & 15, kz = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the nine (dx, dy) of a chunk follow one another on one XCD (workgroups go
  // round robin over 8)
  const int full = chunks / 8 * 72, g = blockIdx.x;
  const int chunk = g < full ? g / 72 * 8 + g % 8 : chunks / 8 * 8 + (g - full) % (chunks % 8);
  const int dd = g < full ? g / 8 % 9 : (g - full) / (chunks % 8);
  const int dx = dd / 3 - 1, dy = dd % 3 - 1;
  const int c0 = blockIdx.y * 16 * NT, cp = (ci_n + 15) / 16 * 16;
  const int64_t lines = (int64_t)gx * gy;
  const int64_t per = (lines + chunks - 1) / chunks;
  const int64_t l1 = min((chunk + 1) * per, lines);
  f64x4 acc[3][2][NT];
  double sb[2] = {0.0, 0.0};
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < NT; ++b) acc[k][a][b] = f64x4{0.0, 0.0, 0.0, 0.0};
  // lane group kz goes over points kz R .. kz R + R - 1 of a line; four points
  // are loaded while the last four are multiplied
  const int R = (gz + 3) / 4;
  struct Four {
    float a[4][2], b[4][NT];  // gradients of point j0 + s, inputs of the next
    float b0[2][NT];          // inputs before and at the line's first point
    int j0;
  };
  uint32_t bo[NT];  // the lane's place; channels past the last: the last
  const uint32_t ao = kz * R * kCnnW + m;
#pragma unroll
  for (int t = 0; t < NT; ++t) bo[t] = kz * R * ci_n + min(c0 + 16 * t + m, ci_n - 1);
  int64_t l = chunk * per + w;
  int x = l / gy, y = l % gy, j0 = 0;
  const float *dl = nullptr, *il = nullptr;
  auto line = [&] {  // the next line whose neighbour is in the grid
    while (l < l1 && (x + dx < 0 || y + dy < 0 || x + dx >= gx || y + dy >= gy)) {
      l += 4;
      for (y += 4; y >= gy; y -= gy) ++x;
    }
    dl = d + l * gz * kCnnW;
    il = in + (l + dx * (int64_t)gy + dy) * gz * ci_n;
  };
  auto load = [&](Four &e) {
    // inputs of point kz R + j, zero outside the line
    auto edge = [&](int j, float (&v)[NT]) {
      const int q = kz * R + j, qc = min(max(q, 0), gz - 1) - kz * R;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const float f = il[(int64_t)bo[t] + qc * ci_n];
        v[t] = q >= 0 && q < gz ? f : 0.0f;
      }
    };
    e.j0 = j0;
    if (j0 == 0) {
      edge(-1, e.b0[0]);
      edge(0, e.b0[1]);
    }
    if (3 * R + j0 + 4 < gz) {  // all points and their neighbours in the line
      const float *pa = dl + j0 * kCnnW, *pb = il + (int64_t)(j0 + 1) * ci_n;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
#pragma unroll
        for (int t = 0; t < 2; ++t) e.a[s][t] = (pa + s * kCnnW + 16 * t)[ao];
#pragma unroll
        for (int t = 0; t < NT; ++t) e.b[s][t] = (pb + s * ci_n)[bo[t]];
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int p = kz * R + j0 + s, pc = min(p, gz - 1);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const float f = dl[pc * kCnnW + 16 * t + m];
          e.a[s][t] = p < gz ? f : 0.0f;
        }
        edge(j0 + s + 1, e.b[s]);
      }
    }
    j0 += 4;
    if (j0 >= R) {
      j0 = 0;
      l += 4;
      for (y += 4; y >= gy; y -= gy) ++x;
      line();
    }
  };
  line();
  Four next;
#pragma unroll
  for (int t = 0; t < NT; ++t) next.b0[0][t] = next.b0[1][t] = 0.0f;
  double before[NT], here[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) before[t] = here[t] = 0.0;
  bool more = l < l1;
  if (more) load(next);
  while (more) {
    const Four e = next;
    more = l < l1;
    if (more) load(next);
    if (e.j0 == 0) {
#pragma unroll
      for (int t = 0; t < NT; ++t) before[t] = e.b0[0][t], here[t] = e.b0[1][t];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (e.j0 + s >= R) break;
      const double da[2] = {e.a[s][0], e.a[s][1]};
#pragma unroll
      for (int t = 0; t < 2; ++t) sb[t] += da[t];
#pragma unroll
      for (int u = 0; u < NT; ++u) {
        const double after = e.b[s][u];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          acc[0][t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(da[t], before[u], acc[0][t][u], 0, 0, 0);
          acc[1][t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(da[t], here[u], acc[1][t][u], 0, 0, 0);
          acc[2][t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(da[t], after, acc[2][t][u], 0, 0, 0);
        }
        before[u] = here[u];
        here[u] = after;
      }
    }
  }
  double v[3 * 2 * NT * 4];
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[((k * 2 + t) * NT + u) * 4 + i] = acc[k][t][u][i];
  wave_sums(v, lds);
  double *p = part + chunk * len;
  if (w == 0)
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int co = 16 * t + kz + 4 * i, ci = c0 + 16 * u + m;
            if (ci < cp)
              p[((dd * 3 + k) * kCnnW + co) * (int64_t)cp + ci] =
                  v[((k * 2 + t) * NT + u) * 4 + i];
          }
  // bias: the offset (0, 0) passes over every point once
  if (dd == 4 && blockIdx.y == 0) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      sb[t] += __shfl_xor(sb[t], 16, 64);
      sb[t] += __shfl_xor(sb[t], 32, 64);
    }
    wave_sums(sb, lds);
    if (w == 0 && kz == 0)
#pragma unroll
      for (int t = 0; t < 2; ++t) p[27 * kCnnW * (int64_t)cp + 16 * t + m] = sb[t];
  }
}
// head: part[chunk][co * 32 + ci] = sum_p d[p][co] a[p][ci], then co_n sums of
// d.  blockIdx.y: 64 output channels.  640 channels of 85 x 85 x 57 points:
// 33.9 ms with a workgroup per channel, 0.34 ms now (0.23 at the matrix rate;
// 0.37 with every address and bound worked out per lane).
__global__ __launch_bounds__(256, 3) void k_head_bwd_w(
    int64_t P, int co_n, const float *__restrict__ d, const float *__restrict__ act,
    double *__restrict__ part, int64_t len) {
  __shared__ double lds[4 * 2 * 4 * 64];
  const int lane = threadIdx.x & 63, m = lane & 15, kp = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int co0 = blockIdx.y * 64;
  const int64_t per = (P + gridDim.x - 1) / gridDim.x;
  const int64_t p1 = min((blockIdx.x + 1) * per, P);
  f64x4 acc[4][2];
  double sb[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u) acc[t][u] = f64x4{0.0, 0.0, 0.0, 0.0};
  // eight points (two instructions' worth) are loaded while the last eight
  // are multiplied
  struct Eight {
    float a[2][4], b[2][2];
  };
  int64_t p0 = blockIdx.x * per + 8 * w;
  const uint32_t ao = kp * co_n + m, bo = kp * kCnnW + m;  // the lane's place
  auto load = [&](Eight &e) {
    if (co0 + 64 <= co_n && p0 + 8 <= p1) {
      // inside: the wavefront's addresses and the lane's place, no tests
      const float *pa = d + p0 * co_n + co0, *pb = act + p0 * kCnnW;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int t = 0; t < 4; ++t) e.a[s][t] = (pa + 4 * s * (int64_t)co_n + 16 * t)[ao];
#pragma unroll
        for (int u = 0; u < 2; ++u) e.b[s][u] = (pb + 4 * s * kCnnW + 16 * u)[bo];
      }
    } else {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int64_t p = p0 + 4 * s + kp;
#pragma unroll
        for (int t = 0; t < 4; ++t)
          e.a[s][t] = p < p1 && co0 + 16 * t + m < co_n ? d[p * co_n + co0 + 16 * t + m] : 0.0f;
#pragma unroll
        for (int u = 0; u < 2; ++u) e.b[s][u] = p < p1 ? act[p * kCnnW + 16 * u + m] : 0.0f;
      }
    }
    p0 += 32;
  };
  Eight next;
  bool more = p0 < p1;
  if (more) load(next);
  while (more) {
    const Eight e = next;
    more = p0 < p1;
    if (more) load(next);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        sb[t] += e.a[s][t];
#pragma unroll
        for (int u = 0; u < 2; ++u)
          acc[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)e.a[s][t], (double)e.b[s][u],
                                                           acc[t][u], 0, 0, 0);
      }
  }
  double v[4 * 2 * 4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[(t * 2 + u) * 4 + i] = acc[t][u][i];
  wave_sums(v, lds);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    sb[t] += __shfl_xor(sb[t], 16, 64);
    sb[t] += __shfl_xor(sb[t], 32, 64);
  }
  wave_sums(sb, lds);
  if (w != 0) return;
  double *o = part + blockIdx.x * len;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int co = co0 + 16 * t + kp + 4 * i;
        if (co < co_n) o[(int64_t)co * kCnnW + 16 * u + m] = v[(t * 2 + u) * 4 + i];
      }
    if (kp == 0 && co0 + 16 * t + m < co_n)
      o[(int64_t)co_n * kCnnW + co0 + 16 * t + m] = sb[t];
  }
}

// grad[..] = sum of the chunks' partials, in order; conv: partials
// [k][co][cp] and 32 of the bias to W[co][ci][k], b; else as they stand.
// A sum that is not finite is taken again by the workgroup, point by point,
// without the points whose gradient is zero: the matrix units multiply those
// too, and a zero times an infinite activation (a point that the loss does not
// reach) is NaN.
struct GradIn {  // gradients d [P][co_n], inputs x [P][ci_n] of the layer
  int gx, gy, gz, co_n, ci_n;
  const float *d, *x;
};
__global__ __launch_bounds__(256) void k_grad_sum(int chunks, int64_t len, int conv_ci,
                                                  const double *__restrict__ part, GradIn g,
                                                  float *__restrict__ grad) {
  __shared__ int32_t bad[256];
  __shared__ double lds[4];
  const int64_t t0 = blockIdx.x * (int64_t)blockDim.x, t = t0 + threadIdx.x;
  const int cp = conv_ci ? (conv_ci + 15) / 16 * 16 : kCnnW;
  const int64_t nw = (int64_t)(conv_ci ? 27 : 1) * g.co_n * cp;  // products, then the bias
  auto place = [&](int64_t e) {  // -1: padding
    if (!conv_ci) return e;
    if (e >= nw) return (int64_t)kCnnW * conv_ci * 27 + (e - nw);
    const int ci = e % cp;
    const int64_t r = e / cp;
    return ci >= conv_ci ? (int64_t)-1 : ((r % kCnnW) * conv_ci + ci) * 27 + r / kCnnW;
  };
  const int64_t o = t < len ? place(t) : -1;
  double s = 0.0;
  if (o >= 0)
#pragma unroll 8
    for (int c = 0; c < chunks; ++c) s += part[c * len + t];
  if (o >= 0) grad[o] = (float)s;
  const bool again = o >= 0 && t < nw && !isfinite(s);
  bad[threadIdx.x] = again;
  if (!__syncthreads_or(again)) return;
  for (int e = 0; e < 256; ++e) {
    if (!bad[e]) continue;
    const int64_t r = (t0 + e) / cp;
    const int ci = (t0 + e) % cp, co = r % g.co_n, k = conv_ci ? (int)(r / g.co_n) : 13;
    const int dx = k / 9 - 1, dy = k / 3 % 3 - 1, dz = k % 3 - 1;
    const int64_t P = (int64_t)g.gx * g.gy * g.gz;
    double v = 0.0;
    for (int64_t p = threadIdx.x; p < P; p += 256) {
      const float d = g.d[p * g.co_n + co];
      if (d == 0.0f) continue;
      const int z = p % g.gz + dz, y = p / g.gz % g.gy + dy;
      const int x = (int)(p / ((int64_t)g.gy * g.gz)) + dx;
      if (x < 0 || y < 0 || z < 0 || x >= g.gx || y >= g.gy || z >= g.gz) continue;
      v += (double)d * g.x[(((int64_t)x * g.gy + y) * g.gz + z) * g.ci_n + ci];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) grad[place(t0 + e)] = (float)(lds[0] + lds[1] + lds[2] + lds[3]);
  }
}

}  // namespace nh
