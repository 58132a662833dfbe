// 3-D convolutional network of the learned warm start: forward, backward,
// Adam and the eigenvector-subspace loss, all on the device.
//
// Network: L conv layers (3x3x3, zero padding, ReLU) c_in -> W -> ... -> W,
// then a 1x1x1 head W -> c_out.  Activations are FP32, channels last
// ([point][channel], point = (x*gy + y)*gz + z).  Weights are kept as FP32
// master copies for Adam and used as BF16 in the forward and backward
// products (FP32 accumulation; kernels in nh_cnn_mfma.h).
// Parameter vector: for each conv layer W_l[co][ci][27], b_l[co]; then the
// head W_h[co][ci], b_h[co].
//
// Loss of one training structure with target eigenvectors v_f (FP64, from
// the plain solver) and predicted vectors y_e (the head output mapped to
// atoms): L = mean_e (1 - ||P_e y_e||^2 / ||y_e||^2), P_e the projector on
// the degenerate cluster of target e (a Kramers pair in the spin model).
// It is invariant to the phase of each state and to rotations inside a
// degenerate pair.
#include <chrono>
#include <cstring>
#include <vector>

#include "nh_blockla.h"
#include "nh_cnn_mfma.h"
#include "nh_vector.h"

struct nh_cnn {
  nh_context *ctx = nullptr;
  int device = 0;  // the context may be destroyed before the network
  int c_in = 0, width = 0, layers = 0, c_out = 0;
  int64_t n_params = 0;
  std::vector<int64_t> w_off, b_off;  // per layer (conv layers, then head)
  float *master = nullptr;            // FP32 parameters
  uint16_t *bf = nullptr;             // BF16 copy used by the products
  uint16_t *packed = nullptr;         // .. in the order of the matrix operands
  int64_t n_packed = 0;
  nh::PackList pack{};                // .. its parts
  std::vector<std::vector<int>> fwd_seg;  // per conv layer: parts of 32 input channels
  std::vector<int> bwd_seg;               // per conv layer (0: none)
  int head_seg = 0, headt_seg = 0;
  float *grad = nullptr, *m1 = nullptr, *m2 = nullptr;
  int64_t step = 0;
  // activations for the current grid
  int64_t cap_points = 0;
  std::vector<float *> act;  // per conv layer, [P][W] (after the relu)
  float *in = nullptr;
  // head output or its gradient [P][c_out], gradients before a relu [P][W],
  // partial sums: allocated by the calls that need them
  int64_t cap_out = 0, cap_grad = 0;
  size_t cap_part = 0;
  float *out = nullptr, *dpre[2] = {nullptr, nullptr};
  double *part = nullptr;
};

namespace nh {
namespace {

__global__ void k_to_bf16(int64_t n, const float *__restrict__ a,
                          uint16_t *__restrict__ b) {
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * blockDim.x)
    b[k] = f_to_bf16(a[k]);
}

__global__ void k_adam(int64_t n, float *__restrict__ w,
                       const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, float lr, float b1, float b2,
                       float c1, float c2, float eps) {
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * blockDim.x) {
    const float gk = g[k];
    const float mk = b1 * m[k] + (1.0f - b1) * gk;
    const float vk = b2 * v[k] + (1.0f - b2) * gk * gk;
    m[k] = mk;
    v[k] = vk;
    w[k] -= lr * (mk / c1) / (sqrtf(vk / c2) + eps);
  }
}

// Gradient w.r.t. the start block, g_e = sum_f v_f M[f][e] + D[e] y_e, to the
// head output's gradient (points without atoms keep the zeros they were
// given): one pass over the targets and the prediction, no gradient block in
// between.
__global__ __launch_bounds__(256) void k_loss_grad(
    int64_t A, int nb, int nf, int ne, int c_out, const int32_t *__restrict__ point,
    const int32_t *__restrict__ slot, const double2 *__restrict__ V,
    const double2 *__restrict__ Y, int64_t ld, const double2 *__restrict__ MD,
    float *__restrict__ dout) {
  __shared__ double2 m[17 * 8];  // M[f][e], then D[e]
  for (int t = threadIdx.x; t < 17 * 8; t += blockDim.x) m[t] = MD[t];
  __syncthreads();
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < A * nb;
       t += (int64_t)gridDim.x * blockDim.x) {
    double2 g[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] = make_double2(0.0, 0.0);
    for (int f = 0; f < nf; ++f) {
      const double2 v = V[f * ld + t];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const double2 c = m[f * 8 + e];
        g[e].x += v.x * c.x - v.y * c.y;
        g[e].y += v.x * c.y + v.y * c.x;
      }
    }
    const int64_t a = t / nb;
    float *dst = dout + (int64_t)point[a] * c_out + 2 * (slot[a] * nb + t % nb);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < ne) {
        const double2 y = Y[e * ld + t];
        const double d = m[16 * 8 + e].x;
        dst[4 * e * nb] = (float)(g[e].x + d * y.x);
        dst[4 * e * nb + 1] = (float)(g[e].y + d * y.y);
      }
  }
}

int g1(int64_t n, int b = 256) {
  int64_t g = (n + b - 1) / b;
  return (int)(g < 1 ? 1 : (g > 65535 ? 65535 : g));
}

// (re)allocate *p for `bytes`
template <typename T>
nh_status regrow(nh_cnn *c, T **p, size_t bytes) {
  (void)hipFree(*p);
  *p = nullptr;
  return device_malloc(c->ctx, (void **)p, bytes);
}

nh_status ensure_acts(nh_cnn *c, int64_t P) {
  if (P <= c->cap_points) return NH_OK;
  c->cap_points = 0;
  c->act.resize(c->layers, nullptr);
  for (int l = 0; l < c->layers; ++l)
    NH_TRY(regrow(c, &c->act[l], P * c->width * sizeof(float)));
  NH_TRY(regrow(c, &c->in, P * c->c_in * sizeof(float)));
  c->cap_points = P;
  return NH_OK;
}
nh_status ensure_out(nh_cnn *c, int64_t P) {
  if (P <= c->cap_out) return NH_OK;
  c->cap_out = 0;
  NH_TRY(regrow(c, &c->out, P * c->c_out * sizeof(float)));
  c->cap_out = P;
  return NH_OK;
}
nh_status ensure_grads(nh_cnn *c, int64_t P) {
  if (P <= c->cap_grad) return NH_OK;
  c->cap_grad = 0;
  for (float *&q : c->dpre) NH_TRY(regrow(c, &q, P * c->width * sizeof(float)));
  c->cap_grad = P;
  return NH_OK;
}
nh_status ensure_part(nh_cnn *c, size_t count) {
  if (count <= c->cap_part) return NH_OK;
  c->cap_part = 0;
  NH_TRY(regrow(c, &c->part, count * sizeof(double)));
  c->cap_part = count;
  return NH_OK;
}

template <bool BWD>
void launch_conv(nh_cnn *c, int gx, int gy, int gz, const ConvTile &tile, int ld,
                 const PackSeg &g, bool last, const float *in, const uint16_t *bias, const float *mask, float *out) {
  const dim3 grid((gz + tile.tz - 1) / tile.tz * ((gy + tile.ty - 1) / tile.ty),
                  (gx + tile.seg - 1) / tile.seg);
  const uint4 *W = reinterpret_cast<const uint4 *>(c->packed + g.dst);
  if (BWD || g.ks == 2)
    hipLaunchKernelGGL((k_conv<2, BWD>), grid, dim3(256), 0, c->ctx->stream, gx, gy, gz,
                       tile, ld, g.ci0, in, W, bias, last, mask, out);
  else
    hipLaunchKernelGGL((k_conv<1, false>), grid, dim3(256), 0, c->ctx->stream, gx, gy, gz,
                       tile, ld, g.ci0, in, W, bias, last, mask, out);
}

// the conv layers: act[l] for every point
nh_status forward(nh_cnn *c, int gx, int gy, int gz) {
  const ConvTile tile = conv_tile(gx, gy, gz);
  const float *src = c->in;
  int ci = c->c_in;
  for (int l = 0; l < c->layers; ++l) {
    const auto &segs = c->fwd_seg[l];
    for (size_t k = 0; k < segs.size(); ++k)
      launch_conv<false>(c, gx, gy, gz, tile, ci, c->pack.s[segs[k]], k + 1 == segs.size(), src,
                         k == 0 ? c->bf + c->b_off[l] : nullptr, nullptr, c->act[l]);
    src = c->act[l];
    ci = c->width;
  }
  NH_HIP(hipGetLastError());
  return NH_OK;
}
// the head at every point, to c->out
nh_status head(nh_cnn *c, int64_t P) {
  const int L = c->layers;
  hipLaunchKernelGGL(k_head_fwd, dim3(g1(P, 128)), dim3(256), 0, c->ctx->stream, P, c->c_out,
                     c->act[L - 1],
                     reinterpret_cast<const uint4 *>(c->packed + c->pack.s[c->head_seg].dst),
                     c->bf + c->b_off[L], c->out);
  NH_HIP(hipGetLastError());
  return NH_OK;
}
// the head at the atoms, to the start block
nh_status head_map(nh_cnn *c, int ne, const int32_t *point, const int32_t *slot, double2 *Y) {
  const nh_context *x = c->ctx;
  const int L = c->layers;
  hipLaunchKernelGGL(k_head_map, dim3(g1(x->n_atoms, 128)), dim3(256), 0, x->stream,
                     (int64_t)x->n_atoms, x->nb, ne, c->c_out, point, slot, c->act[L - 1],
                     reinterpret_cast<const uint4 *>(c->packed + c->pack.s[c->head_seg].dst),
                     c->bf + c->b_off[L], Y, x->n);
  NH_HIP(hipGetLastError());
  return NH_OK;
}

// parameter gradient of sum(out * dout), dout [P][c_out]
nh_status backward(nh_cnn *c, int gx, int gy, int gz, const float *dout) {
  const int64_t P = (int64_t)gx * gy * gz;
  hipStream_t st = c->ctx->stream;
  const int L = c->layers, W = c->width;
  NH_TRY(ensure_grads(c, P));
  // chunks of points, none smaller than a few lines: as many workgroups as
  // run at a time (4 a compute unit for the head; the conv layers with their
  // nine offsets 3, up to 16 channels 4: 85 x 85 x 57 points 415 us, with half
  // as many 445; 225 and 259)
  const int co_tiles = (c->c_out + 63) / 64;
  const int hch = (int)std::max<int64_t>(1, std::min<int64_t>(P / 256, 1024 / co_tiles));
  const int64_t hlen = (int64_t)c->c_out * (W + 1);
  auto conv_chunks = [&](int ci) {
    return (int)std::max<int64_t>(1, std::min<int64_t>((int64_t)gx * gy / 8, ci <= 16 ? 113 : 85));
  };
  const int cmax = std::max((c->c_in + 15) / 16 * 16, W);
  NH_TRY(ensure_part(c, std::max(hch * hlen, (int64_t)conv_chunks(1) * (27 * W * cmax + W))));
  auto sum = [&](int chunks, int64_t len, int conv_ci, const float *d, const float *x,
                 float *grad) {
    const GradIn g{gx, gy, gz, conv_ci ? W : c->c_out, conv_ci ? conv_ci : W, d, x};
    hipLaunchKernelGGL(k_grad_sum, dim3((len + 255) / 256), dim3(256), 0, st, chunks, len,
                       conv_ci, c->part, g, grad);
  };
  hipLaunchKernelGGL(k_head_bwd_w, dim3(hch, co_tiles), dim3(256), 0, st, P, c->c_out, dout,
                     c->act[L - 1], c->part, hlen);
  sum(hch, hlen, 0, dout, c->act[L - 1], c->grad + c->w_off[L]);
  hipLaunchKernelGGL(k_head_bwd_data, dim3(g1(P, 128)), dim3(256), 0, st, P, c->c_out, dout,
                     reinterpret_cast<const uint4 *>(c->packed + c->pack.s[c->headt_seg].dst),
                     c->act[L - 1], c->dpre[0]);
  const ConvTile tile = conv_tile(gx, gy, gz);
  for (int l = L - 1; l >= 0; --l) {
    const int ci = l == 0 ? c->c_in : W;
    const float *in = l == 0 ? c->in : c->act[l - 1];
    const int64_t len = 27 * W * (int64_t)((ci + 15) / 16 * 16) + W;
    const int cch = conv_chunks(ci);
    if (ci <= 16)
      hipLaunchKernelGGL(k_conv_bwd_w<1>, dim3(9 * cch), dim3(256), 0, st, gx, gy, gz, ci,
                         cch, c->dpre[0], in, c->part, len);
    else
      hipLaunchKernelGGL(k_conv_bwd_w<2>, dim3(9 * cch, (ci + 31) / 32), dim3(256), 0, st, gx,
                         gy, gz, ci, cch, c->dpre[0], in, c->part, len);
    sum(cch, len, ci, c->dpre[0], in, c->grad + c->w_off[l]);
    if (l > 0) {
      launch_conv<true>(c, gx, gy, gz, tile, W, c->pack.s[c->bwd_seg[l]], true, c->dpre[0], nullptr,
                        c->act[l - 1], c->dpre[1]);
      std::swap(c->dpre[0], c->dpre[1]);
    }
  }
  NH_HIP(hipGetLastError());
  return NH_OK;
}

void init_layout(nh_cnn *c) {
  c->w_off.clear();
  c->b_off.clear();
  int64_t off = 0;
  int ci = c->c_in;
  for (int l = 0; l < c->layers; ++l) {
    c->w_off.push_back(off);
    off += (int64_t)c->width * ci * 27;
    c->b_off.push_back(off);
    off += c->width;
    ci = c->width;
  }
  c->w_off.push_back(off);
  off += (int64_t)c->c_out * ci;
  c->b_off.push_back(off);
  off += c->c_out;
  c->n_params = off;
  // packed operands (k_pack_weights)
  int64_t dst = 0;
  auto add = [&](int kind, int ci_n, int ci0, int ks, int co_n, int64_t src, int64_t frags) {
    c->pack.s[c->pack.n] = PackSeg{kind, ci_n, ci0, ks, co_n, src, dst, frags};
    dst += frags * 512;
    return c->pack.n++;
  };
  c->pack.n = 0;
  ci = c->c_in;
  for (int l = 0; l < c->layers; ++l) {
    c->fwd_seg.emplace_back();
    for (int ci0 = 0; ci0 < ci; ci0 += 32) {
      const int ks = std::min(2, (ci - ci0 + 15) / 16);
      c->fwd_seg[l].push_back(add(kPackConv, ci, ci0, ks, c->width, c->w_off[l], 27 * ks));
    }
    c->bwd_seg.push_back(l == 0 ? 0 : add(kPackConvT, ci, 0, 2, c->width, c->w_off[l], 54));
    ci = c->width;
  }
  // the head's rows are padded to whole blocks of k_head_map
  const int64_t blocks = (c->c_out + kMapRows - 1) / kMapRows;
  c->head_seg = add(kPackHead, ci, 0, 2, c->c_out, c->w_off[c->layers],
                    blocks * (kMapRows / 32) * 2);
  c->headt_seg = add(kPackHeadT, ci, 0, 1, c->c_out, c->w_off[c->layers], (c->c_out + 15) / 16);
  c->n_packed = dst;
}

nh_status sync_bf16(nh_cnn *c) {
  hipLaunchKernelGGL(k_to_bf16, dim3(g1(c->n_params)), dim3(256), 0,
                     c->ctx->stream, c->n_params, c->master, c->bf);
  hipLaunchKernelGGL(k_pack_weights, dim3(54, c->pack.n), dim3(256), 0, c->ctx->stream,
                     c->pack, c->bf, c->packed);
  NH_HIP(hipGetLastError());
  return NH_OK;
}

nh_status upload_feats(nh_cnn *c, const float *feat, int64_t P) {
  NH_TRY(ensure_acts(c, P));
  NH_HIP(hipMemcpyAsync(c->in, feat, P * c->c_in * sizeof(float),
                        hipMemcpyHostToDevice, c->ctx->stream));
  return NH_OK;
}

}  // namespace
}  // namespace nh

using namespace nh;

extern "C" {

nh_status nh_cnn_create(nh_context *ctx, int c_in, int width, int layers,
                        int c_out, uint64_t seed, nh_cnn **out) {
  NH_CHECK(ctx && out && c_in > 0 && c_in <= 64 && width == 32 && layers >= 1 &&
               layers <= 8 && c_out > 0,
           NH_ERR_ARG, "nh_cnn_create: bad shape");
  (void)hipGetLastError();
  NH_HIP(hipSetDevice(ctx->device));
  nh_cnn *c = new nh_cnn();
  c->ctx = ctx;
  c->device = ctx->device;
  c->c_in = c_in;
  c->width = width;
  c->layers = layers;
  c->c_out = c_out;
  init_layout(c);
  std::vector<float> w(c->n_params, 0.0f);
  uint64_t s = 0x9E3779B97F4A7C15ull ^ seed;
  auto gauss = [&]() {
    double u[2];
    for (double &v : u) {
      s = s * 6364136223846793005ull + 1442695040888963407ull;
      v = ((double)(s >> 11) + 0.5) / 9007199254740992.0;
    }
    return std::sqrt(-2.0 * std::log(u[0])) * std::cos(6.283185307179586 * u[1]);
  };
  int ci = c_in;
  for (int l = 0; l <= layers; ++l) {
    const bool head = l == layers;
    const int fan = head ? ci : ci * 27;
    const int co = head ? c_out : width;
    const double sd = std::sqrt(2.0 / fan) * (head ? 0.5 : 1.0);
    for (int64_t k = 0; k < (int64_t)co * fan; ++k) w[c->w_off[l] + k] = (float)(sd * gauss());
    ci = width;
  }
  nh_status st = NH_OK;
  auto mk = [&](void **p, size_t bytes) {
    if (st == NH_OK && device_malloc(c->ctx, p, bytes) != NH_OK) {
      set_error("nh_cnn_create: out of device memory");
      st = NH_ERR_NOMEM;
    }
  };
  mk((void **)&c->master, c->n_params * sizeof(float));
  mk((void **)&c->bf, c->n_params * sizeof(uint16_t));
  mk((void **)&c->packed, c->n_packed * sizeof(uint16_t));
  mk((void **)&c->grad, c->n_params * sizeof(float));
  mk((void **)&c->m1, c->n_params * sizeof(float));
  mk((void **)&c->m2, c->n_params * sizeof(float));
  if (st == NH_OK) {
    hipError_t e = hipMemcpy(c->master, w.data(), c->n_params * sizeof(float),
                             hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(c->m1, 0, c->n_params * sizeof(float));
    if (e == hipSuccess) e = hipMemset(c->m2, 0, c->n_params * sizeof(float));
    if (e == hipSuccess) e = hipMemset(c->grad, 0, c->n_params * sizeof(float));
    if (e != hipSuccess) {
      nh_cnn_destroy(c);
      NH_CHECK(false, NH_ERR_HIP, "network set-up: %s", hipGetErrorString(e));
    }
    st = sync_bf16(c);
  }
  if (st != NH_OK) {
    nh_cnn_destroy(c);
    return st;
  }
  *out = c;
  return NH_OK;
}

void nh_cnn_destroy(nh_cnn *c) {
  if (!c) return;
  (void)hipSetDevice(c->device);
  for (float *q : c->act) (void)hipFree(q);
  void *ps[] = {c->master, c->bf, c->packed, c->grad, c->m1, c->m2, c->in, c->out,
                c->dpre[0], c->dpre[1], c->part};
  for (void *q : ps)
    if (q) (void)hipFree(q);
  delete c;
}

int64_t nh_cnn_num_params(const nh_cnn *c) { return c ? c->n_params : 0; }

nh_status nh_cnn_get_params(nh_cnn *c, float *host) {
  NH_CHECK(c && host, NH_ERR_ARG, "nh_cnn_get_params: bad arguments");
  NH_HIP(hipMemcpy(host, c->master, c->n_params * sizeof(float), hipMemcpyDeviceToHost));
  return NH_OK;
}

nh_status nh_cnn_set_params(nh_cnn *c, const float *host) {
  NH_CHECK(c && host, NH_ERR_ARG, "nh_cnn_set_params: bad arguments");
  NH_HIP(hipMemcpy(c->master, host, c->n_params * sizeof(float), hipMemcpyHostToDevice));
  NH_TRY(sync_bf16(c));
  NH_HIP(hipStreamSynchronize(c->ctx->stream));
  return NH_OK;
}

nh_status nh_cnn_forward(nh_cnn *c, const float *feat, int gx, int gy, int gz,
                         float *out) {
  NH_CHECK(c && feat && out && gx > 0 && gy > 0 && gz > 0, NH_ERR_ARG,
           "nh_cnn_forward: bad arguments");
  (void)hipGetLastError();
  const int64_t P = (int64_t)gx * gy * gz;
  NH_TRY(upload_feats(c, feat, P));
  NH_TRY(ensure_out(c, P));
  NH_TRY(forward(c, gx, gy, gz));
  NH_TRY(head(c, P));
  NH_HIP(hipMemcpyAsync(out, c->out, P * c->c_out * sizeof(float),
                        hipMemcpyDeviceToHost, c->ctx->stream));
  NH_HIP(hipStreamSynchronize(c->ctx->stream));
  return NH_OK;
}

nh_status nh_cnn_backward(nh_cnn *c, const float *feat, int gx, int gy, int gz,
                          const float *dout, float *grad) {
  NH_CHECK(c && feat && dout && grad, NH_ERR_ARG, "nh_cnn_backward: bad arguments");
  (void)hipGetLastError();
  const int64_t P = (int64_t)gx * gy * gz;
  NH_TRY(upload_feats(c, feat, P));
  NH_TRY(ensure_out(c, P));
  NH_TRY(forward(c, gx, gy, gz));
  float *d = c->out;  // holds dout
  NH_HIP(hipMemcpyAsync(d, dout, P * c->c_out * sizeof(float),
                        hipMemcpyHostToDevice, c->ctx->stream));
  NH_TRY(backward(c, gx, gy, gz, d));
  NH_HIP(hipMemcpyAsync(grad, c->grad, c->n_params * sizeof(float),
                        hipMemcpyDeviceToHost, c->ctx->stream));
  NH_HIP(hipStreamSynchronize(c->ctx->stream));
  return NH_OK;
}

nh_status nh_cnn_bind(nh_cnn *c, nh_context *ctx) {
  NH_CHECK(c && ctx, NH_ERR_ARG, "nh_cnn_bind: null argument");
  NH_CHECK(ctx->device == c->device, NH_ERR_ARG,
           "nh_cnn_bind: context on another device");
  // every network call synchronises its stream before returning, so no
  // work is pending on the previous context's stream
  c->ctx = ctx;
  return NH_OK;
}

nh_status nh_cnn_start_block(nh_cnn *c, const float *feat, int gx, int gy,
                             int gz, const int32_t *atom_point,
                             const int32_t *atom_slot, int n_states,
                             nh_cplx *block, int ptr_kind) {
  NH_CHECK(c && feat && atom_point && atom_slot && block && n_states > 0 &&
               n_states * 2 * c->ctx->nb * 2 <= c->c_out,
           NH_ERR_ARG, "nh_cnn_start_block: bad arguments");
  (void)hipGetLastError();
  nh_context *x = c->ctx;
  const int64_t P = (int64_t)gx * gy * gz, A = x->n_atoms;
  NH_TRY(upload_feats(c, feat, P));
  NH_TRY(forward(c, gx, gy, gz));
  std::vector<void *> mem;  // from the context's pool
  auto mk = [&](void **p, size_t bytes) -> nh_status {
    NH_TRY(pool_alloc(x, p, bytes));
    mem.push_back(*p);
    return NH_OK;
  };
  int32_t *dp = nullptr, *ds = nullptr;
  double2 *tmp = nullptr;
  nh_status st = mk((void **)&dp, A * sizeof(int32_t));
  if (st == NH_OK) st = mk((void **)&ds, A * sizeof(int32_t));
  if (st == NH_OK && ptr_kind == NH_PTR_HOST)
    st = mk((void **)&tmp, (size_t)n_states * x->n * sizeof(double2));
  hipError_t e = hipSuccess;
  if (st == NH_OK) {
    e = hipMemcpyAsync(dp, atom_point, A * sizeof(int32_t), hipMemcpyHostToDevice, x->stream);
    if (e == hipSuccess)
      e = hipMemcpyAsync(ds, atom_slot, A * sizeof(int32_t), hipMemcpyHostToDevice, x->stream);
    if (e == hipSuccess)
      st = head_map(c, n_states, dp, ds, tmp ? tmp : reinterpret_cast<double2 *>(block));
    if (st == NH_OK && e == hipSuccess && tmp)
      e = hipMemcpyAsync(block, tmp, (size_t)n_states * x->n * sizeof(double2),
                         hipMemcpyDeviceToHost, x->stream);
  }
  const hipError_t es = hipStreamSynchronize(x->stream);
  if (e == hipSuccess) e = es;
  for (void *q : mem) pool_release(x, q);
  NH_TRY(st);
  NH_CHECK(e == hipSuccess, NH_ERR_HIP, "nh_cnn_start_block: %s", hipGetErrorString(e));
  return NH_OK;
}

nh_status nh_cnn_train_step(nh_cnn *c, const float *feat, int gx, int gy, int gz,
                            const int32_t *atom_point, const int32_t *atom_slot,
                            const nh_cplx *targets, int n_targets,
                            const int32_t *cluster, int n_states,
                            const int32_t *out_cluster, double lr, double *loss,
                            float *grad) {
  NH_CHECK(c && feat && atom_point && atom_slot && targets && cluster &&
               out_cluster && loss && n_targets >= 1 && n_targets <= 16 &&
               n_states >= 1 && n_states <= 8 &&
               n_states * 2 * c->ctx->nb * 2 <= c->c_out,
           NH_ERR_ARG, "nh_cnn_train_step: bad arguments");
  (void)hipGetLastError();
  nh_context *x = c->ctx;
  const int64_t P = (int64_t)gx * gy * gz, A = x->n_atoms, N = x->n;
  const int ne = n_states;
  NH_TRY(upload_feats(c, feat, P));
  NH_TRY(forward(c, gx, gy, gz));
  // device scratch from the context's pool: point/slot maps, Y (prediction),
  // host targets' copy
  hipPointerAttribute_t pa{};
  const bool on_device = hipPointerGetAttributes(&pa, targets) == hipSuccess &&
                         pa.type == hipMemoryTypeDevice && pa.device == x->device &&
                         reinterpret_cast<uintptr_t>(targets) % sizeof(double2) == 0;
  (void)hipGetLastError();  // pageable host memory is not a registered pointer
  std::vector<void *> mem;
  auto mk = [&](void **p, size_t bytes) -> nh_status {
    NH_TRY(pool_alloc(x, p, bytes));
    mem.push_back(*p);
    return NH_OK;
  };
  auto cleanup = [&]() {
    for (void *q : mem) pool_release(x, q);
  };
  int32_t *dp, *ds;
  double2 *Y, *Vh = nullptr;
  double *part, *sum, *dM;
  nh_status st = ensure_out(c, P);
  if (st == NH_OK) st = mk((void **)&dp, A * sizeof(int32_t));
  if (st == NH_OK) st = mk((void **)&ds, A * sizeof(int32_t));
  if (st == NH_OK) st = mk((void **)&Y, (size_t)ne * N * sizeof(double2));
  if (st == NH_OK && !on_device) st = mk((void **)&Vh, (size_t)n_targets * N * sizeof(double2));
  if (st == NH_OK) st = mk((void **)&part, (size_t)512 * 2 * 64 * sizeof(double));
  if (st == NH_OK) st = mk((void **)&sum, 3 * 128 * sizeof(double));
  if (st == NH_OK) st = mk((void **)&dM, 17 * 8 * sizeof(double2));
  if (st != NH_OK) {
    cleanup();
    return st;
  }
  hipStream_t s = x->stream;
  // an asynchronous call that fails ends the step with the buffers released
#define TS_HIP(call)                                                            \
  do {                                                                          \
    const hipError_t e_ = (call);                                               \
    if (e_ != hipSuccess) {                                                     \
      cleanup();                                                                \
      NH_CHECK(false, NH_ERR_HIP, "train step: %s", hipGetErrorString(e_));    \
    }                                                                           \
  } while (0)
  TS_HIP(hipMemcpyAsync(dp, atom_point, A * sizeof(int32_t), hipMemcpyHostToDevice, s));
  TS_HIP(hipMemcpyAsync(ds, atom_slot, A * sizeof(int32_t), hipMemcpyHostToDevice, s));
  if (!on_device)
    TS_HIP(hipMemcpyAsync(Vh, targets, (size_t)n_targets * N * sizeof(double2),
                          hipMemcpyDefault, s));
  const double2 *V = on_device ? reinterpret_cast<const double2 *>(targets) : Vh;
  if (head_map(c, ne, dp, ds, Y) != NH_OK) {
    cleanup();
    return NH_ERR_HIP;
  }
  // C = V^H Y (up to 16 x 8, two halves of 8 rows) and the norms of Y
  std::vector<double> h(2 * 128, 0.0), hb(16);
  for (int half = 0; 8 * half < n_targets; ++half) {
    hipLaunchKernelGGL((k_gram<8>), dim3(512), dim3(256), 0, s, N,
                       std::min(8, n_targets - 8 * half), ne, V + (int64_t)half * 8 * N, N, Y,
                       N, part);
    hipLaunchKernelGGL(k_sum_cols, dim3(128), dim3(128), 0, s, 512, 128, part, sum + 128 * half);
    TS_HIP(hipMemcpyAsync(h.data() + half * 128, sum + 128 * half, 128 * sizeof(double),
                   hipMemcpyDeviceToHost, s));
  }
  hipLaunchKernelGGL((k_coldot<8>), dim3(512), dim3(256), 0, s, N, ne, Y, N, Y, N, part);
  hipLaunchKernelGGL(k_sum_cols, dim3(16), dim3(128), 0, s, 512, 16, part, sum + 256);
  TS_HIP(hipMemcpyAsync(hb.data(), sum + 256, 16 * sizeof(double), hipMemcpyDeviceToHost, s));
  hipError_t e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    cleanup();
    NH_CHECK(false, NH_ERR_HIP, "train step: %s", hipGetErrorString(e));
  }
  // C[f][e] = <v_f, y_e>
  auto C = [&](int f, int ee) {
    const double *q = h.data() + (f / 8) * 128 + 2 * ((f % 8) * 8 + ee);
    return cd(q[0], q[1]);
  };
  // L = mean_e (1 - a_e / b_e), a_e = sum over the targets of e's cluster of
  // |C[f][e]|^2, b_e = ||y_e||^2;  G_e = dL/dRe(y_e) + i dL/dIm(y_e)
  //     = 2 (-sum_f v_f C[f][e] / b_e + a_e y_e / b_e^2) / ne
  std::vector<cd> M(17 * 8, 0.0);  // M[f][e], then D[e]
  double L = 0.0;
  for (int ee = 0; ee < ne; ++ee) {
    const double b = std::max(hb[2 * ee], 1e-300);
    double a = 0.0;
    for (int f = 0; f < n_targets; ++f)
      if (cluster[f] == out_cluster[ee]) a += std::norm(C(f, ee));
    L += (1.0 - a / b) / ne;
    for (int f = 0; f < n_targets; ++f)
      if (cluster[f] == out_cluster[ee]) M[f * 8 + ee] = -2.0 * C(f, ee) / (b * ne);
    M[16 * 8 + ee] = 2.0 * a / (b * b * ne);
  }
  *loss = L;
  TS_HIP(hipMemcpyAsync(dM, M.data(), M.size() * sizeof(cd), hipMemcpyHostToDevice, s));
  // dL/d(out): real and imaginary parts of the complex gradient
  TS_HIP(hipMemsetAsync(c->out, 0, P * c->c_out * sizeof(float), s));
  hipLaunchKernelGGL(k_loss_grad, dim3(g1(A * x->nb)), dim3(256), 0, s, A, x->nb, n_targets,
                     ne, c->c_out, dp, ds, V, Y, N, reinterpret_cast<const double2 *>(dM),
                     c->out);
  TS_HIP(hipGetLastError());
#undef TS_HIP
  {
    nh_status bs = backward(c, gx, gy, gz, c->out);
    if (bs != NH_OK) {
      cleanup();
      return bs;
    }
    if (grad)
      e = hipMemcpyAsync(grad, c->grad, c->n_params * sizeof(float),
                         hipMemcpyDeviceToHost, s);
  }
  if (e == hipSuccess && lr > 0.0) {
    c->step += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - std::pow(b1, (float)c->step);
    const float c2 = 1.0f - std::pow(b2, (float)c->step);
    hipLaunchKernelGGL(k_adam, dim3(g1(c->n_params)), dim3(256), 0, s,
                       c->n_params, c->master, c->grad, c->m1, c->m2, (float)lr,
                       b1, b2, c1, c2, 1e-8f);
    sync_bf16(c);
  }
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  cleanup();
  NH_CHECK(e == hipSuccess, NH_ERR_HIP, "train step: %s", hipGetErrorString(e));
  return NH_OK;
}

}  // extern "C"
