// The bond products of nh_sk_apply.h and the table they stand for, on the host.
#include <cmath>

#include "../../nemo3d_amd/csrc/nh_sk_apply.h"

using namespace nh;

namespace {
template <typename R>
void apply(int cation, const R *k, const R *x, R *y) {
  R xx[10], yy[10];
  for (int i = 0; i < 10; ++i) xx[i] = x[i], yy[i] = 0;
  if (cation) sk_apply<true, R>(k, xx, yy);
  else sk_apply<false, R>(k, xx, yy);
  for (int i = 0; i < 10; ++i) y[i] = yy[i];
}
// y = T x or T^t x, term after term
template <typename R>
void table(int cation, const double *dir, const double *v, const double *x, double *y) {
  R vr[21], T[100];
  for (int i = 0; i < 21; ++i) vr[i] = (R)v[i];
  sk_table<R>((R)dir[0], (R)dir[1], (R)dir[2], vr, T);
  for (int o = 0; o < 10; ++o) {
    R s = 0;
    for (int c = 0; c < 10; ++c) s = std::fma(T[cation ? c * 10 + o : o * 10 + c], (R)x[c], s);
    y[o] = (double)s;
  }
}
}  // namespace

extern "C" {
// kind 0: FP64 record and product, 1: the FP32 ones; 2, 3, 4: the table in
// 80 bits (to FP64), FP64, FP32
void sk_product(int kind, int cation, const double *dir, const double *v, const double *x,
                double *y) {
  double k[24];
  sk_record(dir[0], dir[1], dir[2], v, k);
  if (kind == 0) {
    apply(cation, k, x, y);
  } else if (kind == 1) {
    float kf[24], xf[10], yf[10];
    sk_round(k, kf);
    for (int i = 0; i < 10; ++i) xf[i] = (float)x[i];
    apply(cation, kf, xf, yf);
    for (int i = 0; i < 10; ++i) y[i] = yf[i];
  } else if (kind == 2) {
    table<long double>(cation, dir, v, x, y);
  } else if (kind == 3) {
    table<double>(cation, dir, v, x, y);
  } else {
    table<float>(cation, dir, v, x, y);
  }
}
}
