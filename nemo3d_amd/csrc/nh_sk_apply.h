// Product of one bond's sp3d5s* block with one real component vector.
//
// The 10x10 block T (rows: anion orbitals, columns: cation orbitals; table
// in nh_sk.h) is applied without being formed.  With n the bond's direction,
// sd the five d functions along n, p and d the vector's p and d parts, M(d)
// the symmetric traceless matrix of the d part and w = M(d) n, its parts are
//   s, s*      numbers times xs, x_s*, n.p and sd.d;
//   p-p        ppp p + (pps - ppp) n (n.p);
//   p-d, d-p   padcp w + A n (sd.d), A = padcs - (2/sqrt 3) padcp, and its
//              transpose with pcdas, pcdap;
//   d-d        ddd d + B M^T(n w) + A' sd (sd.d), B = ddp - ddd,
//              A' = dds - ddd - (4/3) B
// (M^T(n w): the five components of the symmetric product of n and w).
// The identities behind these forms hold for the true sqrt 3; the table has
// the reference's literal s (6.5e-13 off), in the first four d functions and
// in M's z2 part.  What that changes is linear in z = n^2 - (l^2 + m^2)/2, the
// fifth d function: in FP64 the z2 column of p-d has (2 s / 3) in the place of
// (2 / s) and the z2 row and column of A' sd sd^T the factor s^2 / 3, added as
// kz (relative to the table in 80 bits, directions 0.002 / 0.01 / 0.03 off
// (111): 1.4e-15 / 7.0e-15 / 2.1e-14 without, 2.0e-16 with them; the table in
// FP64 1.5e-16).
// That is 93 operations per vector and about 45 per bond for
// the scaled vectors, against 100 and about 250 for forming T.
//
// Every matrix element is a sum of products of two numbers that are
// precomputed per bond, added in the same order in both orientations (the
// anion row applies T, the cation row its transpose: what one projects on,
// the other expands along), so the two rows of a bond are exact transposes
// of each other in floating point and H stays exactly Hermitian.  All
// multiply-adds are explicit: every kernel that applies a bond rounds alike.
#pragma once

#include "nh_sk.h"

namespace nh {

// The 24 numbers of a bond record.  Pairs whose members swap in the
// transposed product are neighbours (one 16-byte load in FP64).
enum : int {
  K_L = 0, K_M = 1, K_N = 2, K_DDD = 3,
  K_SSS = 4, K_STSTS = 5, K_STASS = 6, K_SASTS = 7,
  K_SAPC = 8, K_SCPA = 9, K_STAPC = 10, K_STCPA = 11,
  K_SADC = 12, K_SCDA = 13, K_STADC = 14, K_STCDA = 15,
  K_PADP = 16, K_PCDP = 17, K_APD = 18, K_ADP = 19,
  K_PPP = 20, K_PPC = 21, K_DB = 22, K_DA = 23
};

constexpr double kRecC2 = 2.0 / kSqrt3Ref, kRecC3 = 3.0 / (kSqrt3Ref * kSqrt3Ref);
// Record of the direction (l, m, n) and the 21 integrals v (parameters
// 10..30; the signs of the integrals with the lower angular momentum on the
// cation as in sk_table).
template <typename R>
__host__ __device__ __forceinline__ void sk_record(R l, R m, R n, const R *v, R *k) {
  constexpr R c2 = R(kRecC2), c3 = R(kRecC3);
  k[K_L] = l;
  k[K_M] = m;
  k[K_N] = n;
  k[K_SSS] = v[0];
  k[K_STSTS] = v[1];
  k[K_STASS] = v[2];
  k[K_SASTS] = v[3];
  k[K_SAPC] = v[4];
  k[K_SCPA] = -v[5];
  k[K_STAPC] = v[6];
  k[K_STCPA] = -v[7];
  k[K_SADC] = v[8];
  k[K_SCDA] = v[9];
  k[K_STADC] = v[10];
  k[K_STCDA] = v[11];
  k[K_PPP] = v[13];
  k[K_PPC] = v[12] - v[13];
  k[K_PADP] = v[16];
  k[K_PCDP] = -v[17];
  k[K_APD] = v[14] - c2 * v[16];
  k[K_ADP] = c2 * v[17] - v[15];
  k[K_DDD] = v[20];
  k[K_DB] = v[19] - v[20];
  k[K_DA] = c3 * ((v[18] - v[20]) - R(4.0 / 3.0) * (v[19] - v[20]));
}

// The FP32 record of an FP64 one: the combinations take up the rounding of the
// integrals in them, so that what T has of the others (dds = K_DDD + 4/3 K_DB +
// K_DA / c3, pps = K_PPP + K_PPC, ..) is rounded once
__host__ __device__ __forceinline__ void sk_round(const double (&d)[24], float (&k)[24]) {
#pragma unroll
  for (int i = 0; i < 24; ++i) k[i] = (float)d[i];
  auto lost = [&](int i) { return d[i] - (double)k[i]; };
  k[K_PPC] = (float)(d[K_PPC] + lost(K_PPP));
  k[K_APD] = (float)(d[K_APD] + kRecC2 * lost(K_PADP));
  k[K_ADP] = (float)(d[K_ADP] + kRecC2 * lost(K_PCDP));
  k[K_DB] = (float)(d[K_DB] + lost(K_DDD));
  k[K_DA] = (float)(d[K_DA] + kRecC3 * (lost(K_DDD) + (4.0 / 3.0) * lost(K_DB)));
}

__host__ __device__ __forceinline__ double sk_fma(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}
__host__ __device__ __forceinline__ float sk_fma(float a, float b, float c) {
  return __builtin_fmaf(a, b, c);
}

// y += T x (CATION = false: x on the cation, y on the anion) or y += T^t x
// (CATION = true: x on the anion, y on the cation); k: the bond's record.
template <bool CATION, typename R>
__host__ __device__ __forceinline__ void sk_apply(const R *k, const R (&x)[10], R (&y)[10]) {
#pragma clang fp contract(off)
  const R l = k[K_L], m = k[K_M], n = k[K_N];
  constexpr R s3 = R(kSqrt3Ref), kp = R(kSqrt3Ref / 3.0);
  // members of the swapping pairs: xy = element from y's role to x's role
  const R ss_a = CATION ? k[K_SASTS] : k[K_STASS];  // y_s* from x_s
  const R ss_b = CATION ? k[K_STASS] : k[K_SASTS];  // y_s from x_s*
  const R sp = CATION ? k[K_SCPA] : k[K_SAPC], ps = CATION ? k[K_SAPC] : k[K_SCPA];
  const R tp = CATION ? k[K_STCPA] : k[K_STAPC], pt = CATION ? k[K_STAPC] : k[K_STCPA];
  const R sd_ = CATION ? k[K_SCDA] : k[K_SADC], ds = CATION ? k[K_SADC] : k[K_SCDA];
  const R td = CATION ? k[K_STCDA] : k[K_STADC], dt = CATION ? k[K_STADC] : k[K_STCDA];
  const R pdp = CATION ? k[K_PCDP] : k[K_PADP], dpp = CATION ? k[K_PADP] : k[K_PCDP];
  const R apd = CATION ? k[K_ADP] : k[K_APD], adp = CATION ? k[K_APD] : k[K_ADP];
  const R ppc = k[K_PPC], ppp = k[K_PPP], ddd = k[K_DDD], db = k[K_DB], da = k[K_DA];
  const R *p = x + 2, *d = x + 5;
  // sd and the projections on it and on n.  FP32: sd's five functions are
  // formed and projected on in FP64 and rounded once (as products of rounded
  // products their errors, alike in all three of (111), made up most of the
  // product's error)
  R g[5], t;
  if constexpr (sizeof(R) == 8) {
    const R l2 = l * l, m2 = m * m;
    g[0] = s3 * (m * l), g[1] = s3 * (m * n), g[2] = s3 * (n * l);
    g[3] = (R(0.5) * s3) * (l2 - m2), g[4] = n * n - R(0.5) * (l2 + m2);
    t = g[0] * d[0];
#pragma unroll
    for (int c = 1; c < 5; ++c) t = sk_fma(g[c], d[c], t);
  } else {
    const double dl = l, dm = m, dn = n, m2 = dm * dm;
    const double sl = kSqrt3Ref * dl, sn = kSqrt3Ref * dn;
    const double e[5] = {sl * dm, sn * dm, sl * dn,
                         (0.5 * kSqrt3Ref) * sk_fma(dl, dl, -m2),
                         sk_fma(dn, dn, -0.5 * sk_fma(dl, dl, m2))};
    double td_ = e[0] * (double)d[0];
#pragma unroll
    for (int c = 1; c < 5; ++c) td_ = sk_fma(e[c], (double)d[c], td_);
    t = R(td_);
#pragma unroll
    for (int c = 0; c < 5; ++c) g[c] = R(e[c]);
  }
  const R s = sk_fma(n, p[2], sk_fma(m, p[1], l * p[0]));
  y[0] = sk_fma(td, t, sk_fma(tp, s, sk_fma(ss_a, x[1], sk_fma(k[K_STSTS], x[0], y[0]))));
  y[1] = sk_fma(sd_, t, sk_fma(sp, s, sk_fma(ss_b, x[0], sk_fma(k[K_SSS], x[1], y[1]))));
  // w = M(d) n; the z2 part enters as (-1, -1, 2) kp
  const R kl = kp * l, km = kp * m, kn = (kp * n) * R(2);
  const R wx = sk_fma(n, d[2], sk_fma(m, d[0], sk_fma(-kl, d[4], l * d[3])));
  const R wy = sk_fma(n, d[1], sk_fma(l, d[0], sk_fma(-km, d[4], -(m * d[3]))));
  const R wz = sk_fma(m, d[1], sk_fma(l, d[2], kn * d[4]));
  // the literal's part (none in FP32): p-d z2 column, d-d z2 row and column
  constexpr bool kExact = sizeof(R) == 8;
  constexpr R s2m3 = R(kSqrt3Ref * kSqrt3Ref - 3.0);
  const R kz = kExact ? (-(R(2) / R(3)) * s2m3 / s3) * g[4] : R(0);
  const R e4 = kExact ? ((s2m3 / R(3)) * g[4]) * da : R(0);
  // p rows: ppp p + pdp w, then along n, along A n, then the p-p projection
  R cp = sk_fma(ps, x[1], pt * x[0]);
  if constexpr (kExact) cp = sk_fma(kz * pdp, d[4], cp);
  const R al = apd * l, am = apd * m, an = apd * n;
  const R cl = ppc * l, cm = ppc * m, cn = ppc * n;
  R sc;
  if constexpr (CATION) sc = sk_fma(cn, p[2], sk_fma(cm, p[1], cl * p[0]));
  y[2] = sk_fma(al, t, sk_fma(l, cp, sk_fma(pdp, wx, sk_fma(ppp, p[0], y[2]))));
  y[3] = sk_fma(am, t, sk_fma(m, cp, sk_fma(pdp, wy, sk_fma(ppp, p[1], y[3]))));
  y[4] = sk_fma(an, t, sk_fma(n, cp, sk_fma(pdp, wz, sk_fma(ppp, p[2], y[4]))));
  if constexpr (CATION) {
    y[2] = sk_fma(l, sc, y[2]);
    y[3] = sk_fma(m, sc, y[3]);
    y[4] = sk_fma(n, sc, y[4]);
  } else {
    y[2] = sk_fma(cl, s, y[2]);
    y[3] = sk_fma(cm, s, y[3]);
    y[4] = sk_fma(cn, s, y[4]);
  }
  // d rows: ddd d, then the symmetric products, then along sd
  R y5 = sk_fma(ddd, d[0], y[5]), y6 = sk_fma(ddd, d[1], y[6]), y7 = sk_fma(ddd, d[2], y[7]),
    y8 = sk_fma(ddd, d[3], y[8]);
  // z2-z2: the table's element has no sqrt(3); the reference's literal one
  // (1.2e-12 off) enters here through kp^2, which this takes back
  R ddd4 = ddd;
  if constexpr (sizeof(R) == 8) {
    constexpr R e = R(1.0 / 3.0 - (kSqrt3Ref / 3.0) * (kSqrt3Ref / 3.0));
    ddd4 = sk_fma(sk_fma(R(3) * e, n * n, e), db, ddd);
  }
  R y9 = sk_fma(ddd4, d[4], y[9]);
  const R bl = db * l, bm = db * m, bn = db * n;
  const R kbl = db * kl, kbm = db * km, kbn = db * kn;
  if constexpr (CATION) {
    // w along B n, expanded with the p part along n
    const R vx = sk_fma(bn, d[2], sk_fma(bm, d[0], sk_fma(-kbl, d[4], bl * d[3])));
    const R vy = sk_fma(bn, d[1], sk_fma(bl, d[0], sk_fma(-kbm, d[4], -(bm * d[3]))));
    const R vz = sk_fma(bm, d[1], sk_fma(bl, d[2], kbn * d[4]));
    const R hx = sk_fma(dpp, p[0], vx), hy = sk_fma(dpp, p[1], vy), hz = sk_fma(dpp, p[2], vz);
    y5 = sk_fma(l, hy, sk_fma(m, hx, y5));
    y6 = sk_fma(n, hy, sk_fma(m, hz, y6));
    y7 = sk_fma(n, hx, sk_fma(l, hz, y7));
    y8 = sk_fma(-m, hy, sk_fma(l, hx, y8));
    y9 = sk_fma(-km, hy, sk_fma(-kl, hx, sk_fma(kn, hz, y9)));
  } else {
    const R hx = dpp * p[0], hy = dpp * p[1], hz = dpp * p[2];
    y5 = sk_fma(bl, wy, sk_fma(bm, wx, sk_fma(l, hy, sk_fma(m, hx, y5))));
    y6 = sk_fma(bn, wy, sk_fma(bm, wz, sk_fma(n, hy, sk_fma(m, hz, y6))));
    y7 = sk_fma(bn, wx, sk_fma(bl, wz, sk_fma(n, hx, sk_fma(l, hz, y7))));
    y8 = sk_fma(-bm, wy, sk_fma(bl, wx, sk_fma(-m, hy, sk_fma(l, hx, y8))));
    y9 = sk_fma(-km, hy, sk_fma(-kl, hx, sk_fma(kn, hz, y9)));
    y9 = sk_fma(-kbm, wy, sk_fma(-kbl, wx, sk_fma(kbn, wz, y9)));
  }
  // sd (xs, x_s* parts, A n.p), A' sd (sd.d)
  const R sq = sk_fma(adp * n, p[2], sk_fma(adp * m, p[1], (adp * l) * p[0]));
  const R cs = sk_fma(ds, x[1], sk_fma(dt, x[0], sq));
  R ta;
  if constexpr (CATION) {
    ta = (da * g[0]) * d[0];
#pragma unroll
    for (int c = 1; c < 5; ++c) ta = sk_fma(da * g[c], d[c], ta);
  } else {
    ta = t;
  }
  const R cs4 = kExact ? sk_fma(e4, d[4], cs) : cs;
  if constexpr (kExact) y9 = sk_fma(kz * dpp, s, y9);
  const R yd[4] = {y5, y6, y7, y8};
#pragma unroll
  for (int c = 0; c < 4; ++c)
    y[5 + c] = sk_fma(CATION ? g[c] : da * g[c], ta, sk_fma(g[c], cs4, yd[c]));
  y9 = sk_fma(g[4], cs, y9);
  if constexpr (kExact) y9 = sk_fma(e4, t, y9);
  y[9] = sk_fma(CATION ? g[4] : da * g[4], ta, y9);
}

}  // namespace nh
