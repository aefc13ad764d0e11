// weno.h — WENO5-JS face reconstructions of the level-set solvers and their
// reverse-mode derivatives (the adjoint advection).  Device code for gfx950.
#pragma once

#include <hip/hip_runtime.h>

namespace fcfd {

// WENO5-JS face values (level_set_rk3_solver.f90:162-216): with the five
// samples g0..g4, differences e_m = g_{m+1} - g_m and smoothness indicators
//   beta_k = 13 t_k^2 + 3 s_k^2,  t_k = e_{k+1} - e_k (k = 0, 1, 2),
//   s = (3 e1 - e0, e1 + e2, 3 e2 - e3),
// the left-biased value is g2 + (sum_k a_k c_k) / (6 sum_k a_k) with
//   c = (5 e1 - 2 e0, e1 + 2 e2, 4 e2 - e3)  (the candidate values less g2,
// times 6) and a_k = d_k / (EPS + beta_k)^2, d = (1, 6, 3).  A common factor
// of the a_k cancels, so beta and EPS are taken divided by 3, and in FP64
// every a_k is multiplied by q1 q2 q3 (q_k = ((EPS + beta_k) / 3)^2), which
// needs one reciprocal instead of three and a sum's.  With |phi| and |u| of
// O(1) the products stay far inside the FP64 range (q >= 1e-27, a product of
// two >= 1e-54).  The right-biased value is the mirror image: the left one of
// the samples in reverse order.
//
// Written in differences a value takes 47 FP64 operations, with explicit fma
// so that it does not depend on how the caller is compiled; the weights,
// normalised, times the candidate stencils took about 70.

// 1 / x to about an ulp: the hardware's estimate and two Newton steps.  The
// reciprocal only scales the WENO correction of g2.
__device__ __forceinline__ double weno_rcp(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(r, fma(-x, r, 1.0), r);
}

// a_k (times q1 q2 q3) of the samples' differences
__device__ __forceinline__ void weno_terms(double e0, double e1, double e2, double e3, double EPS, double &a1,
                                           double &a2, double &a3) {
#pragma clang fp contract(off)
    const double eps3 = EPS * (1.0 / 3.0), t1 = e1 - e0, t2 = e2 - e1, t3 = e3 - e2;
    const double s1 = fma(3.0, e1, -e0), s2 = e1 + e2, s3 = fma(3.0, e2, -e3);
    const double b1 = fma(13.0 / 3.0, t1 * t1, fma(s1, s1, eps3));
    const double b2 = fma(13.0 / 3.0, t2 * t2, fma(s2, s2, eps3));
    const double b3 = fma(13.0 / 3.0, t3 * t3, fma(s3, s3, eps3));
    const double q1 = b1 * b1, q2 = b2 * b2, q3 = b3 * b3;
    a1 = q2 * q3;
    a2 = 6.0 * (q1 * q3);
    a3 = 3.0 * (q1 * q2);
}

__device__ __forceinline__ double weno_left(double g0, double g1, double g2, double g3, double g4, double EPS) {
#pragma clang fp contract(off)
    const double e0 = g1 - g0, e1 = g2 - g1, e2 = g3 - g2, e3 = g4 - g3;
    double a1, a2, a3;
    weno_terms(e0, e1, e2, e3, EPS, a1, a2, a3);
    const double c1 = fma(5.0, e1, -2.0 * e0), c2 = fma(2.0, e2, e1), c3 = fma(4.0, e2, -e3);
    const double num = fma(a3, c3, fma(a2, c2, a1 * c1));
    return fma(num, weno_rcp(6.0 * (a1 + (a2 + a3))), g2);
}

// The same value as the weighted sum of the samples, in the reference's
// order.  For the MPLS_RisingBubble reinitialisation: its mass corrections
// divide by small mass differences and amplify a change of rounding about
// 1e5 times, so its values keep the rounding of the reference's sum (seven
// operations more).
__device__ __forceinline__ double weno_left_sum(double g0, double g1, double g2, double g3, double g4, double EPS) {
    double a1, a2, a3;
    weno_terms(g1 - g0, g2 - g1, g3 - g2, g4 - g3, EPS, a1, a2, a3);
    const double r = weno_rcp(a1 + (a2 + a3)), w1 = a1 * r, w2 = a2 * r, w3 = a3 * r;
    constexpr double r6 = 1.0 / 6.0;
    return w1 * (1.0 / 3.0) * g0 - (7.0 * w1 + w2) * r6 * g1 + (11.0 * w1 + 5.0 * w2 + 2.0 * w3) * r6 * g2 +
           (2.0 * w2 + 5.0 * w3) * r6 * g3 - w3 * r6 * g4;
}

// right-biased face value from f(i-1..i+3)
__device__ __forceinline__ double weno_right(double f0, double f1, double f2, double f3, double f4, double EPS) {
    return weno_left(f4, f3, f2, f1, f0, EPS);
}

// FP32: a_k = d_k / q_k, because the products of the FP64 form underflow
// where the flux is locally flat (beta = 0 on all three stencils: q = 1e-27).
__device__ __forceinline__ float weno_rcp(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    return fmaf(r, fmaf(-x, r, 1.0f), r);
}

__device__ __forceinline__ float weno_left(float g0, float g1, float g2, float g3, float g4, float EPS) {
#pragma clang fp contract(off)
    const float e0 = g1 - g0, e1 = g2 - g1, e2 = g3 - g2, e3 = g4 - g3, eps3 = EPS * (1.0f / 3.0f);
    const float t1 = e1 - e0, t2 = e2 - e1, t3 = e3 - e2;
    const float s1 = fmaf(3.0f, e1, -e0), s2 = e1 + e2, s3 = fmaf(3.0f, e2, -e3);
    const float b1 = fmaf(13.0f / 3.0f, t1 * t1, fmaf(s1, s1, eps3));
    const float b2 = fmaf(13.0f / 3.0f, t2 * t2, fmaf(s2, s2, eps3));
    const float b3 = fmaf(13.0f / 3.0f, t3 * t3, fmaf(s3, s3, eps3));
    const float r1 = weno_rcp(b1), r2 = weno_rcp(b2), r3 = weno_rcp(b3);
    const float a1 = r1 * r1, a2 = 6.0f * (r2 * r2), a3 = 3.0f * (r3 * r3);
    const float c1 = fmaf(5.0f, e1, -2.0f * e0), c2 = fmaf(2.0f, e2, e1), c3 = fmaf(4.0f, e2, -e3);
    const float num = fmaf(a3, c3, fmaf(a2, c2, a1 * c1));
    return fmaf(num, weno_rcp(6.0f * (a1 + (a2 + a3))), g2);
}

__device__ __forceinline__ float weno_right(float f0, float f1, float f2, float f3, float f4, float EPS) {
    return weno_left(f4, f3, f2, f1, f0, EPS);
}

// ---------------------------------------------------------------- adjoints
// The weights' parts that the reverse mode needs, by precision (see above):
// a_k and 1 / b_k of b_k = (EPS + beta_k) / 3.  FP64 takes the three
// reciprocals from that of the product (b >= 3e-14, a product >= 3e-41).
__device__ __forceinline__ void weno_adj_weights(const double (&b)[3], double (&a)[3], double (&ib)[3]) {
    const double q0 = b[0] * b[0], q1 = b[1] * b[1], q2 = b[2] * b[2];
    a[0] = q1 * q2;
    a[1] = 6.0 * (q0 * q2);
    a[2] = 3.0 * (q0 * q1);
    const double b01 = b[0] * b[1], r = weno_rcp(b01 * b[2]);
    ib[0] = b[1] * b[2] * r;
    ib[1] = b[0] * b[2] * r;
    ib[2] = b01 * r;
}
__device__ __forceinline__ void weno_adj_weights(const float (&b)[3], float (&a)[3], float (&ib)[3]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) ib[k] = weno_rcp(b[k]);
    a[0] = ib[0] * ib[0];
    a[1] = 6.0f * (ib[1] * ib[1]);
    a[2] = 3.0f * (ib[2] * ib[2]);
}
__device__ __forceinline__ double weno_fma(double x, double y, double z) { return fma(x, y, z); }
__device__ __forceinline__ float weno_fma(float x, float y, float z) { return fmaf(x, y, z); }

// d(weno_left)/dg_m times vb, into gb[0..4], for the forward's form
// V = g2 + N r, N = sum a_k c_k, r = 1 / (6 sum a_k): dV/dc_k = a_k r and,
// with da_k/db_k = -2 a_k / b_k, dV/db_k = -2 a_k r (c_k - 6 N r) / b_k;
// then back through t, s and c to the differences e and the samples.  The
// weights a_k r are formed before vb comes in: where the samples are flat
// (b = EPS / 3) r is 2e-29 in FP32, and vb r would lose the bits of a vb
// below 6e-10 and vanish below 1e-17.  T =
// double or float (the weights of that precision's forward).  About 105
// operations, where differentiating the normalised weights took about 160.
template <typename T>
__device__ __forceinline__ void weno_left_adj(const T *g, T EPS, T vb, T *gb) {
    const T e0 = g[1] - g[0], e1 = g[2] - g[1], e2 = g[3] - g[2], e3 = g[4] - g[3];
    const T eps3 = EPS * (T)(1.0 / 3.0), c133 = (T)(13.0 / 3.0), two = 2, three = 3;
    const T t[3] = {e1 - e0, e2 - e1, e3 - e2};
    const T s[3] = {weno_fma(three, e1, -e0), e1 + e2, weno_fma(three, e2, -e3)};
    const T c[3] = {weno_fma((T)5, e1, -two * e0), weno_fma(two, e2, e1), weno_fma((T)4, e2, -e3)};
    T b[3], a[3], ib[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) b[k] = weno_fma(c133, t[k] * t[k], weno_fma(s[k], s[k], eps3));
    weno_adj_weights(b, a, ib);
    const T r = weno_rcp((T)6 * (a[0] + (a[1] + a[2])));
    const T m = (T)-6 * (weno_fma(a[2], c[2], weno_fma(a[1], c[1], a[0] * c[0])) * r);   // -6 N r
    T cb[3], tb[3], sb[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        cb[k] = (a[k] * r) * vb;
        const T bb = (-two * cb[k]) * ((c[k] + m) * ib[k]);
        tb[k] = ((two * c133) * bb) * t[k];
        sb[k] = (two * bb) * s[k];
    }
    const T eb0 = weno_fma(-two, cb[0], -(tb[0] + sb[0]));
    const T eb1 = weno_fma((T)5, cb[0], cb[1]) + weno_fma(three, sb[0], sb[1]) + (tb[0] - tb[1]);
    const T eb2 = weno_fma(two, cb[1], (T)4 * cb[2]) + weno_fma(three, sb[2], sb[1]) + (tb[1] - tb[2]);
    const T eb3 = (tb[2] - sb[2]) - cb[2];
    gb[0] = -eb0;
    gb[1] = eb0 - eb1;
    gb[2] = vb + (eb1 - eb2);
    gb[3] = eb2 - eb3;
    gb[4] = eb3;
}

// d(weno_right)/df_m times vb, into fb[0..4]: the mirror image
template <typename T>
__device__ __forceinline__ void weno_right_adj(const T *f, T EPS, T vb, T *fb) {
    const T g[5] = {f[4], f[3], f[2], f[1], f[0]};
    T gb[5];
    weno_left_adj<T>(g, EPS, vb, gb);
#pragma unroll
    for (int m = 0; m < 5; ++m) fb[m] = gb[4 - m];
}

}  // namespace fcfd
