// acx_cweno_core.h -- the CWENO4 reconstruction of one cell and component,
// restricted to what face averages need (shared by the stage kernel, the
// label kernel of the learned indicator and the ensemble kernel).
//
// 3d/weno4/plane_wave/reconstruction.c:38-259: R4 derivatives (:90-108),
// IS_R4 (:110-116), seven R3 stencils (:121-203), weights with p = 4 and
// eps = 1e-12 (:118,205-218), CWENO combination (:223-257).
#pragma once
#include "acx_device.h"
#include "acx_internal.h"

namespace acx {

template <typename T> struct Axis3 { T c1[3], c2[3], c3[3]; };

// 1/t in FP64: hardware reciprocal estimate refined by one Newton step.
// Measured on gfx950 over 2^20 seeded t in [1e-50, 2e50]: the estimate alone
// has |r t - 1| up to 4.6e-8 (2^-24.4), one step brings it to 2.2e-15
// (2^-48.7), which puts the weights within about 20 units in the last place.
// Enough for what cweno_weights serves in FP64, the training labels, which
// compare the weights' deviation with a threshold; the stage kernels take
// rcp64_full.
__device__ __forceinline__ double rcp64(double t)
{
    double r = __builtin_amdgcn_rcp(t);
    const double e = fma(-t, r, 1.0);
    return fma(r, e, r);
}

// 1/t in FP64 to the last place or so: the estimate r = (1 - e)/t with
// |e| <= 2^-24.4 refined by r (1 + e + e^2), which leaves e^3.
__device__ __forceinline__ double rcp64_full(double t)
{
    const double r = __builtin_amdgcn_rcp(t);
    const double e = fma(-t, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

template <typename T>
__device__ __forceinline__ T pos_pow4_inv(T g, T t)
{
    T t2 = t * t;
    return g * rcp64(t2 * t2);
}

// Linear 4th-order polynomial along each axis (reconstruction.c:90-101)
template <typename T>
__device__ __forceinline__ void axis_linear(T m2, T m1, T u0, T p1, T p2, T &c1, T &c2, T &c3)
{
    c1 = T(1.0 / 120.0) * (T(11) * m2 - T(82) * m1 + T(82) * p1 - T(11) * p2);
    c2 = T(0.5) * (m1 - T(2) * u0 + p1);
    c3 = T(1.0 / 12.0) * (-m2 + T(2) * (m1 - p1) + p2);
}

// Smoothness indicators and normalised nonlinear weights of one cell and
// component; get(q) returns stencil slot q (0: centre; 1-4, 5-8, 9-12: the
// x, y, z arms m2 m1 p1 p2; 13-16 xy, 17-20 yz, 21-24 zx diagonals; 25-32
// corners).  wt = wt_ratio (reconstruction.c:236), w3[7] the R3 weights.
// The indicators are accumulated in three groups (axis arms, edge diagonals,
// corners); with LDS-backed values the memory clobbers between the groups keep
// only one group live at a time.
template <typename T, typename Get>
__device__ __forceinline__ void cweno_weights(Get get, const CwArgs &p, T &wt, T (&w3)[7])
{
    const T k13 = T(13.0 / 3.0), k7 = T(7.0 / 6.0);
    T is4, is3[7], cx, cy, cz;
    {   // axis arms: R4 x/y/z derivatives and the sided R3 stencils (reconstruction.c:90-101,121-203)
        const T u0 = get(0);
        const T xm2 = get(1), xm1 = get(2), xp1 = get(3), xp2 = get(4);
        const T ym2 = get(5), ym1 = get(6), yp1 = get(7), yp2 = get(8);
        const T zm2 = get(9), zm1 = get(10), zp1 = get(11), zp2 = get(12);
        T ux, uy, uz, uxx, uyy, uzz, uxxx, uyyy, uzzz;
        axis_linear(xm2, xm1, u0, xp1, xp2, ux, uxx, uxxx);
        axis_linear(ym2, ym1, u0, yp1, yp2, uy, uyy, uyyy);
        axis_linear(zm2, zm1, u0, zp1, zp2, uz, uzz, uzzz);
        is4 = ux * ux + uy * uy + uz * uz + k13 * (uxx * uxx + uyy * uyy + uzz * uzz) +
              T(0.2) * (ux * uxxx + uy * uyyy + uz * uzzz) + T(39.06) * (uxxx * uxxx + uyyy * uyyy + uzzz * uzzz);
        cx = T(0.5) * (xp1 - xm1);
        cy = T(0.5) * (yp1 - ym1);
        cz = T(0.5) * (zp1 - zm1);
        const T dx1 = T(-1.5) * u0 + T(2) * xp1 - T(0.5) * xp2, dxx1 = T(0.5) * (u0 - T(2) * xp1 + xp2);
        const T dx2 = T(-2) * xm1 + T(0.5) * xm2 + T(1.5) * u0, dxx2 = T(0.5) * (xm2 - T(2) * xm1 + u0);
        const T dy3 = T(-1.5) * u0 + T(2) * yp1 - T(0.5) * yp2, dyy3 = T(0.5) * (u0 - T(2) * yp1 + yp2);
        const T dy4 = T(-2) * ym1 + T(0.5) * ym2 + T(1.5) * u0, dyy4 = T(0.5) * (ym2 - T(2) * ym1 + u0);
        const T dz5 = T(-1.5) * u0 + T(2) * zp1 - T(0.5) * zp2, dzz5 = T(0.5) * (u0 - T(2) * zp1 + zp2);
        const T dz6 = T(-2) * zm1 + T(0.5) * zm2 + T(1.5) * u0, dzz6 = T(0.5) * (zm2 - T(2) * zm1 + u0);
        // central R3 shares the R4 second derivatives
        const T Cx = cx * cx + k13 * uxx * uxx, Cy = cy * cy + k13 * uyy * uyy, Cz = cz * cz + k13 * uzz * uzz;
        is3[0] = Cx + Cy + Cz;
        is3[1] = (dx1 * dx1 + k13 * dxx1 * dxx1) + Cy + Cz;
        is3[2] = (dx2 * dx2 + k13 * dxx2 * dxx2) + Cy + Cz;
        is3[3] = Cx + (dy3 * dy3 + k13 * dyy3 * dyy3) + Cz;
        is3[4] = Cx + (dy4 * dy4 + k13 * dyy4 * dyy4) + Cz;
        is3[5] = Cx + Cy + (dz5 * dz5 + k13 * dzz5 * dzz5);
        is3[6] = Cx + Cy + (dz6 * dz6 + k13 * dzz6 * dzz6);
    }
    asm volatile("" ::: "memory");
    {   // edge diagonals: mixed derivatives (reconstruction.c:102-107, sided R3 cross terms)
        const T ym1 = get(6), yp1 = get(7), zm1 = get(10), zp1 = get(11), xm1 = get(2), xp1 = get(3);
        const T xy_pp = get(13), xy_pm = get(14), xy_mp = get(15), xy_mm = get(16);
        const T yz_pp = get(17), yz_pm = get(18), yz_mp = get(19), yz_mm = get(20);
        const T zx_pp = get(21), zx_pm = get(22), zx_mp = get(23), zx_mm = get(24);
        const T uxy = T(0.25) * (xy_mm - xy_mp - xy_pm + xy_pp);
        const T uyz = T(0.25) * (yz_mm - yz_mp - yz_pm + yz_pp);
        const T uxz = T(0.25) * (zx_mm - zx_mp - zx_pm + zx_pp);
        const T uxxy = T(0.25) * (-xy_mm + xy_mp - xy_pm + xy_pp) + T(0.5) * (ym1 - yp1);
        const T uxyy = T(0.5) * (xm1 - xp1) + T(0.25) * (xy_pp - xy_mm - xy_mp + xy_pm);
        const T uyyz = T(0.25) * (-yz_mm + yz_mp - yz_pm + yz_pp) + T(0.5) * (zm1 - zp1);
        const T uyzz = T(0.5) * (ym1 - yp1) + T(0.25) * (yz_pp - yz_mm - yz_mp + yz_pm);
        const T uxxz = T(0.25) * (-zx_mm + zx_pm - zx_mp + zx_pp) + T(0.5) * (zm1 - zp1);
        const T uxzz = T(0.5) * (xm1 - xp1) + T(0.25) * (zx_pp - zx_mm - zx_pm + zx_mp);
        is4 += k7 * (uxy * uxy + uyz * uyz + uxz * uxz) +
               T(4.7) * (uxxy * uxxy + uxxz * uxxz + uxyy * uxyy + uxzz * uxzz + uyyz * uyyz + uyzz * uyzz);
        const T dxy1 = T(0.5) * (xy_pp - xy_pm) - cy, dxz1 = T(0.5) * (zx_pp - zx_mp) - cz;
        const T dxy2 = T(0.5) * (xy_mm - xy_mp) + cy, dxz2 = T(0.5) * (zx_mm - zx_pm) + cz;
        const T dxy3 = T(0.5) * (xy_pp - xy_mp) - cx, dyz3 = T(0.5) * (yz_pp - yz_pm) - cz;
        const T dxy4 = T(0.5) * (xy_mm - xy_pm) + cx, dyz4 = T(0.5) * (yz_mm - yz_mp) + cz;
        const T dyz5 = T(0.5) * (yz_pp - yz_mp) - cy, dxz5 = T(0.5) * (zx_pp - zx_pm) - cx;
        const T dyz6 = T(0.5) * (yz_mm - yz_pm) + cy, dxz6 = T(0.5) * (zx_mm - zx_mp) + cx;
        const T Cxy = k7 * uxy * uxy, Cyz = k7 * uyz * uyz, Cxz = k7 * uxz * uxz;
        is3[0] += Cxy + Cyz + Cxz;
        is3[1] += k7 * dxy1 * dxy1 + Cyz + k7 * dxz1 * dxz1;
        is3[2] += k7 * dxy2 * dxy2 + Cyz + k7 * dxz2 * dxz2;
        is3[3] += k7 * dxy3 * dxy3 + k7 * dyz3 * dyz3 + Cxz;
        is3[4] += k7 * dxy4 * dxy4 + k7 * dyz4 * dyz4 + Cxz;
        is3[5] += Cxy + k7 * dyz5 * dyz5 + k7 * dxz5 * dxz5;
        is3[6] += Cxy + k7 * dyz6 * dyz6 + k7 * dxz6 * dxz6;
    }
    asm volatile("" ::: "memory");
    {   // corners: u_xyz (reconstruction.c:108)
        const T uxyz = T(0.125) * (get(25) - get(26) - get(27) - get(28) + get(29) + get(30) + get(31) - get(32));
        is4 += T(61.0 / 48.0) * uxyz * uxyz;
    }

    // nonlinear weights, p = 4, eps = 1e-12 (reconstruction.c:118,205-218)
    const T eps = T(1.0e-12);
    const T g4 = T(p.g4), g3c = T(p.g3c), g3s = T(p.g3s);
    T w4;
    if constexpr (sizeof(T) == 8) {
        w4 = pos_pow4_inv(g4, is4 + eps);
        T total = w4;
        w3[0] = pos_pow4_inv(g3c, is3[0] + eps);
        total += w3[0];
#pragma unroll
        for (int k = 1; k < 7; ++k) {
            w3[k] = pos_pow4_inv(g3s, is3[k] + eps);
            total += w3[k];
        }
        const T it = rcp64(total);
        wt = (w4 * it) * T(p.inv_g4);
#pragma unroll
        for (int k = 0; k < 7; ++k) w3[k] *= it;
    } else {
        // FP32: ratio form gamma_k ((IS_min+eps)/(IS_k+eps))^4, identical after
        // normalisation but free of the underflow of (IS+eps)^4 ~ 1e-48.
        T t4 = is4 + eps, tm = t4, t3[7];
#pragma unroll
        for (int k = 0; k < 7; ++k) { t3[k] = is3[k] + eps; tm = fminf(tm, t3[k]); }
        auto rw = [&](T g, T t) { T r = tm * __builtin_amdgcn_rcpf(t); r = r * r; return g * r * r; };
        w4 = rw(g4, t4);
        T total = w4;
        w3[0] = rw(g3c, t3[0]);
        total += w3[0];
#pragma unroll
        for (int k = 1; k < 7; ++k) { w3[k] = rw(g3s, t3[k]); total += w3[k]; }
        const T it = __builtin_amdgcn_rcpf(total);
        wt = w4 * it * T(p.inv_g4);
#pragma unroll
        for (int k = 0; k < 7; ++k) w3[k] *= it;
    }
}

// CWENO combination (reconstruction.c:223-257) for the face-relevant
// coefficients only, from the 13 axis values (u0 and the x, y, z arms
// m2, m1, p1, p2) and the weights.  lin = sum gamma_k R3_k, nl = sum w_k R3_k.
template <typename T>
__device__ __forceinline__ void cweno_combine(T u0, T xm2, T xm1, T xp1, T xp2, T ym2, T ym1, T yp1, T yp2, T zm2,
                                              T zm1, T zp1, T zp2, T wt, const T (&w3)[7], const CwArgs &p,
                                              Axis3<T> &o)
{
    const T g3s = T(p.g3s);
    const T gc = T(p.g3c) + T(4) * g3s;           // weight of stencils central along an axis
    T ux, uy, uz, uxx, uyy, uzz, uxxx, uyyy, uzzz;
    axis_linear(xm2, xm1, u0, xp1, xp2, ux, uxx, uxxx);
    axis_linear(ym2, ym1, u0, yp1, yp2, uy, uyy, uyyy);
    axis_linear(zm2, zm1, u0, zp1, zp2, uz, uzz, uzzz);
    const T cx = T(0.5) * (xp1 - xm1), cy = T(0.5) * (yp1 - ym1), cz = T(0.5) * (zp1 - zm1);
    const T dx1 = T(-1.5) * u0 + T(2) * xp1 - T(0.5) * xp2, dxx1 = T(0.5) * (u0 - T(2) * xp1 + xp2);
    const T dx2 = T(-2) * xm1 + T(0.5) * xm2 + T(1.5) * u0, dxx2 = T(0.5) * (xm2 - T(2) * xm1 + u0);
    const T dy3 = T(-1.5) * u0 + T(2) * yp1 - T(0.5) * yp2, dyy3 = T(0.5) * (u0 - T(2) * yp1 + yp2);
    const T dy4 = T(-2) * ym1 + T(0.5) * ym2 + T(1.5) * u0, dyy4 = T(0.5) * (ym2 - T(2) * ym1 + u0);
    const T dz5 = T(-1.5) * u0 + T(2) * zp1 - T(0.5) * zp2, dzz5 = T(0.5) * (u0 - T(2) * zp1 + zp2);
    const T dz6 = T(-2) * zm1 + T(0.5) * zm2 + T(1.5) * u0, dzz6 = T(0.5) * (zm2 - T(2) * zm1 + u0);
    const T Wx = w3[0] + w3[3] + w3[4] + w3[5] + w3[6];
    const T Wy = w3[0] + w3[1] + w3[2] + w3[5] + w3[6];
    const T Wz = w3[0] + w3[1] + w3[2] + w3[3] + w3[4];
    o.c1[0] = wt * (ux - (gc * cx + g3s * (dx1 + dx2))) + (Wx * cx + w3[1] * dx1 + w3[2] * dx2);
    o.c2[0] = wt * (uxx - (gc * uxx + g3s * (dxx1 + dxx2))) + (Wx * uxx + w3[1] * dxx1 + w3[2] * dxx2);
    o.c3[0] = wt * uxxx;
    o.c1[1] = wt * (uy - (gc * cy + g3s * (dy3 + dy4))) + (Wy * cy + w3[3] * dy3 + w3[4] * dy4);
    o.c2[1] = wt * (uyy - (gc * uyy + g3s * (dyy3 + dyy4))) + (Wy * uyy + w3[3] * dyy3 + w3[4] * dyy4);
    o.c3[1] = wt * uyyy;
    o.c1[2] = wt * (uz - (gc * cz + g3s * (dz5 + dz6))) + (Wz * cz + w3[5] * dz5 + w3[6] * dz6);
    o.c2[2] = wt * (uzz - (gc * uzz + g3s * (dzz5 + dzz6))) + (Wz * uzz + w3[5] * dzz5 + w3[6] * dzz6);
    o.c3[2] = wt * uzzz;
}

// Full CWENO4 from a register array of the 33 stencil values: returns the
// axis coefficients (c1,c2,c3 per axis) and wt_ratio; wn (if not null)
// receives the eight normalised weights (R4, R3[0..6]).
template <typename T>
__device__ __forceinline__ T cweno_axes(const T (&s)[33], const CwArgs &p, Axis3<T> &o, T *wn = nullptr)
{
    T wt, w3[7];
    cweno_weights<T>([&](int q) { return s[q]; }, p, wt, w3);
    if (wn) {
        wn[0] = wt * T(p.g4);
#pragma unroll
        for (int k = 0; k < 7; ++k) wn[1 + k] = w3[k];
    }
    cweno_combine<T>(s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7], s[8], s[9], s[10], s[11], s[12], wt, w3, p, o);
    return wt;
}

// CWENO4 of one cell and component straight to its six face quantities
// (ACOUSTIC4: face-averaged values; WAVE2: h times the face-averaged normal
// gradients), the same scheme as cweno_weights + cweno_combine in far fewer
// operations.  The stage kernels are bound by the issue of these operations:
// about 240 FP64 instructions per cell and component, 3 of them reciprocals,
// against 515 with 9; in FP32 about 280 with 9 against 515 with 9 (the patch of
// a 256^3 selective stage 84 -> 66 us).  get(q): stencil slots of
// cweno_weights.  The memory clobbers keep one group of LDS values live at a
// time.  cweno_faces with full = false (per lane) gives the linear 4th-order
// polynomial: the same combination with n1 = n2 = 0 and the c3 share alone, so
// a wavefront with both kinds of lanes runs the common part once (66 -> 58 us
// with the loads of k_cweno).
//
// Per axis, from the first differences e1 .. e4 of m2, m1, u0, p1, p2:
//   A, B, C = e4-e3, e3-e2, e2-e1 (second), a, c = A-B, B-C (third),
//   S = e2+e3, T = a+c, F = a-c (fourth)
// and with Sh = S/2 (the central first derivative) the indicators are
//   central       cx^2 + 13/3 uxx^2        = Sh^2 + 13/12 B^2
//   one-sided +   dx1^2 + 13/3 dxx1^2      = (e3 - A/2)^2 + 13/12 A^2
//   one-sided -                              (e2 + C/2)^2 + 13/12 C^2
//   4th order     ux^2 + 13/3 uxx^2 + ux uxxx/5 + 39.06 uxxx^2
//                                          = Sh^2 + 13/12 B^2 + T (0.278125 T - Sh/6)
// For a pair of axes with the diagonals pp pm mp mm: al, be = (pp-pm)/2 - Shb,
// (mp-mm)/2 - Shb and ph, ps = (pp-mp)/2 - Sha, (pm-mm)/2 - Sha are the mixed
// derivatives of the four sided stencils; M = (al-be)^2 = (ph-ps)^2 is 4 u_ab^2,
// and the mixed third derivatives are (al+be)/2, (ph+ps)/2, whose squares follow
// from the others: (al+be)^2 = 2(al^2+be^2) - M.
// With normalised weights n4 (R4), n1, n2 (sided +, -) along an axis, and
// gamma_R4 + sum gamma_R3 = 1, the combination of reconstruction.c:223-257 is
//   2 c1  = S - n1 a - n2 c + n4 (g3s - 11/60)/g4 T
//   2 c2  = B + n1 a - n2 c - n4 g3s/g4 F
//   12 c3 = n4/g4 T
// Beside a jump (p1, p2 across it) the smooth sided stencil takes all the
// weight, n2 -> 1, and B - n2 c would leave the rounding of B, the jump's size,
// in a result of the size of C, the background's.  Where the sided stencils leave
// the others less than 1/1024, the sums of that axis start from the dominating
// stencil instead, with w = 1 - n2 summed from all other weights:
//   2 c2 = C + w c + n1 a - ...,  2 c1 = 2 e2 + C + w c - n1 a + ...
// (on the other side A - w a - n2 c and 2 e3 - A + w a - n2 c).  Above 1/1024 the
// indicators are within a factor of 23 and the jump within 5 of the background.
// The branch costs 2 to 3 % of a 256^3 ACOUSTIC4 step (4.36 -> 4.46 ms), where one
// wavefront in a hundred takes it, and 3 to 13 % of a 70 x 45 x 61 WAVE2 right-hand
// side (12.3 -> 12.6 .. 13.8 us), whose odd walls are jumps in a third of the
// wavefronts; these sums without a branch would add 7 % of the instructions
// everywhere.
// In FP64 the eight reciprocals 1/IS come from two, each of a product of four IS
// (in range whenever IS^4 is), each refined to full precision.  In FP32, where
// (IS + eps)^4 ~ 1e-48 underflows, the weights are gamma (IS_min / IS)^4.
template <int SYS, typename T, typename Get>
__device__ __forceinline__ void cweno_weights4(Get get, const CwArgs &p, const T (&S)[3], const T (&B)[3],
                                               const T (&a)[3], const T (&c)[3], const T (&e2)[3], const T (&e3)[3],
                                               const T (&A)[3], const T (&Cc)[3], T (&n)[6], T &is, T &ke, T &ko,
                                               T &rest)
{
    const T k13 = T(13.0 / 12.0), k7 = T(7.0 / 6.0), eps = T(1.0e-12);
    T C[3], P[3], M[3], Sh[3], is4;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const T G = a[d] + c[d];
        const T D1 = fma(T(-0.5), A[d], e3[d]), D2 = fma(T(0.5), Cc[d], e2[d]);
        Sh[d] = T(0.5) * S[d];
        C[d] = fma(Sh[d], Sh[d], fma(k13 * B[d], B[d], T(0.5) * eps));   // a sum of two carries eps
        P[d] = fma(D1, D1, (k13 * A[d]) * A[d]);
        M[d] = fma(D2, D2, (k13 * Cc[d]) * Cc[d]);
        const T t = fma(Sh[d], T(-1.0 / 6.0), T(0.278125) * G);
        is4 = d == 0 ? G * t : fma(G, t, is4);
    }
    const T Cyz = C[1] + C[2], Czx = C[2] + C[0], Cxy = C[0] + C[1];
    T t0 = Cyz + (C[0] - T(0.5) * eps);
    is4 += t0;
    asm volatile("" ::: "memory");
    // mixed derivatives of one pair of axes
    auto pair = [&](int q, T Sa, T Sb, T &al, T &be, T &ph, T &ps, T &m) {
        const T pp = get(q), pm = get(q + 1), mp = get(q + 2), mm = get(q + 3);
        al = fma(T(0.5), pp - pm, -Sb);
        be = fma(T(0.5), mp - mm, -Sb);
        ph = fma(T(0.5), pp - mp, -Sa);
        const T x = al - be;
        ps = ph - x;
        m = x * x;
    };
    T q[6], Mxy, Myz, Mzx;
    {
        T al, be, ph, ps;
        pair(13, Sh[0], Sh[1], al, be, ph, ps, Mxy);   // (x, y): x+, x-, y+, y-
        q[0] = al * al; q[1] = be * be; q[2] = ph * ph; q[3] = ps * ps;
        asm volatile("" ::: "memory");
        pair(17, Sh[1], Sh[2], al, be, ph, ps, Myz);   // (y, z): y+, y-, z+, z-
        q[2] = fma(al, al, q[2]); q[3] = fma(be, be, q[3]); q[4] = ph * ph; q[5] = ps * ps;
        asm volatile("" ::: "memory");
        pair(21, Sh[2], Sh[0], al, be, ph, ps, Mzx);   // (z, x): z+, z-, x+, x-
        q[4] = fma(al, al, q[4]); q[5] = fma(be, be, q[5]); q[0] = fma(ph, ph, q[0]); q[1] = fma(ps, ps, q[1]);
    }
    asm volatile("" ::: "memory");
    const T Ms = (Mxy + Myz) + Mzx;
    const T Q = ((q[0] + q[1]) + (q[2] + q[3])) + (q[4] + q[5]);
    t0 = fma(T(0.25) * k7, Ms, t0);
    is4 = fma(T(2.35), Q, is4);
    is4 = fma(T(0.25 * 7.0 / 6.0 - 2.35), Ms, is4);
    {
        const T z = ((get(25) - get(26)) - (get(27) - get(29))) - ((get(28) - get(30)) - (get(31) - get(32)));
        is4 = fma(T(61.0 / 3072.0) * z, z, is4);
    }
    const T t1 = fma(k7, fma(T(0.25), Myz, q[0]), P[0] + Cyz), t2 = fma(k7, fma(T(0.25), Myz, q[1]), M[0] + Cyz);
    const T t3 = fma(k7, fma(T(0.25), Mzx, q[2]), P[1] + Czx), t4 = fma(k7, fma(T(0.25), Mzx, q[3]), M[1] + Czx);
    const T t5 = fma(k7, fma(T(0.25), Mxy, q[4]), P[2] + Cxy), t6 = fma(k7, fma(T(0.25), Mxy, q[5]), M[2] + Cxy);

    // gamma / IS^4, p = 4 (reconstruction.c:205-218)
    T r4, r0;
    if constexpr (sizeof(T) == 8) {
        auto inv4 = [](T &w, T &x, T &y, T &z) {
            const T wx = w * x, yz = y * z;
            const T r = rcp64_full(wx * yz);
            const T rwx = r * yz, ryz = r * wx;
            const T iw = rwx * x, ix = rwx * w, iy = ryz * z, iz = ryz * y;
            w = iw; x = ix; y = iy; z = iz;
        };
        r4 = is4; r0 = t0; n[0] = t1; n[1] = t2; n[2] = t3; n[3] = t4; n[4] = t5; n[5] = t6;
        inv4(r4, r0, n[0], n[1]);
        inv4(n[2], n[3], n[4], n[5]);
    } else {
        const T tm = fminf(fminf(fminf(is4, t0), fminf(t1, t2)), fminf(fminf(t3, t4), fminf(t5, t6)));
        auto ratio = [&](T t) { return tm * __builtin_amdgcn_rcpf(t); };
        r4 = ratio(is4); r0 = ratio(t0);
        n[0] = ratio(t1); n[1] = ratio(t2); n[2] = ratio(t3); n[3] = ratio(t4); n[4] = ratio(t5); n[5] = ratio(t6);
    }
    auto pow4 = [](T r) { const T r2 = r * r; return r2 * r2; };
    const T g3s = T(p.g3s);
    T w4 = T(p.g4) * pow4(r4);
#pragma unroll
    for (int k = 0; k < 6; ++k) n[k] = pow4(n[k]);
    const T sided = ((n[0] + n[1]) + (n[2] + n[3])) + (n[4] + n[5]);
    const T central = fma(T(p.g3c), pow4(r0), w4);
    const T sum = fma(g3s, sided, central);
    T it;
    if constexpr (sizeof(T) == 8) it = rcp64_full(sum);
    else it = __builtin_amdgcn_rcpf(sum);
    is = g3s * it;
    rest = central * it;
    w4 *= it;
    ke = T(p.k2) * w4;
    ko = T(SYS == ACX_ACOUSTIC4 ? p.k1a : p.k1w) * w4;
}

template <int SYS, typename T, typename Get>
__device__ __forceinline__ void cweno_faces(Get get, const CwArgs &p, bool full, T (&fm)[3], T (&fp)[3])
{
    const T u0 = get(0);
    T S[3], B[3], a[3], c[3], n[6] = {};
    T e2[3], e3[3], A[3], Cc[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const T m2 = get(1 + 4 * d), m1 = get(2 + 4 * d), p1 = get(3 + 4 * d), p2 = get(4 + 4 * d);
        const T e1 = m1 - m2, e4 = p2 - p1;
        e2[d] = u0 - m1;
        e3[d] = p1 - u0;
        A[d] = e4 - e3[d];
        Cc[d] = e2[d] - e1;
        B[d] = e3[d] - e2[d];
        S[d] = e2[d] + e3[d];
        a[d] = A[d] - B[d];
        c[d] = B[d] - Cc[d];
    }
    T is = T(0), ke = T(0), ko = T(-1.0 / 6.0), rest = T(1);
    if (full) cweno_weights4<SYS, T>(get, p, S, B, a, c, e2, e3, A, Cc, n, is, ke, ko, rest);
    // faces of axis d from E = 2 c2 (less the share of c3) and O = 2 c1 (plus it)
    auto faces = [&](int d, T E, T O) {
        if constexpr (SYS == ACX_ACOUSTIC4) {
            const T even = fma(T(1.0 / 12.0), E, u0);
            fm[d] = fma(T(-0.25), O, even);
            fp[d] = fma(T(0.25), O, even);
        } else {
            fm[d] = T(0.5) * (O - E);
            fp[d] = T(0.5) * (O + E);
        }
    };
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const T h1 = n[2 * d] * a[d], h2 = n[2 * d + 1] * c[d];
        const T G = a[d] + c[d], F = a[d] - c[d];
        faces(d, fma(-ke, F, fma(is, h1 - h2, B[d])), fma(ko, G, fma(-is, h1 + h2, S[d])));
    }
    if (rest < T(1.0 / 1024.0)) {
        asm volatile("" ::: "memory");   // the axis values are read again
        const T half = T(0.5) * (((n[0] + n[1]) + (n[2] + n[3])) + (n[4] + n[5]));
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            if (n[k] > half) {
                const int d = k / 2, m = k % 2;   // m = 0: cells 0, +1, +2 of the axis; 1: 0, -1, -2
                const T v1 = get(m ? 2 + 4 * d : 3 + 4 * d), v2 = get(m ? 1 + 4 * d : 4 + 4 * d);
                const T t = v1 - u0, X = (v2 - v1) - t, Y = fma(T(2), t, -X);
                T others = T(0);
#pragma unroll
                for (int q = 0; q < 6; ++q) others += q == k ? T(0) : n[q];
                const T g = fma(is, others, rest) * (m ? c[d] : a[d]), h = (is * n[k ^ 1]) * (m ? a[d] : c[d]);
                const T G = a[d] + c[d], F = a[d] - c[d];
                faces(d, fma(-ke, F, m ? X + (h + g) : X - (h + g)), fma(ko, G, (m ? -Y : Y) + (g - h)));
            }
        }
    }
}

} // namespace acx
