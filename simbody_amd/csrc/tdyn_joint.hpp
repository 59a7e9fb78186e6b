// Articulated-body recursion in joint frames, FP64.
//
// The reference sweeps work in Ground: every body's rotation, hinge matrix
// and inertia are re-expressed there in each sweep.  The same recursion is
// much shorter in each body's own mobilizer frame M (fixed in the body, at
// the joint):
//   * mass properties about M are constants;
//   * the hinge columns are unit vectors, so D = H^T P H is a block of P,
//     P H are columns of P, and the rows of P+ along the hinge vanish;
//   * in terms of the acceleration of M's origin (not the spatial
//     acceleration) the only velocity that enters the dynamics is the
//     body's angular velocity w, and gravity is an upward acceleration of
//     Ground, so no pose is needed unless body forces are given in Ground.
// Going from a body to its parent is a planar rotation by the joint angle
// (Pin: z; Universal: y, then x after the elimination; Slider: none; Ball: a
// full rotation of the 3x3 mass block that is left of P+), the constant
// rotation R_MF between the parent's M and the joint's F frame (identity in
// most models), and a shift by r, F's origin in the parent's M frame.
//
// Same results as RigidBodyNodeSpec.cpp:249-446 and RigidBodyNode.cpp:54-213
// in exact arithmetic.
#pragma once
#include "tdyn_internal.hpp"
#include "tdyn_math.hpp"
#include "tdyn_chain.hpp"

namespace tdyn {
namespace joint {

using d3 = v3<double>;
using dm = m33<double>;
using chain::NormSums;

#define TDJ __device__ __forceinline__

// Symmetric 3x3, xx yy zz xy xz yz, by index pair.
struct sym { double a[6]; };
constexpr int sidx(int i, int j) {
    return i == j ? i : (i + j == 1 ? 3 : i + j == 2 ? 4 : 5);
}
// Articulated inertia about a frame's origin, [J F; F^T M].
struct art { sym M, J; double F[9]; };
struct wf { d3 w, v; };          // moment/force or angular/linear pair

template <int I> TDJ double& at(d3& v) { if constexpr (I == 0) return v.x; else if constexpr (I == 1) return v.y; else return v.z; }

// (v_I, v_J) -> (c v_I - s v_J, s v_I + c v_J); inverse with -s.
template <int I, int J> TDJ d3 planar(d3 v, double c, double s) {
    const double a = at<I>(v), b = at<J>(v);
    at<I>(v) = c*a - s*b; at<J>(v) = s*a + c*b;
    return v;
}
template <int I, int J> TDJ void planar(sym& S, double c, double s) {
    constexpr int K = 3 - I - J;
    const double xx = S.a[I], yy = S.a[J], xy = S.a[sidx(I, J)], xz = S.a[sidx(I, K)], yz = S.a[sidx(J, K)];
    const double a = c*xx - s*xy, b = c*xy - s*yy, d = s*xx + c*xy, e = s*xy + c*yy;
    S.a[I] = c*a - s*b; S.a[J] = s*d + c*e; S.a[sidx(I, J)] = s*a + c*b;
    S.a[sidx(I, K)] = c*xz - s*yz; S.a[sidx(J, K)] = s*xz + c*yz;
}
template <int I, int J> TDJ void planar(double* F, double c, double s) {
#pragma unroll
    for (int k = 0; k < 3; ++k) { const double a = F[3*I+k], b = F[3*J+k]; F[3*I+k] = c*a - s*b; F[3*J+k] = s*a + c*b; }
#pragma unroll
    for (int k = 0; k < 3; ++k) { const double a = F[3*k+I], b = F[3*k+J]; F[3*k+I] = c*a - s*b; F[3*k+J] = s*a + c*b; }
}
TDJ sym rot(const dm& R, const sym& S) {
    const s33<double> r = rotate_sym(R, s33<double>{S.a[0], S.a[1], S.a[2], S.a[3], S.a[4], S.a[5]});
    return {{r.xx, r.yy, r.zz, r.xy, r.xz, r.yz}};
}
TDJ void rot(const dm& R, double* F) {
    double T[9];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) T[3*r+c] = R.a[3*r]*F[c] + R.a[3*r+1]*F[3+c] + R.a[3*r+2]*F[6+c];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) F[3*r+c] = T[3*r]*R.a[3*c] + T[3*r+1]*R.a[3*c+1] + T[3*r+2]*R.a[3*c+2];
}
TDJ d3 mulsym(const sym& S, const d3& v) {
    return {S.a[0]*v.x + S.a[3]*v.y + S.a[4]*v.z, S.a[3]*v.x + S.a[1]*v.y + S.a[5]*v.z, S.a[4]*v.x + S.a[5]*v.y + S.a[2]*v.z};
}
TDJ d3 row(const double* F, int r) { return {F[3*r], F[3*r+1], F[3*r+2]}; }
TDJ d3 colv(const double* F, int c) { return {F[c], F[3+c], F[6+c]}; }
TDJ d3 mulF(const double* F, const d3& v) { return {dot(row(F, 0), v), dot(row(F, 1), v), dot(row(F, 2), v)}; }
TDJ d3 mulFt(const double* F, const d3& v) { return {dot(colv(F, 0), v), dot(colv(F, 1), v), dot(colv(F, 2), v)}; }

// About a new origin, r from it to the old one:
// F' = F + [r]x M, J' = J + [r]x F^T - F' [r]x.
TDJ void shift(art& P, const d3& r) {
    const d3 c0 = cross(r, d3{P.M.a[0], P.M.a[3], P.M.a[4]}), c1 = cross(r, d3{P.M.a[3], P.M.a[1], P.M.a[5]}),
             c2 = cross(r, d3{P.M.a[4], P.M.a[5], P.M.a[2]});
    const d3 a0 = cross(r, row(P.F, 0)), a1 = cross(r, row(P.F, 1)), a2 = cross(r, row(P.F, 2));
    P.F[0] += c0.x; P.F[1] += c1.x; P.F[2] += c2.x;
    P.F[3] += c0.y; P.F[4] += c1.y; P.F[5] += c2.y;
    P.F[6] += c0.z; P.F[7] += c1.z; P.F[8] += c2.z;
    const d3 b0 = cross(row(P.F, 0), r), b1 = cross(row(P.F, 1), r), b2 = cross(row(P.F, 2), r);
    P.J.a[0] += a0.x - b0.x; P.J.a[1] += a1.y - b1.y; P.J.a[2] += a2.z - b2.z;
    P.J.a[3] += a0.y - b1.x; P.J.a[4] += a0.z - b2.x; P.J.a[5] += a1.z - b2.y;
}
// The same where only the mass block is not zero.
TDJ void shift_mass(art& P, const d3& r) {
    const d3 c0 = cross(r, d3{P.M.a[0], P.M.a[3], P.M.a[4]}), c1 = cross(r, d3{P.M.a[3], P.M.a[1], P.M.a[5]}),
             c2 = cross(r, d3{P.M.a[4], P.M.a[5], P.M.a[2]});
    P.F[0] = c0.x; P.F[1] = c1.x; P.F[2] = c2.x;
    P.F[3] = c0.y; P.F[4] = c1.y; P.F[5] = c2.y;
    P.F[6] = c0.z; P.F[7] = c1.z; P.F[8] = c2.z;
    const d3 b0 = cross(row(P.F, 0), r), b1 = cross(row(P.F, 1), r), b2 = cross(row(P.F, 2), r);
    P.J = {{-b0.x, -b1.y, -b2.z, -b1.x, -b2.x, -b2.y}};
}

// The same after a Pin about z (row z of F and of J zero), after a Universal
// (row x zero; J is j e e^T and F is e f^T with e normal to x).
TDJ void shift_pin(art& P, const d3& r) {
    const d3 c0 = cross(r, d3{P.M.a[0], P.M.a[3], P.M.a[4]}), c1 = cross(r, d3{P.M.a[3], P.M.a[1], P.M.a[5]}),
             c2 = cross(r, d3{P.M.a[4], P.M.a[5], P.M.a[2]});
    const d3 a0 = cross(r, row(P.F, 0)), a1 = cross(r, row(P.F, 1));
    P.F[0] += c0.x; P.F[1] += c1.x; P.F[2] += c2.x;
    P.F[3] += c0.y; P.F[4] += c1.y; P.F[5] += c2.y;
    P.F[6] = c0.z; P.F[7] = c1.z; P.F[8] = c2.z;
    const d3 b0 = cross(row(P.F, 0), r), b1 = cross(row(P.F, 1), r), b2 = cross(row(P.F, 2), r);
    P.J.a[0] += a0.x - b0.x; P.J.a[1] += a1.y - b1.y; P.J.a[2] = -b2.z;
    P.J.a[3] += a0.y - b1.x; P.J.a[4] = a0.z - b2.x; P.J.a[5] = a1.z - b2.y;
}
TDJ void shift_universal(art& P, const d3& r) {
    const d3 c0 = cross(r, d3{P.M.a[0], P.M.a[3], P.M.a[4]}), c1 = cross(r, d3{P.M.a[3], P.M.a[1], P.M.a[5]}),
             c2 = cross(r, d3{P.M.a[4], P.M.a[5], P.M.a[2]});
    const d3 a1 = cross(r, row(P.F, 1)), a2 = cross(r, row(P.F, 2));
    P.F[0] = c0.x; P.F[1] = c1.x; P.F[2] = c2.x;
    P.F[3] += c0.y; P.F[4] += c1.y; P.F[5] += c2.y;
    P.F[6] += c0.z; P.F[7] += c1.z; P.F[8] += c2.z;
    const d3 b0 = cross(row(P.F, 0), r), b1 = cross(row(P.F, 1), r), b2 = cross(row(P.F, 2), r);
    P.J.a[0] = -b0.x; P.J.a[1] += a1.y - b1.y; P.J.a[2] += a2.z - b2.z;
    P.J.a[3] = -b1.x; P.J.a[4] = -b2.x; P.J.a[5] += a1.z - b2.y;
}

// sin and cos for |x| < 2^20, the library's beyond.  x - k pi/2 in three parts
// (Cody and Waite): the first is exact in one fused multiply-add, the second a
// product with its error, subtracted with the error of the difference (next to
// a multiple of pi/2 the difference is as small as the product's rounding
// would be), so that r + lo is the remainder to 2^-100.  Then polynomials in
// r^2 through the Chebyshev nodes of [0, (pi/4)^2] (largest error 2e-17) and lo
// to first order: 46 instructions where the library's small-argument path takes
// 130, under 1 ulp as that is.  One angle per body and derivative made it a
// sixth of a chain derivative.
TDJ bool big_angle(double x) { return !(fabs(x) < 1048576.0); }
TDJ void sincos_small(double x, double* sp, double* cp) {
#pragma clang fp contract(off)
    const double k = rint(x * 0.6366197723675814);
    const double t = fma(-k, 1.5707963267948966, x);
    const double p = k * 6.123233995736766e-17, pe = fma(k, 6.123233995736766e-17, -p);
    const double r = t - p, rb = r - t;
    const double re = (t - (r - rb)) - (p + rb);
    const double lo = fma(-k, -1.4973849048591698e-33, re - pe);
    const double z = r*r;
    const double ps = fma(z, fma(z, fma(z, fma(z, fma(z, 1.591810123027412e-10, -2.5051131455427946e-08),
                                                2.755731610068303e-06), -0.0001984126983675497),
                                 0.008333333333330946), -0.16666666666666666);
    const double pc = fma(z, fma(z, fma(z, fma(z, fma(z, -1.1382614868556325e-11, 2.0876146024689747e-09),
                                                -2.7557317270560326e-07), 2.4801587298763433e-05),
                                 -0.0013888888888887395), 0.041666666666666664);
    const double hz = 0.5*z;
    const double sn = r + fma(r*z, ps, fma(-hz, lo, lo));
    const double w = 1.0 - hz;
    const double cs = w + (((1.0 - w) - hz) + fma(z*z, pc, -(r*lo)));
    const int n = (int)k;
    const double a = (n & 1) ? cs : sn, b = (n & 1) ? sn : cs;
    *sp = (n & 2) ? -a : a;
    *cp = ((n + 1) & 2) ? -b : b;
}
TDJ void sincos_joint(double x, double* sp, double* cp) {
    if (big_angle(x)) { sincos(x, sp, cp); return; }
    sincos_small(x, sp, cp);
}

// ---------------------------------------------------------------------------
// Joints.  J axes: where the hinge columns are unit vectors.  Pin: the body's
// M axes; Slider: the same (= F axes); Universal: F turned by the first angle;
// Ball: M axes; Free: F axes.
// ---------------------------------------------------------------------------
template <int T> struct Dim {
    static constexpr int D = T <= SLIDER ? 1 : T == UNIVERSAL ? 2 : T == BALL ? 3 : 6;
    static constexpr int NQ = T <= SLIDER ? 1 : T == UNIVERSAL ? 2 : T == BALL ? 4 : 7;
    static constexpr bool quat = T == BALL || T == FREE;
    // hand-over values per body: G without its known entries, DI*eps; trig
    static constexpr int G = jt_g(T), TC = jt_tc(T);
};

template <int T> struct Jnt {
    double c0, s0, c1, s1;      // Pin: c0 s0; Universal: both angles
    dm R;                       // Ball, Free: R_FM
    d3 p;                       // Slider, Free: p_FM
    // trig / normalization values of q
    static TDJ void trig(const double* q, double* tc) {
        if constexpr (T == PIN) sincos_joint(q[0], &tc[1], &tc[0]);
        else if constexpr (T == UNIVERSAL) { sincos_joint(q[0], &tc[1], &tc[0]); sincos_joint(q[1], &tc[3], &tc[2]); }
        else if constexpr (Dim<T>::quat) tc[0] = 1.0 / sqrt(q[0]*q[0] + q[1]*q[1] + q[2]*q[2] + q[3]*q[3]);
    }
    TDJ void set(const double* q, const double* tc) {
        if constexpr (T == PIN) { c0 = tc[0]; s0 = tc[1]; }
        else if constexpr (T == UNIVERSAL) { c0 = tc[0]; s0 = tc[1]; c1 = tc[2]; s1 = tc[3]; }
        else if constexpr (T == SLIDER) p = {q[0], 0.0, 0.0};
        else {
            R = quat_rot(q[0]*tc[0], q[1]*tc[0], q[2]*tc[0], q[3]*tc[0]);
            if constexpr (T == FREE) p = {q[4], q[5], q[6]};
        }
    }
    TDJ d3 toJ(const d3& v) const {          // F -> J
        if constexpr (T == PIN) return planar<0, 1>(v, c0, -s0);
        else if constexpr (T == UNIVERSAL) return planar<1, 2>(v, c0, -s0);
        else if constexpr (T == BALL) return mulT(R, v);
        else return v;
    }
    TDJ d3 fromJ(const d3& v) const {        // J -> F
        if constexpr (T == PIN) return planar<0, 1>(v, c0, s0);
        else if constexpr (T == UNIVERSAL) return planar<1, 2>(v, c0, s0);
        else if constexpr (T == BALL) return mul(R, v);
        else return v;
    }
    TDJ d3 toB(const d3& v) const {          // J -> M
        if constexpr (T == UNIVERSAL) return planar<2, 0>(v, c1, -s1);
        else if constexpr (T == FREE) return mulT(R, v);
        else return v;
    }
    TDJ d3 fromB(const d3& v) const {        // M -> J
        if constexpr (T == UNIVERSAL) return planar<2, 0>(v, c1, s1);
        else if constexpr (T == FREE) return mul(R, v);
        else return v;
    }
    // angular velocity across the joint, J axes
    TDJ d3 wrel(const double* u) const {
        if constexpr (T == PIN) return {0.0, 0.0, u[0]};
        else if constexpr (T == UNIVERSAL) return {u[0], u[1], 0.0};
        else if constexpr (T == BALL) return mulT(R, d3{u[0], u[1], u[2]});
        else if constexpr (T == FREE) return {u[0], u[1], u[2]};
        else return zero3<double>();
    }
    // w + wrel, J axes
    TDJ d3 add_wrel(const d3& w, const double* u) const {
        if constexpr (T == PIN) return {w.x, w.y, w.z + u[0]};
        else if constexpr (T == UNIVERSAL) return {w.x + u[0], w.y + u[1], w.z};
        else if constexpr (T == SLIDER) return w;
        else return w + wrel(u);
    }
    // bias of the angular acceleration, J axes: wp x wrel plus the turning
    // of the hinge columns; wp: the parent's angular velocity in J axes
    TDJ d3 bias_w(const d3& wp, const double* u) const {
        if constexpr (T == PIN) return {wp.y*u[0], -(wp.x*u[0]), 0.0};
        else if constexpr (T == UNIVERSAL)
            return {-(wp.z*u[1]), wp.z*u[0], (wp.x*u[1] - wp.y*u[0]) + u[0]*u[1]};
        else if constexpr (T == SLIDER) return zero3<double>();
        else return cross(wp, wrel(u));
    }
};

// Constant of body b's model: PA = cdptr (one model) or PrmT (one per lane).
template <bool IDF, class PA> TDJ d3 toF(const PA& P, const d3& v) {     // parent's M -> F
    if constexpr (IDF) return v;
    else {
        dm R; for (int i = 0; i < 9; ++i) R.a[i] = P[JC_R + i];
        return mulT(R, v);
    }
}
template <bool IDF, class PA> TDJ d3 fromF(const PA& P, const d3& v) {
    if constexpr (IDF) return v;
    else {
        dm R; for (int i = 0; i < 9; ++i) R.a[i] = P[JC_R + i];
        return mul(R, v);
    }
}
// F's origin (Slider, Free: M's origin) in the parent's M frame
template <int T, bool IDF, class PA> TDJ d3 arm(const PA& P, const Jnt<T>& J) {
    const d3 l = {P[JC_L], P[JC_L + 1], P[JC_L + 2]};
    if constexpr (T == SLIDER || T == FREE) return l + fromF<IDF>(P, J.p);
    else return l;
}
// w x (w x r)
TDJ d3 centripetal(const d3& w, const d3& r) {
    const double a = dot(w, r), b = dot(w, w);
    return {a*w.x - b*r.x, a*w.y - b*r.y, a*w.z - b*r.z};
}
// bias of the acceleration of M's origin, J axes; w: the parent's angular
// velocity (its M axes), wF the same in F axes
template <int T, bool IDF, class PA>
TDJ d3 bias_v(const PA& P, const Jnt<T>& J, const d3& w, const d3& wF, const d3& r, const double* u) {
    d3 k = toF<IDF>(P, centripetal(w, r));
    if constexpr (T == SLIDER) { k.y += 2*u[0]*wF.z; k.z -= 2*u[0]*wF.y; }
    if constexpr (T == FREE) k = k + 2.0*cross(wF, d3{u[3], u[4], u[5]});
    return J.toJ(k);
}

// Base to tip: the body's angular velocity from its parent's (M axes each).
template <int T, bool IDF, class PA>
TDJ d3 out_w(const PA& P, const Jnt<T>& J, const d3& w, const double* u) {
    return J.toB(J.add_wrel(J.toJ(toF<IDF>(P, w)), u));
}
// Ground rotation of M: R_GM = R_GMp R_MF R_FM; `in` undoes it.
template <int T> TDJ dm joint_rot(const Jnt<T>& J) {
    if constexpr (T == PIN) return {{J.c0, -J.s0, 0, J.s0, J.c0, 0, 0, 0, 1}};
    else if constexpr (T == SLIDER) return ident<double>();
    else if constexpr (T == UNIVERSAL)
        return {{J.c1, 0, J.s1, J.s1*J.s0, J.c0, -J.s0*J.c1, -J.s1*J.c0, J.s0, J.c0*J.c1}};
    else return J.R;
}
template <int T, bool IDF, class PA> TDJ dm out_R(const PA& P, const Jnt<T>& J, const dm& R) {
    if constexpr (IDF) return mul(R, joint_rot<T>(J));
    else {
        dm C; for (int i = 0; i < 9; ++i) C.a[i] = P[JC_R + i];
        return mul(mul(R, C), joint_rot<T>(J));
    }
}
template <int T, bool IDF, class PA> TDJ dm in_R(const PA& P, const Jnt<T>& J, const dm& R) {
    const dm A = chain::mulABt(R, joint_rot<T>(J));
    if constexpr (IDF) return A;
    else {
        dm C; for (int i = 0; i < 9; ++i) C.a[i] = P[JC_R + i];
        return chain::mulABt(A, C);
    }
}

// LDL^T solve of the symmetric positive definite 6x6 [J F; F^T M] x = b, in
// the elimination order of its rows; `bad` when a pivot is not above 1e-13
// of its diagonal entry.
TDJ bool solve6(const art& P, const double* b, double* x) {
    double A[6][6];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            A[i][j] = P.J.a[sidx(i, j)]; A[3+i][3+j] = P.M.a[sidx(i, j)];
            A[3+j][i] = P.F[3*i+j];
        }
    bool bad = false;
    double dg[6], ip[6], y[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) dg[k] = A[k][k];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        bad = bad || !(A[k][k] > 1e-13 * dg[k]);
        ip[k] = 1.0 / A[k][k];
#pragma unroll
        for (int i = k + 1; i < 6; ++i) {
            const double f = A[i][k] * ip[k];
#pragma unroll
            for (int j = k + 1; j <= i; ++j) A[i][j] -= f * A[j][k];
        }
    }
    // A[i][k] (i > k) holds L[i][k] d_k
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        double s = b[i];
#pragma unroll
        for (int k = 0; k < i; ++k) s -= A[i][k] * ip[k] * y[k];
        y[i] = s;
    }
#pragma unroll
    for (int i = 5; i >= 0; --i) {
        double s = y[i];
#pragma unroll
        for (int k = i + 1; k < 6; ++k) s -= A[k][i] * x[k];
        x[i] = s * ip[i];
    }
    return bad;
}

// ---------------------------------------------------------------------------
// Elimination of one joint, J axes.  In: P and z of the body with its
// children, tau the applied mobility forces along the hinge columns (TAU).  Out: G
// (Dim::G values without the known ones) and DI*eps into g[], and P, z become
// P+ and z + G eps (the bias P+ ab is added by the caller).  Returns whether D
// was not positive definite.
// ---------------------------------------------------------------------------
template <int T, bool TAU> TDJ bool eliminate(art& P, wf& z, const double* tau, double* g) {
    double* F = P.F;
    auto ta = [&](int k) { return TAU ? tau[k] : 0.0; };
    auto ep = [&](int k, double z) { return TAU ? tau[k] - z : -z; };
    if constexpr (T == PIN) {
        const double D = P.J.a[2], o = 1.0 / D;
        const double ux = P.J.a[4], uy = P.J.a[5];
        const d3 uv = row(F, 2);
        const double gx = ux*o, gy = uy*o;
        const d3 gv = {uv.x*o, uv.y*o, uv.z*o};
        const double eps = ep(0, z.w.z);
        z.w.x += gx*eps; z.w.y += gy*eps; z.w.z = ta(0);
        z.v = z.v + eps*gv;
        P.J.a[0] -= gx*ux; P.J.a[1] -= gy*uy; P.J.a[3] -= gx*uy;
        P.J.a[2] = 0; P.J.a[4] = 0; P.J.a[5] = 0;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            F[k] -= gx*F[6+k]; F[3+k] -= gy*F[6+k];
        }
        F[6] = 0; F[7] = 0; F[8] = 0;
        P.M.a[0] -= gv.x*uv.x; P.M.a[1] -= gv.y*uv.y; P.M.a[2] -= gv.z*uv.z;
        P.M.a[3] -= gv.x*uv.y; P.M.a[4] -= gv.x*uv.z; P.M.a[5] -= gv.y*uv.z;
        g[0] = gx; g[1] = gy; g[2] = gv.x; g[3] = gv.y; g[4] = gv.z; g[5] = o*eps;
        return !(D > 0.0);
    } else if constexpr (T == SLIDER) {
        const double D = P.M.a[0], o = 1.0 / D;
        const d3 ua = colv(F, 0);
        const double uy = P.M.a[3], uz = P.M.a[4];
        const d3 ga = {ua.x*o, ua.y*o, ua.z*o};
        const double gy = uy*o, gz = uz*o;
        const double eps = ep(0, z.v.x);
        z.w = z.w + eps*ga;
        z.v.x = ta(0); z.v.y += gy*eps; z.v.z += gz*eps;
        P.J.a[0] -= ga.x*ua.x; P.J.a[1] -= ga.y*ua.y; P.J.a[2] -= ga.z*ua.z;
        P.J.a[3] -= ga.x*ua.y; P.J.a[4] -= ga.x*ua.z; P.J.a[5] -= ga.y*ua.z;
        F[0] = 0; F[3] = 0; F[6] = 0;
        F[1] -= ga.x*uy; F[4] -= ga.y*uy; F[7] -= ga.z*uy;
        F[2] -= ga.x*uz; F[5] -= ga.y*uz; F[8] -= ga.z*uz;
        P.M.a[1] -= gy*uy; P.M.a[2] -= gz*uz; P.M.a[5] -= gy*uz;
        P.M.a[0] = 0; P.M.a[3] = 0; P.M.a[4] = 0;
        g[0] = ga.x; g[1] = ga.y; g[2] = ga.z; g[3] = gy; g[4] = gz; g[5] = o*eps;
        return !(D > 0.0);
    } else if constexpr (T == UNIVERSAL) {
        const double dxx = P.J.a[0], dyy = P.J.a[1], dxy = P.J.a[3];
        const double det = dxx*dyy - dxy*dxy, o = 1.0 / det;
        const double i00 = o*dyy, i11 = o*dxx, i01 = -(o*dxy);
        const double ax = P.J.a[4], ay = P.J.a[5];                // angular z entries of P H
        const d3 fx = row(F, 0), fy = row(F, 1);
        const double gzx = ax*i00 + ay*i01, gzy = ax*i01 + ay*i11;
        const d3 gx = {fx.x*i00 + fy.x*i01, fx.y*i00 + fy.y*i01, fx.z*i00 + fy.z*i01};
        const d3 gy = {fx.x*i01 + fy.x*i11, fx.y*i01 + fy.y*i11, fx.z*i01 + fy.z*i11};
        const double e0 = ep(0, z.w.x), e1 = ep(1, z.w.y);
        z.w.x = ta(0); z.w.y = ta(1); z.w.z += gzx*e0 + gzy*e1;
        z.v.x += gx.x*e0 + gy.x*e1; z.v.y += gx.y*e0 + gy.y*e1; z.v.z += gx.z*e0 + gy.z*e1;
        P.J.a[2] -= gzx*ax + gzy*ay;
        P.J.a[0] = 0; P.J.a[1] = 0; P.J.a[3] = 0; P.J.a[4] = 0; P.J.a[5] = 0;
#pragma unroll
        for (int k = 0; k < 3; ++k) { F[6+k] -= gzx*F[k] + gzy*F[3+k]; F[k] = 0; F[3+k] = 0; }
        P.M.a[0] -= gx.x*fx.x + gy.x*fy.x; P.M.a[1] -= gx.y*fx.y + gy.y*fy.y; P.M.a[2] -= gx.z*fx.z + gy.z*fy.z;
        P.M.a[3] -= gx.x*fx.y + gy.x*fy.y; P.M.a[4] -= gx.x*fx.z + gy.x*fy.z; P.M.a[5] -= gx.y*fx.z + gy.y*fy.z;
        g[0] = gzx; g[1] = gx.x; g[2] = gx.y; g[3] = gx.z; g[4] = gzy; g[5] = gy.x; g[6] = gy.y; g[7] = gy.z;
        g[8] = i00*e0 + i01*e1; g[9] = i01*e0 + i11*e1;
        return !(det > 0.0);
    } else if constexpr (T == BALL) {
        const double* A = P.J.a;
        const double c00 = A[1]*A[2] - A[5]*A[5], c01 = A[5]*A[4] - A[3]*A[2], c02 = A[3]*A[5] - A[1]*A[4];
        const double det = A[0]*c00 + A[3]*c01 + A[4]*c02, o = 1.0 / det;
        const double i00 = o*c00, i01 = o*c01, i02 = o*c02, i11 = o*(A[0]*A[2] - A[4]*A[4]),
                     i12 = o*(A[3]*A[4] - A[0]*A[5]), i22 = o*(A[0]*A[1] - A[3]*A[3]);
        // G_v[l][j] = sum_i F[i][l] DI[i][j]
        double G[9];
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            G[3*l]   = F[l]*i00 + F[3+l]*i01 + F[6+l]*i02;
            G[3*l+1] = F[l]*i01 + F[3+l]*i11 + F[6+l]*i12;
            G[3*l+2] = F[l]*i02 + F[3+l]*i12 + F[6+l]*i22;
        }
        const d3 e = {ep(0, z.w.x), ep(1, z.w.y), ep(2, z.w.z)};
        z.w = {ta(0), ta(1), ta(2)};
        z.v = z.v + mulF(G, e);
#pragma unroll
        for (int l = 0; l < 3; ++l)
#pragma unroll
            for (int m = l; m < 3; ++m)
                P.M.a[sidx(l, m)] -= G[3*l]*F[m] + G[3*l+1]*F[3+m] + G[3*l+2]*F[6+m];
#pragma unroll
        for (int k = 0; k < 9; ++k) { F[k] = 0; g[k] = G[k]; }
#pragma unroll
        for (int k = 0; k < 6; ++k) P.J.a[k] = 0;
        g[9]  = i00*e.x + i01*e.y + i02*e.z;
        g[10] = i01*e.x + i11*e.y + i12*e.z;
        g[11] = i02*e.x + i12*e.y + i22*e.z;
        return !(det > 0.0);
    } else {
        // Free: the whole 6x6; P+ = 0 and G = identity
        const double b[6] = {ep(0, z.w.x), ep(1, z.w.y), ep(2, z.w.z), ep(3, z.v.x), ep(4, z.v.y), ep(5, z.v.z)};
        const bool bad = solve6(P, b, g);
        z.w = {ta(0), ta(1), ta(2)}; z.v = {ta(3), ta(4), ta(5)};
#pragma unroll
        for (int k = 0; k < 6; ++k) { P.M.a[k] = 0; P.J.a[k] = 0; }
#pragma unroll
        for (int k = 0; k < 9; ++k) F[k] = 0;
        return bad;
    }
}
// z += P+ ab (only the entries of P+ that are not zero)
template <int T> TDJ void add_bias(const art& P, wf& z, const d3& aw, const d3& av) {
    const double* F = P.F;
    if constexpr (T == PIN) {
        z.w.x += (P.J.a[0]*aw.x + P.J.a[3]*aw.y) + dot(row(F, 0), av);
        z.w.y += (P.J.a[3]*aw.x + P.J.a[1]*aw.y) + dot(row(F, 1), av);
        const d3 m = mulsym(P.M, av);
        z.v.x += m.x + (F[0]*aw.x + F[3]*aw.y);
        z.v.y += m.y + (F[1]*aw.x + F[4]*aw.y);
        z.v.z += m.z + (F[2]*aw.x + F[5]*aw.y);
    } else if constexpr (T == SLIDER) {
        z.w.x += F[1]*av.y + F[2]*av.z; z.w.y += F[4]*av.y + F[5]*av.z; z.w.z += F[7]*av.y + F[8]*av.z;
        z.v.y += P.M.a[1]*av.y + P.M.a[5]*av.z; z.v.z += P.M.a[5]*av.y + P.M.a[2]*av.z;
    } else if constexpr (T == UNIVERSAL) {
        z.w.z += P.J.a[2]*aw.z + dot(row(F, 2), av);
        const d3 m = mulsym(P.M, av);
        z.v.x += m.x + F[6]*aw.z; z.v.y += m.y + F[7]*aw.z; z.v.z += m.z + F[8]*aw.z;
    } else if constexpr (T == BALL) {
        z.v = z.v + mulsym(P.M, av);
    }
}
// P+, z+ from J axes to F axes (TAU: with applied mobility forces; without, a
// Ball transmits no moment)
template <int T, bool TAU> TDJ void to_F(const Jnt<T>& J, art& P, wf& z) {
    if constexpr (T != BALL || TAU) z.w = J.fromJ(z.w);
    z.v = J.fromJ(z.v);
    double* F = P.F;
    if constexpr (T == PIN) {
        planar<0, 1>(P.M, J.c0, J.s0);
        const double xx = P.J.a[0], yy = P.J.a[1], xy = P.J.a[3], c = J.c0, s = J.s0;
        const double a = c*xx - s*xy, b = c*xy - s*yy, d = s*xx + c*xy, e = s*xy + c*yy;
        P.J.a[0] = c*a - s*b; P.J.a[1] = s*d + c*e; P.J.a[3] = s*a + c*b;
#pragma unroll
        for (int k = 0; k < 3; ++k) { const double p = F[k], q = F[3+k]; F[k] = c*p - s*q; F[3+k] = s*p + c*q; }
#pragma unroll
        for (int k = 0; k < 2; ++k) { const double p = F[3*k], q = F[3*k+1]; F[3*k] = c*p - s*q; F[3*k+1] = s*p + c*q; }
    } else if constexpr (T == UNIVERSAL) {
        planar<1, 2>(P.M, J.c0, J.s0);
        const double j = P.J.a[2], c = J.c0, s = J.s0;
        P.J.a[1] = s*s*j; P.J.a[5] = -(s*c*j); P.J.a[2] = c*c*j;
        const double fy = c*F[7] - s*F[8], fz = s*F[7] + c*F[8], fx = F[6];
        F[3] = -s*fx; F[4] = -s*fy; F[5] = -s*fz;
        F[6] = c*fx; F[7] = c*fy; F[8] = c*fz;
    } else if constexpr (T == BALL) {
        P.M = rot(J.R, P.M);
    }
}
// P, z from M axes to J axes
template <int T> TDJ void to_J(const Jnt<T>& J, art& P, wf& z) {
    if constexpr (T == UNIVERSAL) {
        planar<2, 0>(P.M, J.c1, J.s1); planar<2, 0>(P.J, J.c1, J.s1); planar<2, 0>(P.F, J.c1, J.s1);
    } else if constexpr (T == FREE) {
        P.M = rot(J.R, P.M); P.J = rot(J.R, P.J); rot(J.R, P.F);
    }
    z.w = J.fromB(z.w); z.v = J.fromB(z.v);
}
// P+, z+ from F axes at F's origin to the parent's M frame
template <int T, bool IDF, bool TAU, class PA> TDJ void to_parent(const PA& C, art& P, wf& z, const d3& r) {
    if constexpr (!IDF) {
        dm R; for (int i = 0; i < 9; ++i) R.a[i] = C[JC_R + i];
        P.M = rot(R, P.M);
        if constexpr (T != BALL) { P.J = rot(R, P.J); rot(R, P.F); }
        if constexpr (T != BALL || TAU) z.w = mul(R, z.w);
        z.v = mul(R, z.v);
    }
    if constexpr (T == BALL) shift_mass(P, r);
    else if constexpr (T == PIN && IDF) shift_pin(P, r);
    else if constexpr (T == UNIVERSAL && IDF) shift_universal(P, r);
    else shift(P, r);
    if constexpr (T == BALL && !TAU) z.w = cross(r, z.v);
    else z.w = z.w + cross(r, z.v);
}
// P and z of the rigid body itself added (M axes)
template <class PA> TDJ void add_body(const PA& C, art& P) {
    const double m = C[JC_M];
    const d3 c = {C[JC_C], C[JC_C + 1], C[JC_C + 2]};
    P.M.a[0] += m; P.M.a[1] += m; P.M.a[2] += m;
#pragma unroll
    for (int k = 0; k < 6; ++k) P.J.a[k] += C[JC_I + k];
    P.F[1] -= c.z; P.F[2] += c.y; P.F[3] += c.z; P.F[5] -= c.x; P.F[6] -= c.y; P.F[7] += c.x;
}
// the body's velocity-dependent force, w x (I w) and w x (w x c)
template <class PA> TDJ wf gyro(const PA& C, const d3& w) {
    const sym I = {{C[JC_I], C[JC_I + 1], C[JC_I + 2], C[JC_I + 3], C[JC_I + 4], C[JC_I + 5]}};
    const d3 c = {C[JC_C], C[JC_C + 1], C[JC_C + 2]};
    return {cross(w, mulsym(I, w)), centripetal(w, c)};
}
TDJ art zero_art() { art P; for (int k = 0; k < 6; ++k) { P.M.a[k] = 0; P.J.a[k] = 0; } for (int k = 0; k < 9; ++k) P.F[k] = 0; return P; }

// One body of the tip-to-base sweep: P, z (M axes, its children's share in)
// with the body added, the joint eliminated and the rest taken to the
// parent's M frame; w: the body's angular velocity, wpar its parent's (M axes
// each; not recovered from w, whose rounding would be the parent's where the
// body turns much faster).  z already holds minus the applied force.  root:
// nothing is handed on.  VEL: with the velocity terms (else u, w and wpar are
// not read).
template <int T, bool IDF, bool TAU, bool VEL = true, class PA>
TDJ bool in_body(const PA& C, const Jnt<T>& J, const double* u, const double* tau, art& P, wf& z, const d3& w,
                 const d3& wpar, double* g, bool root) {
    add_body(C, P);
    if constexpr (VEL) {
        const wf b = gyro(C, w);
        z.w = z.w + b.w; z.v = z.v + b.v;
    }
    to_J<T>(J, P, z);
    bool bad;
    if constexpr (T == BALL && TAU) {
        const d3 t = mulT(J.R, d3{tau[0], tau[1], tau[2]});     // given in F
        const double tm[3] = {t.x, t.y, t.z};
        bad = eliminate<T, TAU>(P, z, tm, g);
    } else bad = eliminate<T, TAU>(P, z, tau, g);
    if (root) return bad;
    const d3 r = arm<T, IDF>(C, J);
    if constexpr (VEL && T != FREE) {
        const d3 wF = toF<IDF>(C, wpar);
        add_bias<T>(P, z, J.bias_w(J.toJ(wF), u), bias_v<T, IDF>(C, J, wpar, wF, r, u));
    }
    to_F<T, TAU>(J, P, z);
    to_parent<T, IDF, TAU>(C, P, z, r);
    return bad;
}
// One body of the base-to-tip acceleration sweep: A (acceleration of M's
// origin and angular acceleration, the parent's in, the body's out, M axes),
// w likewise; g as in_body left it.  ud: udot, along the reference's hinge
// columns.
template <int T, bool IDF, bool VEL = true, class PA>
TDJ void out_body(const PA& C, const Jnt<T>& J, const double* u, const double* g, wf& A, d3& w, double* ud) {
    const d3 r = arm<T, IDF>(C, J);
    d3 av = J.toJ(toF<IDF>(C, A.v + cross(A.w, r)));
    d3 aw = J.toJ(toF<IDF>(C, A.w));
    d3 wp;
    if constexpr (VEL) {
        const d3 wF = toF<IDF>(C, w);
        wp = J.toJ(wF);
        av = av + bias_v<T, IDF>(C, J, w, wF, r, u);
        aw = aw + J.bias_w(wp, u);
    }
    if constexpr (T == PIN) {
        ud[0] = g[5] - ((g[0]*aw.x + g[1]*aw.y + aw.z) + (g[2]*av.x + g[3]*av.y + g[4]*av.z));
        aw.z += ud[0];
    } else if constexpr (T == SLIDER) {
        ud[0] = g[5] - ((g[0]*aw.x + g[1]*aw.y + g[2]*aw.z) + (av.x + g[3]*av.y + g[4]*av.z));
        av.x += ud[0];
    } else if constexpr (T == UNIVERSAL) {
        ud[0] = g[8] - ((aw.x + g[0]*aw.z) + (g[1]*av.x + g[2]*av.y + g[3]*av.z));
        ud[1] = g[9] - ((aw.y + g[4]*aw.z) + (g[5]*av.x + g[6]*av.y + g[7]*av.z));
        aw.x += ud[0]; aw.y += ud[1];
    } else if constexpr (T == BALL) {
        const d3 e = d3{g[9], g[10], g[11]} - (aw + mulFt(g, av));
        const d3 f = mul(J.R, e);
        ud[0] = f.x; ud[1] = f.y; ud[2] = f.z;
        aw = aw + e;
    } else {
        ud[0] = g[0] - aw.x; ud[1] = g[1] - aw.y; ud[2] = g[2] - aw.z;
        ud[3] = g[3] - av.x; ud[4] = g[4] - av.y; ud[5] = g[5] - av.z;
        aw = {g[0], g[1], g[2]}; av = {g[3], g[4], g[5]};
    }
    A.w = J.toB(aw); A.v = J.toB(av);
    if constexpr (VEL) w = J.toB(J.add_wrel(wp, u));
}
// x += H v, x -= H v in J axes (v along the reference's hinge columns)
template <int T> TDJ void add_hinge(const Jnt<T>& J, wf& x, const double* v, double s) {
    if constexpr (T == PIN) x.w.z += s*v[0];
    else if constexpr (T == SLIDER) x.v.x += s*v[0];
    else if constexpr (T == UNIVERSAL) { x.w.x += s*v[0]; x.w.y += s*v[1]; }
    else {
        x.w = x.w + s*J.wrel(v);
        if constexpr (T == FREE) x.v = x.v + s*d3{v[3], v[4], v[5]};
    }
}
// H^T x, J axes
template <int T> TDJ void hinge_t(const Jnt<T>& J, const wf& x, double* t) {
    if constexpr (T == PIN) t[0] = x.w.z;
    else if constexpr (T == SLIDER) t[0] = x.v.x;
    else if constexpr (T == UNIVERSAL) { t[0] = x.w.x; t[1] = x.w.y; }
    else {
        const d3 f = J.fromJ(x.w);
        t[0] = f.x; t[1] = f.y; t[2] = f.z;
        if constexpr (T == FREE) { t[3] = x.v.x; t[4] = x.v.y; t[5] = x.v.z; }
    }
}
// Acceleration (or velocity, with VEL false) of the body from its parent's
// and v = udot (u) of its joint.
template <int T, bool IDF, bool VEL, class PA>
TDJ void out_given(const PA& C, const Jnt<T>& J, const double* u, const double* v, wf& A, d3& w) {
    const d3 r = arm<T, IDF>(C, J);
    wf x{J.toJ(toF<IDF>(C, A.w)), J.toJ(toF<IDF>(C, A.v + cross(A.w, r)))};
    if constexpr (VEL) {
        const d3 wF = toF<IDF>(C, w), wp = J.toJ(wF);
        x.v = x.v + bias_v<T, IDF>(C, J, w, wF, r, u);
        x.w = x.w + J.bias_w(wp, u);
        w = J.toB(J.add_wrel(wp, u));
    }
    add_hinge<T>(J, x, v, 1.0);
    A.w = J.toB(x.w); A.v = J.toB(x.v);
}
// A force on the body (M axes) to its parent's M frame.
template <int T, bool IDF, class PA> TDJ wf in_force(const PA& C, const Jnt<T>& J, const wf& x, const d3& r) {
    const d3 f = fromF<IDF>(C, J.fromJ(x.v));
    return {fromF<IDF>(C, J.fromJ(x.w)) + cross(r, f), f};
}
// I A (+ velocity terms): the force that gives the rigid body acceleration A
template <bool VEL, class PA> TDJ wf rigid_force(const PA& C, const wf& A, const d3& w) {
    const sym I = {{C[JC_I], C[JC_I + 1], C[JC_I + 2], C[JC_I + 3], C[JC_I + 4], C[JC_I + 5]}};
    const d3 c = {C[JC_C], C[JC_C + 1], C[JC_C + 2]};
    const double m = C[JC_M];
    wf f{mulsym(I, A.w) + cross(c, A.v), m*A.v + cross(A.w, c)};
    if constexpr (VEL) { f.w = f.w + cross(w, mulsym(I, w)); f.v = f.v + centripetal(w, c); }
    return f;
}

} // namespace joint
} // namespace tdyn
