// Rollouts of batches of one serial chain in the joint-frame recursion
// (tdyn_joint.hpp), FP64: Runge-Kutta-Merson with the reference's step
// control (RungeKuttaMersonIntegrator.cpp:86-140, AbstractIntegratorRep.cpp:
// 137-208, 448-609), one lane per instance, all steps of a launch in one
// kernel.
//
// One derivative is two sweeps.  The tip-to-base sweep eliminates the joints
// and keeps G and DI*eps per body; the base-to-tip sweep forms udot and, body
// by body while its values are in registers, the next stage's state, whose
// angular velocities it propagates on the way (the sweep that a separate
// kinematics pass would be).  So the stage derivatives that Merson's method
// uses only once (stages 1 and 4) never reach memory, and qdot is formed
// again from the stage's q and u where it is needed.
//
// The angular velocities are kept for the sweep back too (three doubles per
// body, in the rows of its G).  Recovered from the tip's by subtraction they
// moved 12 % fewer bytes (65,536 x 32: 11.2 ms for 16 steps, 12.6 as it is),
// but a slow body's carried the rounding of a fast outer one's: udot of two
// arms with a balanced wheel at 1e7 rad/s was off by 5e-11.  (Those of every
// second body only, the others formed from their parents': 5 % faster at this
// size, 4 to 5 % slower for one chain and for 4,001.)
//
// What bounds it.  65,536 chains of 32 bodies are one wavefront per SIMD; a
// step moves 56 kB per instance between the sweeps (half of it G and DI*eps)
// at 4.7 TB/s, near the 4.9 that a plain copy reaches, and issues half as many
// vector instructions as the Ground-frame sweeps did: 0.77 ms per step against
// 1.43 ms.  A few chains are bound by the instruction issue of single
// wavefronts: 430 vector instructions a body and sweep, 66 % of the cycles
// issuing and 29 % waiting (one 10-link pendulum: 1.3 against 2.6 ms for 0.1 s
// at accuracy 1e-8).
#pragma once
#include "tdyn_joint.hpp"
#include "tdyn_rkm_chain.hpp"

namespace tdyn {
namespace joint {

// Rows of one lane's state and hand-over values.  TILE: a wavefront's rows
// are one block, row k at 64*k doubles, so that a body's rows are reached
// from one scalar base with immediate offsets (and a wavefront's data lies in
// a few memory pages); else rows of pitch W = all lanes.
template <bool TILE> struct Row {
    TD_GLOBAL double* b; int W; unsigned l8;
    TDJ size_t pitch() const { if constexpr (TILE) return 64; else return (size_t)W; }
    TDJ Row from(int r) const { return {b + r * pitch(), W, l8}; }
    TDJ TD_GLOBAL double& operator()(int k) const {
        return *(TD_GLOBAL double*)((TD_GLOBAL char*)(b + k * pitch()) + l8);
    }
};
// One model per lane, in the same blocks.
struct PrmT {
    const TD_GLOBAL double* b; unsigned l8;
    TDJ double operator[](int k) const { return *(const TD_GLOBAL double*)((const TD_GLOBAL char*)(b + k * 64) + l8); }
    TDJ PrmT operator+(size_t k) const { return {b + k * 64, l8}; }
};

// Trig rows of one lane: in LDS (one column per lane) or with the others.
template <class R> struct TcG {
    R r;
    TDJ double get(int k) const { return r(k); }
    TDJ void put(int k, double v) const { r(k) = v; }
};
struct TcL {
    double* p;
    TDJ double get(int k) const { return p[k * 64]; }
    TDJ void put(int k, double v) const { p[k * 64] = v; }
};

// What a sweep needs of one body from memory, loaded a body ahead.
template <int NQ, int D> struct InB { double q[NQ], u[D], tc[4], w[3]; };      // (w: the parent's angular velocity)
template <int NQ, int D, int G> struct OutB {
    double q[NQ], u[D], tc[4], g[G], yq[NQ], yu[D], f0[D], fq[NQ], fu[D];
};
using InC = InB<4, 3>;
using OutC = OutB<4, 3, 12>;

// HASF: with applied body forces (given in Ground, so the bodies' rotations are
// carried along).
template <class PA, bool IDF, bool HASF, class Rows, class TC> struct Eval {
    PA prm; const int4* body_j; const int4* body_a;
    int nb, nq;
    Rows sc; TC tc; d3 g; const double* fapp;

    TDJ int4 bj(int b) const { return ldi4(body_j, b - 1); }
    TDJ int4 ba(int b) const { return ldi4(body_a, b - 1); }
    TDJ PA C(int b) const { return prm + (size_t)(b - 1) * PRM_STRIDE; }

    // ---- base to tip: angular velocities (and trig) of a state -----------
    template <int T> TDJ void kin(int b, const int4& j, const double* q, const double* u, d3& w, dm& R) const {
        double t[4];
        Jnt<T> J;
        J.trig(q, t); J.set(q, t);
#pragma unroll
        for (int k = 0; k < Dim<T>::TC; ++k) tc.put(j.z + k, t[k]);
        w = out_w<T, IDF>(C(b), J, w, u);
        const Rows G = sc.from(j.y);        // (read on the way back, before G is written there)
        G(0) = w.x; G(1) = w.y; G(2) = w.z;
        if constexpr (HASF) R = out_R<T, IDF>(C(b), J, R);
    }
    // MODE 0: the state y itself; 1: the first Merson stage y0 + h/3 f0,
    // stored to st (an attempt after a rejected one)
    template <int T> TDJ void head_body(int b, const int4& a, const int4& j, int mode, const Rows& y, const Rows& f0,
                                        const Rows& st, double h, d3& w, dm& R) const {
        constexpr int NQ = Dim<T>::NQ, D = Dim<T>::D;
        double q[NQ], u[D];
        const Rows yq = y.from(a.z), yu = y.from(nq + a.w);
#pragma unroll
        for (int k = 0; k < NQ; ++k) q[k] = yq(k);
#pragma unroll
        for (int k = 0; k < D; ++k) u[k] = yu(k);
        if (mode) {
            const Rows fu = f0.from(nq + a.w), sq = st.from(a.z), su = st.from(nq + a.w);
            double qd[NQ];
            qdot<T>(q, u, qd);
#pragma unroll
            for (int k = 0; k < NQ; ++k) { q[k] = q[k] + (h/3)*qd[k]; sq(k) = q[k]; }
#pragma unroll
            for (int k = 0; k < D; ++k) { u[k] = u[k] + (h/3)*fu(k); su(k) = u[k]; }
        }
        kin<T>(b, j, q, u, w, R);
    }
    TDJ void head(int mode, const Rows& y, const Rows& f0, const Rows& st, double h, d3& w, dm& R) const {
        w = zero3<double>(); R = ident<double>();
#pragma unroll 1
        for (int b = 1; b <= nb; ++b) {
            const int4 a = ba(b), j = bj(b);
            switch (a.y) {
            case PIN:       head_body<PIN>(b, a, j, mode, y, f0, st, h, w, R); break;
            case SLIDER:    head_body<SLIDER>(b, a, j, mode, y, f0, st, h, w, R); break;
            case UNIVERSAL: head_body<UNIVERSAL>(b, a, j, mode, y, f0, st, h, w, R); break;
            case BALL:      head_body<BALL>(b, a, j, mode, y, f0, st, h, w, R); break;
            default:        head_body<FREE>(b, a, j, mode, y, f0, st, h, w, R); break;
            }
        }
    }
    template <int T> static TDJ void qdot(const double* q, const double* u, double* qd) {
        if constexpr (Dim<T>::quat) {
            quat_dot(q, d3{u[0], u[1], u[2]}, qd);
            if constexpr (T == FREE) { qd[4] = u[3]; qd[5] = u[4]; qd[6] = u[5]; }
        } else {
#pragma unroll
            for (int k = 0; k < Dim<T>::D; ++k) qd[k] = u[k];
        }
    }

    // ---- tip to base ------------------------------------------------------
    template <int T, class X> TDJ void in_load(X& x, const int4& a, const int4& j, const Rows& st) const {
        const Rows su = st.from(nq + a.w);
#pragma unroll
        for (int k = 0; k < Dim<T>::D; ++k) x.u[k] = su(k);
        if constexpr (T != PIN && T != UNIVERSAL) {
            const Rows sq = st.from(a.z);
#pragma unroll
            for (int k = 0; k < Dim<T>::NQ; ++k) x.q[k] = sq(k);
        }
#pragma unroll
        for (int k = 0; k < Dim<T>::TC; ++k) x.tc[k] = tc.get(j.z + k);
        const Rows G = sc.from(j.w);
#pragma unroll
        for (int k = 0; k < 3; ++k) x.w[k] = G(k);
    }
    template <int T, class X> TDJ void in_step(const X& x, int b, const int4& j, art& P, wf& z, d3& w, dm& R) const {
        const PA c = C(b);
        Jnt<T> J;
        J.set(x.q, x.tc);
        if constexpr (HASF) {
            const double* f = fapp + 6*b;
            const d3 fm = mulT(R, d3{f[3], f[4], f[5]});
            z.w = z.w - (mulT(R, d3{f[0], f[1], f[2]}) + cross(d3{c[JC_B], c[JC_B + 1], c[JC_B + 2]}, fm));
            z.v = z.v - fm;
            R = in_R<T, IDF>(c, J, R);
        }
        double g[Dim<T>::G];
        const d3 wpar = {x.w[0], x.w[1], x.w[2]};
        (void)in_body<T, IDF, false>(c, J, x.u, nullptr, P, z, w, wpar, g, b == 1);
        w = wpar;
        const Rows G = sc.from(j.y);
#pragma unroll
        for (int k = 0; k < Dim<T>::G; ++k) G(k) = g[k];
    }
    TDJ void in_load_any(InC& x, const int4& a, const int4& j, const Rows& st) const {
        switch (a.y) {
        case PIN:       in_load<PIN>(x, a, j, st); break;
        case SLIDER:    in_load<SLIDER>(x, a, j, st); break;
        case UNIVERSAL: in_load<UNIVERSAL>(x, a, j, st); break;
        default:        in_load<BALL>(x, a, j, st); break;
        }
    }
    TDJ void in_any(const InC& x, int b, const int4& a, const int4& j, art& P, wf& z, d3& w, dm& R) const {
        switch (a.y) {
        case PIN:       in_step<PIN>(x, b, j, P, z, w, R); break;
        case SLIDER:    in_step<SLIDER>(x, b, j, P, z, w, R); break;
        case UNIVERSAL: in_step<UNIVERSAL>(x, b, j, P, z, w, R); break;
        default:        in_step<BALL>(x, b, j, P, z, w, R); break;
        }
    }
    TDJ void inward(const Rows& st, d3 w, dm R) const {
        art P = zero_art(); wf z{zero3<double>(), zero3<double>()};
        const int4 a1 = ba(1);
        const int b0 = a1.y == FREE ? 2 : 1;        // a Free root is taken last, by itself
        InC A, B;
        int4 aA = ba(nb), jA = bj(nb), aB, jB;
        if (nb >= b0) in_load_any(A, aA, jA, st);
#pragma unroll 1
        for (int b = nb; b >= b0; b -= 2) {
            if (b - 1 >= b0) { aB = ba(b - 1); jB = bj(b - 1); in_load_any(B, aB, jB, st); }
            in_any(A, b, aA, jA, P, z, w, R);
            if (b - 1 < b0) break;
            if (b - 2 >= b0) { aA = ba(b - 2); jA = bj(b - 2); in_load_any(A, aA, jA, st); }
            in_any(B, b - 1, aB, jB, P, z, w, R);
        }
        if (b0 == 2) {
            InB<7, 6> x;
            const int4 j1 = bj(1);
            in_load<FREE>(x, a1, j1, st);
            in_step<FREE>(x, 1, j1, P, z, w, R);
        }
    }

    // ---- base to tip, with the next stage ---------------------------------
    // stage: the one whose derivative is formed (0 f0 .. 4 f4); st: its state.
    struct Rk { Rows y, st, nx, f0, f2, f3, y1; double h; int stage; };
    template <int T, class X> TDJ void out_load(X& x, const int4& a, const int4& j, const Rk& r) const {
        constexpr int NQ = Dim<T>::NQ, D = Dim<T>::D;
        const Rows su = r.st.from(nq + a.w);
#pragma unroll
        for (int k = 0; k < D; ++k) x.u[k] = su(k);
        // q: of quaternions and translations always; of angles where it is
        // the state itself (stage 0) or enters the error estimate (stage 4)
        if (Dim<T>::quat || T == SLIDER || r.stage == 0 || r.stage == 4) {
            const Rows sq = r.st.from(a.z);
#pragma unroll
            for (int k = 0; k < NQ; ++k) x.q[k] = sq(k);
        }
#pragma unroll
        for (int k = 0; k < Dim<T>::TC; ++k) x.tc[k] = tc.get(j.z + k);
        const Rows G = sc.from(j.y);
#pragma unroll
        for (int k = 0; k < Dim<T>::G; ++k) x.g[k] = G(k);
        if (r.stage > 0) {
            const Rows yq = r.y.from(a.z), yu = r.y.from(nq + a.w), f0 = r.f0.from(nq + a.w);
#pragma unroll
            for (int k = 0; k < NQ; ++k) x.yq[k] = yq(k);
#pragma unroll
            for (int k = 0; k < D; ++k) { x.yu[k] = yu(k); x.f0[k] = f0(k); }
        }
        if (r.stage > 2) {
            const Rows f = r.stage == 3 ? r.f2 : r.f3, fq = f.from(a.z), fu = f.from(nq + a.w);
#pragma unroll
            for (int k = 0; k < NQ; ++k) x.fq[k] = fq(k);
#pragma unroll
            for (int k = 0; k < D; ++k) x.fu[k] = fu(k);
        }
    }
    template <int T, class X>
    TDJ void out_step(const X& x, int b, const int4& a, const int4& j, const Rk& r, wf& A, d3& w, d3& wn, dm& R,
                      NormSums& ns) const {
        constexpr int NQ = Dim<T>::NQ, D = Dim<T>::D;
        const PA c = C(b);
        double ud[D], fq[NQ], q[NQ], u[D];
        {
            Jnt<T> J;
            J.set(x.q, x.tc);
            out_body<T, IDF>(c, J, x.u, x.g, A, w, ud);
        }
        qdot<T>(x.q, x.u, fq);
        const double h = r.h;
        const int ui = nq + a.w;
        if (r.stage == 0) {
            const Rows o0 = r.f0.from(ui);
#pragma unroll
            for (int k = 0; k < NQ; ++k) q[k] = x.q[k] + (h/3)*fq[k];
#pragma unroll
            for (int k = 0; k < D; ++k) { o0(k) = ud[k]; u[k] = x.u[k] + (h/3)*ud[k]; }
        } else {
            double f0q[NQ];
            qdot<T>(x.yq, x.yu, f0q);
            if (r.stage == 1) {
#pragma unroll
                for (int k = 0; k < NQ; ++k) q[k] = x.yq[k] + (h/6)*(f0q[k] + fq[k]);
#pragma unroll
                for (int k = 0; k < D; ++k) u[k] = x.yu[k] + (h/6)*(x.f0[k] + ud[k]);
            } else if (r.stage == 2) {
                const Rows oq = r.f2.from(a.z), ou = r.f2.from(ui);
#pragma unroll
                for (int k = 0; k < NQ; ++k) { oq(k) = fq[k]; q[k] = x.yq[k] + (h/8)*(f0q[k] + 3*fq[k]); }
#pragma unroll
                for (int k = 0; k < D; ++k) { ou(k) = ud[k]; u[k] = x.yu[k] + (h/8)*(x.f0[k] + 3*ud[k]); }
            } else if (r.stage == 3) {
                const Rows oq = r.f3.from(a.z), ou = r.f3.from(ui);
#pragma unroll
                for (int k = 0; k < NQ; ++k) { oq(k) = fq[k]; q[k] = x.yq[k] + (h/2)*((f0q[k] - 3*x.fq[k]) + 4*fq[k]); }
#pragma unroll
                for (int k = 0; k < D; ++k) { ou(k) = ud[k]; u[k] = x.yu[k] + (h/2)*((x.f0[k] - 3*x.fu[k]) + 4*ud[k]); }
            } else {
                // y1, its error estimate 0.2 |y1 - y_stage4| and the sums of
                // its norm (IntegratorRep.h:454-523, 644-655)
                const Rows oq = r.y1.from(a.z), ou = r.y1.from(ui);
                double e[NQ];
#pragma unroll
                for (int k = 0; k < NQ; ++k) {
                    q[k] = x.yq[k] + (h/6)*((f0q[k] + 4*x.fq[k]) + fq[k]);
                    oq(k) = q[k];
                    e[k] = 0.2 * fabs(q[k] - x.q[k]);
                }
                if constexpr (Dim<T>::quat) {
                    const d3 v = quat_dot_to_w(q, e);
                    double d4[4]; quat_dot(q, v, d4);
                    ns.sq_quat += d4[0]*d4[0] + d4[1]*d4[1] + d4[2]*d4[2] + d4[3]*d4[3];
                    if constexpr (T == FREE) ns.sq_other += e[4]*e[4] + e[5]*e[5] + e[6]*e[6];
                    const double qe = sqrt(q[0]*q[0] + q[1]*q[1] + q[2]*q[2] + q[3]*q[3]) - 1.0;
                    ns.s2 += qe*qe;
                } else {
#pragma unroll
                    for (int k = 0; k < NQ; ++k) ns.sq_other += e[k]*e[k];
                }
#pragma unroll
                for (int k = 0; k < D; ++k) {
                    u[k] = x.yu[k] + (h/6)*((x.f0[k] + 4*x.fu[k]) + ud[k]);
                    ou(k) = u[k];
                    const double vi = fabs(x.yu[k]);
                    const double us = vi > 1.0 ? 1.0/vi : 1.0;
                    const double xx = us * (0.2 * fabs(u[k] - x.u[k]));
                    ns.su += xx*xx;
                }
                return;
            }
        }
        const Rows nxq = r.nx.from(a.z), nxu = r.nx.from(ui);
#pragma unroll
        for (int k = 0; k < NQ; ++k) nxq(k) = q[k];
#pragma unroll
        for (int k = 0; k < D; ++k) nxu(k) = u[k];
        kin<T>(b, j, q, u, wn, R);
    }
    TDJ void out_load_any(OutC& x, const int4& a, const int4& j, const Rk& r) const {
        switch (a.y) {
        case PIN:       out_load<PIN>(x, a, j, r); break;
        case SLIDER:    out_load<SLIDER>(x, a, j, r); break;
        case UNIVERSAL: out_load<UNIVERSAL>(x, a, j, r); break;
        default:        out_load<BALL>(x, a, j, r); break;
        }
    }
    TDJ void out_any(const OutC& x, int b, const int4& a, const int4& j, const Rk& r, wf& A, d3& w, d3& wn, dm& R,
                     NormSums& ns) const {
        switch (a.y) {
        case PIN:       out_step<PIN>(x, b, a, j, r, A, w, wn, R, ns); break;
        case SLIDER:    out_step<SLIDER>(x, b, a, j, r, A, w, wn, R, ns); break;
        case UNIVERSAL: out_step<UNIVERSAL>(x, b, a, j, r, A, w, wn, R, ns); break;
        default:        out_step<BALL>(x, b, a, j, r, A, w, wn, R, ns); break;
        }
    }
    // wn, R: the next stage's angular velocity and rotation at the tip.
    TDJ void outward(const Rk& r, d3& wn, dm& R, NormSums& ns) const {
        wf A{zero3<double>(), -g};
        d3 w = zero3<double>();
        wn = zero3<double>(); R = ident<double>();
        const int4 a1 = ba(1);
        int b0 = 1;
        if (a1.y == FREE) {
            OutB<7, 6, 6> x;
            const int4 j1 = bj(1);
            out_load<FREE>(x, a1, j1, r);
            out_step<FREE>(x, 1, a1, j1, r, A, w, wn, R, ns);
            b0 = 2;
        }
        if (b0 > nb) return;
        OutC X, Y;
        int4 aX = ba(b0), jX = bj(b0), aY, jY;
        out_load_any(X, aX, jX, r);
#pragma unroll 1
        for (int b = b0; b <= nb; b += 2) {
            if (b + 1 <= nb) { aY = ba(b + 1); jY = bj(b + 1); out_load_any(Y, aY, jY, r); }
            out_any(X, b, aX, jX, r, A, w, wn, R, ns);
            if (b + 1 > nb) break;
            if (b + 2 <= nb) { aX = ba(b + 2); jX = bj(b + 2); out_load_any(X, aX, jX, r); }
            out_any(Y, b + 1, aY, jY, r, A, w, wn, R, ns);
        }
    }
    // udot alone (the derivative of the rollout's state)
    template <int T> TDJ void acc_body(int b, const int4& a, const int4& j, const Rows& y, const Rows& f, wf& A, d3& w) const {
        constexpr int NQ = Dim<T>::NQ, D = Dim<T>::D;
        OutB<NQ, D, Dim<T>::G> x;
        const Rows yq = y.from(a.z), yu = y.from(nq + a.w), fq = f.from(a.z), fu = f.from(nq + a.w), G = sc.from(j.y);
#pragma unroll
        for (int k = 0; k < NQ; ++k) x.q[k] = yq(k);
#pragma unroll
        for (int k = 0; k < D; ++k) x.u[k] = yu(k);
#pragma unroll
        for (int k = 0; k < Dim<T>::TC; ++k) x.tc[k] = tc.get(j.z + k);
#pragma unroll
        for (int k = 0; k < Dim<T>::G; ++k) x.g[k] = G(k);
        double ud[D], qd[NQ];
        Jnt<T> J;
        J.set(x.q, x.tc);
        out_body<T, IDF>(C(b), J, x.u, x.g, A, w, ud);
        qdot<T>(x.q, x.u, qd);
#pragma unroll
        for (int k = 0; k < NQ; ++k) fq(k) = qd[k];
#pragma unroll
        for (int k = 0; k < D; ++k) fu(k) = ud[k];
    }
    TDJ void derivative(const Rows& y, const Rows& f) const {
        d3 w; dm R;
        head(0, y, y, y, 0.0, w, R);
        inward(y, w, R);
        wf A{zero3<double>(), -g};
        w = zero3<double>();
#pragma unroll 1
        for (int b = 1; b <= nb; ++b) {
            const int4 a = ba(b), j = bj(b);
            switch (a.y) {
            case PIN:       acc_body<PIN>(b, a, j, y, f, A, w); break;
            case SLIDER:    acc_body<SLIDER>(b, a, j, y, f, A, w); break;
            case UNIVERSAL: acc_body<UNIVERSAL>(b, a, j, y, f, A, w); break;
            case BALL:      acc_body<BALL>(b, a, j, y, f, A, w); break;
            default:        acc_body<FREE>(b, a, j, y, f, A, w); break;
            }
        }
    }
};

// Row numbers in a lane's block of 11 vectors of ny_max rows (VY and VF0 as
// every rollout has them): y1 in VY0's, f2, f3 and the stage state in VFA, VFB
// and VYS, then G and the trig rows (fewer than 5 ny_max).
enum { R_Y = VY, R_Y1 = VY0, R_F0 = VF0, R_F2 = VFA, R_F3 = VFB, R_ST = VYS, R_G = VY1 };

template <bool TILE> TDJ Row<TILE> block_rows(const RkmArgs& a) {
    const size_t off = TILE ? (size_t)blockIdx.x * NVEC * a.ny_max * 64 : (size_t)blockIdx.x * 64;
    return {(TD_GLOBAL double*)a.vec + off, a.L, threadIdx.x * 8u};
}
// The model of this lane's serving slot.
TDJ PrmT slot_prm(const RkmArgs& a, int nb) {
    return {(const TD_GLOBAL double*)a.prm_lane + blockIdx.x * ((size_t)nb * PRM_STRIDE + 3) * 64, threadIdx.x * 8u};
}
template <class PA, bool IDF, bool HASF, bool TILE, class TC>
TDJ Eval<PA, IDF, HASF, Row<TILE>, TC> make_eval(const RkmArgs& a, int lane, double* lds) {
    Eval<PA, IDF, HASF, Row<TILE>, TC> ev;
    const int4 ta = ldi4(a.T.tree_a, 0);
    ev.nb = ta.x; ev.nq = ta.y;
    ev.body_a = a.T.body_a + ta.w; ev.body_j = a.T.body_j + ta.w;
    ev.sc = block_rows<TILE>(a).from(R_G * a.ny_max);
    if constexpr (std::is_same<TC, TcL>::value) ev.tc = TcL{lds + threadIdx.x};
    else ev.tc = TC{ev.sc.from(a.g_rows)};
    if constexpr (std::is_same<PA, PrmT>::value) {
        ev.prm = slot_prm(a, ta.x);
        const PrmT gl = ev.prm + (size_t)ta.x * PRM_STRIDE;
        ev.g = {gl[0], gl[1], gl[2]};
    } else {
        ev.prm = cptr(a.T.prm_j) + (size_t)ta.w * PRM_STRIDE;
        const cdptr g = cptr(a.T.gravity);
        ev.g = {g[0], g[1], g[2]};
    }
    ev.fapp = HASF ? a.fapp + 6*(size_t)a.off.b_off[lane] : nullptr;
    return ev;
}

template <class PA, bool IDF, bool HASF, bool TILE, class TC>
__device__ __forceinline__ void advance_lane(const RkmArgs& a, int lane, double* lds) {
    const auto ev = make_eval<PA, IDF, HASF, TILE, TC>(a, lane, lds);
    using Rows = Row<TILE>;
    const int4 ta = ldi4(a.T.tree_a, 0);
    const int nb = ta.x, nq = ta.y, nu = ta.z, ny = nq + nu;
    const int4* body_a = a.T.body_a + ta.w;
    const int nquat = ldi4(a.T.tree_b, 0).y;
    const Rows base = block_rows<TILE>(a);
    auto rows = [&](int v) { return base.from(v * a.ny_max); };
    const Rows S0 = rows(R_Y), S1 = rows(R_Y1), ST = rows(R_ST);

    const RkmCfg& cfg = a.cfg;
    const double acc = cfg.accuracy, consTol = cfg.cons_tol;
    double hmin = cfg.min_h, hmax = cfg.max_h;
    if (cfg.fixed_h > 0) { hmin = hmax = cfg.fixed_h; }
    const double projLimit = fmax(2*consTol, sqrt(consTol));
    double t = a.t[lane], hcur = a.h[lane];
    const double tEnd = a.t_end[lane];
    int attempts = a.stats[4*lane], accepted = a.stats[4*lane+1], rejected = a.stats[4*lane+2],
        projections = a.stats[4*lane+3];
    int status = 0, steps = 0;
    bool flip = false;     // current state in S1

    while (steps < cfg.max_steps) {
        if (t >= tEnd) { status = 1; break; }
        // Every active lane has taken the same number of accepted steps in
        // this launch, so flip is wave-uniform; saying so keeps the row
        // bases in scalar registers.
        const bool fl = __builtin_amdgcn_readfirstlane(flip ? 1 : 0) != 0;
        const Rows Y = fl ? S1 : S0, Y1 = fl ? S0 : S1;
        typename Eval<PA, IDF, HASF, Rows, TC>::Rk r{Y, Y, ST, rows(R_F0), rows(R_F2), rows(R_F3), Y1, 0.0, 0};
        d3 w; dm R;
        bool ok = false, first = true;
        double t1 = t;
        do {
            bool limited = false;
            if (tEnd < t + 0.95*hcur) { limited = true; t1 = tEnd; }
            else if (tEnd > t + 1.001*hcur) t1 = t + hcur;
            else t1 = tEnd;
            if (!(t1 > t)) { status = -3; break; }
            if (++attempts > cfg.max_attempts) { status = -2; break; }
            r.h = t1 - t;
            NormSums ns{0.0, 0.0, 0.0, 0.0};
            // the state (first attempt) or stage 1 from the f0 of the
            // rejected attempt
            const bool fst = __builtin_amdgcn_readfirstlane(first ? 1 : 0) != 0;
            ev.head(fst ? 0 : 1, Y, r.f0, ST, r.h, w, R);
#pragma unroll 1
            for (int stage = fst ? 0 : 1; stage < 5; ++stage) {
                r.stage = stage;
                r.st = stage == 0 ? Y : ST;
                ev.inward(r.st, w, R);
                ev.outward(r, w, R, ns);
            }
            first = false;
            const double qn = nq ? sqrt((ns.sq_other + ns.sq_quat) / nq) : 0.0;
            const double un = nu ? sqrt(ns.su / nu) : 0.0;
            const double e1 = qn >= un ? qn : un;
            double err = e1;
            bool converged = true;
            if (!(e1 > 16.0*acc) && nquat > 0) {
                const double qe = sqrt(ns.s2 / nquat);
                if (qe > projLimit) converged = false;
                else if (qe > consTol) {
                    // normalizeQuaternions (SimbodyMatterSubsystemRep.cpp:4448-4475) and
                    // the re-evaluated error norm of the projected estimate
                    ++projections;
                    double sqq = 0;
                    for (int b = 0; b < nb; ++b) {
                        const int4 ba = ldi4(body_a, b);
                        if (ba.y != BALL && ba.y != FREE) continue;
                        double qq[4], n2 = 0, e[4], d4[4];
                        for (int k = 0; k < 4; ++k) {
                            qq[k] = Y1(ba.z + k); n2 += qq[k]*qq[k];
                            e[k] = 0.2 * fabs(qq[k] - ST(ba.z + k));
                        }
                        const double n = sqrt(n2);
                        for (int k = 0; k < 4; ++k) { qq[k] = qq[k] / n; Y1(ba.z + k) = qq[k]; }
                        double d = 0;
                        for (int k = 0; k < 4; ++k) d += e[k] * qq[k];
                        for (int k = 0; k < 4; ++k) e[k] = e[k] - d*qq[k];
                        const d3 v = quat_dot_to_w(qq, e);
                        quat_dot(qq, v, d4);
                        sqq += d4[0]*d4[0] + d4[1]*d4[1] + d4[2]*d4[2] + d4[3]*d4[3];
                    }
                    const double qn2 = nq ? sqrt((ns.sq_other + sqq) / nq) : 0.0;
                    err = qn2 >= un ? qn2 : un;
                }
            }
            if (!converged) err = __builtin_inf();
            ok = adjust_step(err, acc, limited, hmin, hmax, hcur);
            if (!ok) ++rejected;
        } while (!ok);
        if (status < 0) break;
        t = t1;
        flip = !flip;
        ++accepted; ++steps;
    }
    if (flip) for (int k = 0; k < ny; ++k) S0(k) = S1(k);
    if (status == 0 && t >= tEnd) status = 1;
    a.t[lane] = t; a.h[lane] = hcur; a.status[lane] = status;
    a.stats[4*lane] = attempts; a.stats[4*lane+1] = accepted; a.stats[4*lane+2] = rejected; a.stats[4*lane+3] = projections;
}

template <class PA, bool IDF, bool HASF, bool TILE, class TC>
__global__ void __launch_bounds__(64) k_rkm_joint(RkmArgs a) {
    extern __shared__ double lds[];
    const int lane = blockIdx.x * blockDim.x + threadIdx.x;
    if (lane >= a.n_inst || a.status[lane] != 0) return;
    advance_lane<PA, IDF, HASF, TILE, TC>(a, lane, lds);
}
// Serving slots of every kind (SK_*) in one launch: a block takes the slots of
// the blockIdx.y-th kind of a.kinds, so that a request runs in the same code
// whatever its neighbours are, and different kinds run at the same time (one
// build for the whole server would be the slowest: general frames with forces).
template <class TC>
__global__ void __launch_bounds__(64) k_rkm_joint_slots(RkmArgs a) {
    extern __shared__ double lds[];
    const int lane = blockIdx.x * blockDim.x + threadIdx.x;
    int kind = 0;
    for (int k = 0, y = blockIdx.y; k < SK_N; ++k)
        if ((a.kinds >> k & 1) && y-- == 0) kind = k;
    if (lane >= a.n_inst || a.status[lane] != 0) return;
    if (slot_prm(a, ldi4(a.T.tree_a, 0).x)[JC_KIND] != (double)kind) return;
    switch (kind) {
    case 0:                  advance_lane<PrmT, false, false, true, TC>(a, lane, lds); break;
    case SK_IDF:             advance_lane<PrmT, true, false, true, TC>(a, lane, lds); break;
    case SK_FORCES:          advance_lane<PrmT, false, true, true, TC>(a, lane, lds); break;
    case SK_IDF | SK_FORCES: advance_lane<PrmT, true, true, true, TC>(a, lane, lds); break;
    }
}

// f = f(y) of the current rollout state into VF0: the derivative the
// integrator uses.
template <class PA, bool IDF, bool HASF, bool TILE>
__global__ void __launch_bounds__(64) k_joint_f0(RkmArgs a) {
    const int lane = blockIdx.x * blockDim.x + threadIdx.x;
    if (lane >= a.n_inst) return;
    const auto ev = make_eval<PA, IDF, HASF, TILE, TcG<Row<TILE>>>(a, lane, nullptr);
    const Row<TILE> base = block_rows<TILE>(a);
    ev.derivative(base.from(R_Y * a.ny_max), base.from(R_F0 * a.ny_max));
}

} // namespace joint

// Trig rows go to LDS where all wavefronts that a compute unit holds at once
// (one per SIMD, by registers) have room for them.
inline bool joint_trig_in_lds(const RkmArgs& a) {
    return a.tc_rows > 0 && a.tc_rows * 64 * 8 <= 163840 / 4;
}
template <class PA, bool IDF, bool HASF, bool TILE>
hipError_t launch_joint_f(const RkmArgs& a, hipStream_t s, bool f0_only) {
    using namespace joint;
    const dim3 grd((a.n_inst + 63)/64), blk(64);
    if (f0_only) k_joint_f0<PA, IDF, HASF, TILE><<<grd, blk, 0, s>>>(a);
    else if (joint_trig_in_lds(a)) k_rkm_joint<PA, IDF, HASF, TILE, TcL><<<grd, blk, a.tc_rows * 64 * sizeof(double), s>>>(a);
    else k_rkm_joint<PA, IDF, HASF, TILE, TcG<Row<TILE>>><<<grd, blk, 0, s>>>(a);
    return hipGetLastError();
}
inline hipError_t launch_joint_slots(const RkmArgs& a, hipStream_t s) {
    using namespace joint;
    const dim3 grd((a.n_inst + 63)/64, (unsigned)__builtin_popcount((unsigned)a.kinds)), blk(64);
    if (joint_trig_in_lds(a)) k_rkm_joint_slots<TcL><<<grd, blk, a.tc_rows * 64 * sizeof(double), s>>>(a);
    else k_rkm_joint_slots<TcG<Row<true>>><<<grd, blk, 0, s>>>(a);
    return hipGetLastError();
}
template <class PA, bool IDF, bool TILE> hipError_t launch_joint_i(const RkmArgs& a, hipStream_t s, bool f0_only) {
    return a.fapp ? launch_joint_f<PA, IDF, true, TILE>(a, s, f0_only) : launch_joint_f<PA, IDF, false, TILE>(a, s, f0_only);
}

} // namespace tdyn
