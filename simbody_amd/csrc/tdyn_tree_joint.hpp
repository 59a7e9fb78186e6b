// Level-parallel tree evaluator in joint frames (tdyn_joint.hpp): what
// GroupEval does, on padded 3-dof bodies whose recursion runs in each body's
// own mobilizer frame.  A body's joint is eliminated in its F axes; its share
// of the articulated inertia and bias force then goes to the parent's M frame
// in the child's lane, so a parent only adds its children's.  The sweeps hand
// on the angular velocity (and the rotation where body forces are given) in
// place of a pose and a velocity.
//
// What bounds it: the memory behind the records (16,384 trees: 180 MB of
// records, constants and vectors in use at a time; a rollout moves 21 GB at 4.2
// TB/s, realizeAcceleration 1.43 GB at 3.9, of the 4.9 a plain copy reaches),
// and in smaller batches the chain of steps, each a serial run of about 1,500
// instructions of one wavefront per SIMD.  Hence:
// - steps of up to G positions of the breadth-first order, cut where a
//   position's parent (child) is in the step, not at the levels: 11.1 steps
//   for a mean tree of 8 to 128 bodies and 8 lanes where the levels make 12.7;
// - tables two steps and data one step ahead of their use;
// - what parent and child hand over in an LDS ring of 2 G positions; with a
//   ring a lane knows from two indices whether the other one's entry is there;
// - one sweep inward and one outward per derivative of a rollout: the outward
//   sweep forms the next stage's state and passes on its angular velocities.
// 16,384 trees of 8 to 128 bodies with forces, 16 lanes each: realize
// acceleration 371 us (one lane per tree: 3,230); a rollout to 0.02 s 5.9 ms
// (Ground frames, three sweeps a derivative: 11.8).  With 4 / 8 / 32 lanes the
// rollout takes 13.8 / 7.9 / 7.1 ms: with fewer, more records are in use at a
// time, with more, most lanes idle.
#pragma once
#include "tdyn_joint.hpp"
#include "tdyn_joint_const.hpp"

namespace tdyn {
namespace joint {

// Record fields of one breadth-first position: the parent's angular velocity
// in F axes, trig cache and R_GM; G and DI*eps; and what a far parent or child
// reads: P and z for the parent, A, the position's own angular velocity.
// Fields lie in pairs, a pair of a block of BW positions side by side, so that
// a lane moves 16 bytes at a time and a wavefront's lanes share lines (half
// the memory instructions of single fields, at the same time per rollout).
enum { JG_W = 0, JG_TC = 3, JG_R = 7, JG_G = 16, JG_DE = 34, JG_PZ = 38, JG_A = 66, JG_WM = 72, JG_NF = 76, JG_PZ_N = 27 };
static_assert(JG_NF < tgroup::NF, "a request's record room is sized for tgroup::NF");

// A padded generic joint (any mobilizer but Free): X_FM and H_FM in F, the
// rotation as a unit quaternion (its four entries are the trig cache), which
// every mobilizer's lane turns into a matrix in the same instructions; only
// the columns' constant entries are selected by type.  With the matrices, all
// columns and the sines built in a branch per type, which a wavefront of mixed
// types walks one after the other, these took 8 of 30 thousand cycles of a
// step.  Columns 0 and 1 are (a0, 0, b0 | v0, 0, v0z) and (0, c1, d1 | hv1);
// hv1 and hv2 are used where TR, the types with two translations or one after
// a rotation.
struct Gen {
    dm R; d3 p;
    double a0, b0, v0, v0z, c1, d1;
    d3 h2, hv1, hv2;
    int d; bool turns, gimbal, tr;
    static TDJ int angles(int ty) {
        return ty == GIMBAL ? 3 : ty == UNIVERSAL ? 2
             : (ty == SLIDER || ty == TRANSLATION || ty == BALL || ty == WELD) ? 0 : 1;
    }
    static TDJ void trig(int ty, const double* q, double* tc) {
        const int na = angles(ty);
        const double x0 = na > 0 ? 0.5*q[0] : 0.0, x1 = na > 1 ? 0.5*q[1] : 0.0, x2 = na > 2 ? 0.5*q[2] : 0.0;
        double s0, c0, s1, c1, s2 = 0.0, c2 = 1.0;
        const double o = 1.0 / sqrt(q[0]*q[0] + q[1]*q[1] + q[2]*q[2] + q[3]*q[3]);
        sincos_small(x0, &s0, &c0);
        sincos_small(x1, &s1, &c1);
        if (na > 2) sincos_small(x2, &s2, &c2);
        if (big_angle(x0) || big_angle(x1) || big_angle(x2)) {
#pragma unroll 1
            for (int k = 0; k < 3; ++k) {
                double s, c;
                sincos(k == 0 ? x0 : k == 1 ? x1 : x2, &s, &c);
                if (k == 0) { s0 = s; c0 = c; } else if (k == 1) { s1 = s; c1 = c; } else { s2 = s; c2 = c; }
            }
        }
        const bool xy = na > 1, ball = ty == BALL;
        tc[0] = ball ? q[0]*o : c0*c1;
        tc[1] = ball ? q[1]*o : xy ? s0*c1 : 0.0;
        tc[2] = ball ? q[2]*o : c0*s1;
        tc[3] = ball ? q[3]*o : xy ? s0*s1 : s0;
        if (na > 2) {
            const double t0 = tc[0], t1 = tc[1], t2 = tc[2], t3 = tc[3];
            tc[0] = t0*c2 - t3*s2; tc[1] = t1*c2 + t2*s2; tc[2] = t2*c2 - t1*s2; tc[3] = t3*c2 + t0*s2;
        }
    }
    TDJ void set(int ty, const double* q, const double* tc, double pitch) {
        d = mob_dof(ty);
        const bool ball = ty == BALL, univ = ty == UNIVERSAL;
        gimbal = ty == GIMBAL; turns = univ || gimbal;
        tr = ty == TRANSLATION || ty == PLANAR || ty == CYLINDER;
        R = quat_rot(tc[0], tc[1], tc[2], tc[3]);
        v0 = ty == SLIDER || ty == TRANSLATION ? 1.0 : 0.0;
        v0z = ty == SCREW ? pitch : 0.0;
        a0 = ball || turns ? 1.0 : 0.0;
        b0 = ball || turns || v0 != 0.0 || ty == WELD ? 0.0 : 1.0;
        // (a Universal's second axis is M's y)
        c1 = ball ? 1.0 : univ ? R.a[4] : 0.0; d1 = univ ? R.a[7] : 0.0;
        h2 = {0.0, 0.0, ball ? 1.0 : 0.0};
        hv1 = hv2 = zero3<double>();
        // (selected, not multiplied: a Weld's q[0] is another body's)
        p = {v0 != 0.0 ? q[0] : 0.0, 0.0, v0z != 0.0 ? v0z*q[0] : 0.0};
        if (ty == SLIDER || ty == WELD) { R = ident<double>(); }
        if (tr) {
            if (ty == TRANSLATION) { hv1.y = 1.0; hv2.z = 1.0; p.y = q[1]; p.z = q[2]; }
            else if (ty == PLANAR) { hv1.x = 1.0; hv2.y = 1.0; p.x = q[1]; p.y = q[2]; }
            else { hv1.z = 1.0; p.z = q[1]; }
        }
        if (gimbal) {
            h2 = {R.a[2], R.a[5], R.a[8]};
            sincos_joint(q[0], &d1, &c1);
        }
    }
    TDJ d3 wrel(const double* u) const {
        return {a0*u[0] + h2.x*u[2], c1*u[1] + h2.y*u[2], (b0*u[0] + d1*u[1]) + h2.z*u[2]};
    }
    TDJ d3 vrel(const double* u) const {
        d3 v = {v0*u[0], 0.0, v0z*u[0]};
        if (tr) v = v + (u[1]*hv1 + u[2]*hv2);
        return v;
    }
    // bias of the accelerations, F axes; wp: the parent's angular velocity
    TDJ d3 bias_w(const d3& wp, const double* u) const {
        d3 a = cross(wp, wrel(u));
        const double t = turns ? u[0]*u[1] : 0.0;
        a.y -= t*d1; a.z += t*c1;
        if (gimbal) a = a + cross(d3{u[0], u[1]*c1, u[1]*d1}, u[2]*h2);
        return a;
    }
    // h_j . (w | v)
    TDJ double h0(const wf& x) const { return (a0*x.w.x + b0*x.w.z) + (v0*x.v.x + v0z*x.v.z); }
    TDJ double h1(const wf& x) const { const double s = c1*x.w.y + d1*x.w.z; return tr ? s + dot(hv1, x.v) : s; }
    TDJ double hh2(const wf& x) const { const double s = dot(h2, x.w); return tr ? s + dot(hv2, x.v) : s; }
    // a += sum of u_j h_j
    TDJ void add(const double* u, wf& a) const { a.w = a.w + wrel(u); a.v = a.v + vrel(u); }
};
TDJ d3 col(const sym& S, int j) { return {S.a[sidx(0, j)], S.a[sidx(1, j)], S.a[sidx(2, j)]}; }
template <bool IDF, class PA> TDJ d3 gen_arm(const PA& C, const Gen& J) {
    return d3{C[JC_L], C[JC_L + 1], C[JC_L + 2]} + fromF<IDF>(C, J.p);
}
template <bool IDF, class PA> TDJ d3 gen_bias_v(const PA& C, const Gen& J, const d3& w, const d3& wF, const d3& r, const double* u) {
    return toF<IDF>(C, centripetal(w, r)) + 2.0*cross(wF, J.vrel(u));
}
// As in_body; wF: the parent's angular velocity in F axes; g: G (18) and DI*eps
// (3).  ahead: called when C and u are in use no more.
template <bool IDF, class PA, class Fn>
TDJ bool gen_in(const PA& C, const Gen& J, const double* u, art& P, wf& z, const d3& wF, double* g, Fn&& ahead) {
    add_body(C, P);
    const wf b = gyro(C, mulT(J.R, wF + J.wrel(u)));
    // the body's transfer to its parent: bias accelerations (F), arm
    const d3 r = gen_arm<IDF>(C, J);
    const d3 aw = J.bias_w(wF, u), av = gen_bias_v<IDF>(C, J, fromF<IDF>(C, wF), wF, r, u);
    dm Rc;
    if constexpr (!IDF) for (int i = 0; i < 9; ++i) Rc.a[i] = C[JC_R + i];
    ahead();
    P.M = rot(J.R, P.M); P.J = rot(J.R, P.J); rot(J.R, P.F);
    z = {mul(J.R, z.w + b.w), mul(J.R, z.v + b.v)};
    wf U0, U1, U2;
    U0.w = (J.a0*col(P.J, 0) + J.b0*col(P.J, 2)) + (J.v0*colv(P.F, 0) + J.v0z*colv(P.F, 2));
    U0.v = (J.a0*row(P.F, 0) + J.b0*row(P.F, 2)) + (J.v0*col(P.M, 0) + J.v0z*col(P.M, 2));
    U1.w = J.c1*col(P.J, 1) + J.d1*col(P.J, 2);
    U1.v = J.c1*row(P.F, 1) + J.d1*row(P.F, 2);
    U2.w = mulsym(P.J, J.h2); U2.v = mulFt(P.F, J.h2);
    if (J.tr) {
        U1.w = U1.w + mulF(P.F, J.hv1); U1.v = U1.v + mulsym(P.M, J.hv1);
        U2.w = U2.w + mulF(P.F, J.hv2); U2.v = U2.v + mulsym(P.M, J.hv2);
    }
    // unused columns are zero: their D is padded with ones on the diagonal
    const double a0 = J.d > 0 ? J.h0(U0) : 1.0, a1 = J.d > 1 ? J.h1(U1) : 1.0, a2 = J.d > 2 ? J.hh2(U2) : 1.0;
    const double a3 = J.h0(U1), a4 = J.h0(U2), a5 = J.h1(U2);
    const d3 uw[3] = {U0.w, U1.w, U2.w}, uv[3] = {U0.v, U1.v, U2.v};
    const double c00 = a1*a2 - a5*a5, c01 = a5*a4 - a3*a2, c02 = a3*a5 - a1*a4;
    const double det = a0*c00 + a3*c01 + a4*c02, o = 1.0 / det;
    const double i00 = o*c00, i01 = o*c01, i02 = o*c02, i11 = o*(a0*a2 - a4*a4), i12 = o*(a3*a4 - a0*a5),
                 i22 = o*(a0*a1 - a3*a3);
    d3 gw[3], gv[3];
    gw[0] = (i00*uw[0] + i01*uw[1]) + i02*uw[2]; gv[0] = (i00*uv[0] + i01*uv[1]) + i02*uv[2];
    gw[1] = (i01*uw[0] + i11*uw[1]) + i12*uw[2]; gv[1] = (i01*uv[0] + i11*uv[1]) + i12*uv[2];
    gw[2] = (i02*uw[0] + i12*uw[1]) + i22*uw[2]; gv[2] = (i02*uv[0] + i12*uv[1]) + i22*uv[2];
    const double e[3] = {-J.h0(z), -J.h1(z), -J.hh2(z)};
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        g[6*j] = gw[j].x; g[6*j + 1] = gw[j].y; g[6*j + 2] = gw[j].z;
        g[6*j + 3] = gv[j].x; g[6*j + 4] = gv[j].y; g[6*j + 5] = gv[j].z;
    }
    g[18] = (i00*e[0] + i01*e[1]) + i02*e[2];
    g[19] = (i01*e[0] + i11*e[1]) + i12*e[2];
    g[20] = (i02*e[0] + i12*e[1]) + i22*e[2];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        z.w = z.w + e[j]*gw[j]; z.v = z.v + e[j]*gv[j];
        const double ga[3] = {gw[j].x, gw[j].y, gw[j].z}, gl[3] = {gv[j].x, gv[j].y, gv[j].z};
        const double ua[3] = {uw[j].x, uw[j].y, uw[j].z}, ul[3] = {uv[j].x, uv[j].y, uv[j].z};
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                P.F[3*r + c] -= ga[r]*ul[c];
                if (c >= r) { P.J.a[sidx(r, c)] -= ga[r]*ua[c]; P.M.a[sidx(r, c)] -= gl[r]*ul[c]; }
            }
    }
    z.w = z.w + (mulsym(P.J, aw) + mulF(P.F, av));
    z.v = z.v + (mulFt(P.F, aw) + mulsym(P.M, av));
    if constexpr (!IDF) {
        P.M = rot(Rc, P.M); P.J = rot(Rc, P.J); rot(Rc, P.F);
        z.w = mul(Rc, z.w); z.v = mul(Rc, z.v);
    }
    shift(P, r);
    z.w = z.w + cross(r, z.v);
    return !(det > 0.0);
}
// As out_body; wF as above.
template <bool IDF, class PA>
TDJ void gen_out(const PA& C, const Gen& J, const double* u, const double* g, wf& A, const d3& wF, double* ud) {
    const d3 r = gen_arm<IDF>(C, J);
    wf a;
    a.v = toF<IDF>(C, A.v + cross(A.w, r)) + gen_bias_v<IDF>(C, J, fromF<IDF>(C, wF), wF, r, u);
    a.w = toF<IDF>(C, A.w) + J.bias_w(wF, u);
#pragma unroll
    for (int j = 0; j < 3; ++j)
        ud[j] = g[18 + j] - (dot(d3{g[6*j], g[6*j + 1], g[6*j + 2]}, a.w) + dot(d3{g[6*j + 3], g[6*j + 4], g[6*j + 5]}, a.v));
    J.add(ud, a);
    A.w = mulT(J.R, a.w); A.v = mulT(J.R, a.v);
}

// A state or derivative: q (qdot) and u (udot) of one instance.
struct QU { const double *q, *u; };
struct QUW { double *q, *u; };
// What an outward sweep forms besides the derivative k: out = y + H ((c0 f0 +
// cv v) + ck k), k itself where it is kept, and err = 0.2 |out - in|.  hold:
// out is y, and the sweep only prepares the evaluation at y (in the same code,
// so that a rollout's results do not depend on where its launches end).
struct Next {
    const double *y, *f0, *v;
    double *k, *out, *err;
    double c0, cv, ck, H;
    bool hold;
};

extern __shared__ double lds_frontier[];

// IDF: every R_MF is the identity.  HASF: with body forces.
template <bool IDF, bool HASF> struct GroupJoint {
    static constexpr bool kFused = true;
    static constexpr int kFields = JG_PZ_N;       // LDS doubles per slot, 128 slots per wavefront
    static constexpr int kR = HASF ? 9 : 0;
    int nb, nq, nu, l, G, slot0;
    const int4* bfs; const int4* bfs_b; const double* con;
    double* S;
    d3 grav; const double* fapp;
    __device__ GroupJoint(const RkmArgs& a, int inst, int tr, int lane_in_group, int lanes, int group)
        : l(lane_in_group), G(lanes), slot0(group * 2 * lanes) {
        const int4 ta = ldi4(a.T.tree_a, tr);
        nb = ta.x; nq = ta.y; nu = ta.z;
        const int body_off = ta.w;
        bfs = a.T.bfs + body_off; bfs_b = a.T.bfs_b + body_off;
        con = a.T.con_bfs + a.T.lvl[ldi4(a.T.tree_b, tr).w + 1];
        // (pairs on 16 bytes: there is room to spare)
        S = a.scratch + ((a.pool ? a.pool[2*inst + 1] : (long long)inst * a.rec_stride) + 1 & ~1ll);
        const double* g = a.T.gravity + 4*tr;
        grav = V3(g[0], g[1], g[2]);
        fapp = HASF ? a.fapp + 6*(size_t)a.off.b_off[inst] : nullptr;
    }
    // Position j's record and constants; N fields of one from f (even) on.
    TDJ double* rec(int j) const { return S + pair_at(j, JG_NF, 0); }
    TDJ const double* cons(int j) const { return con + pair_at(j, JC_STRIDE, 0); }
    template <int N> static TDJ void ld(const double* r, int f, double* x) {
#pragma unroll
        for (int k = 0; k < N; k += 2) {
            const double2 v = *reinterpret_cast<const double2*>(r + (f + k) * tgroup::BW);
            x[k] = v.x;
            if (k + 1 < N) x[k + 1] = v.y;
        }
    }
    template <int N> static TDJ void sto(double* r, int f, const double* x) {
#pragma unroll
        for (int k = 0; k < N; k += 2)
            *reinterpret_cast<double2*>(r + (f + k) * tgroup::BW) = make_double2(x[k], k + 1 < N ? x[k + 1] : 0.0);
    }
    // Field k of position j in the frontier: a ring of 2 G positions, in which
    // a child's entry outlives the step of a parent at most 2 G before it.
    TDJ double& fr(int k, int j) const { return lds_frontier[128*k + slot0 + (j & (2*G - 1))]; }
    TDJ bool near(int child, int parent) const { return child - parent <= 2*G; }
    TDJ int bcast(int v, int src) const {
        return __builtin_amdgcn_ds_bpermute(4 * (((int)threadIdx.x & ~(G - 1)) | (src & (G - 1))), v);
    }
    // The lane's position at or after (before) s: position j belongs to lane j mod G.
    TDJ int own_up(int s) const { return s + ((l - s) & (G - 1)); }
    TDJ int own_down(int s) const { return s - ((s - l) & (G - 1)); }
    TDJ void tab(int j, int4& e, int4& bt) const {
        const int k = min(max(j, 0), nb - 1);
        e = ldi4(bfs, k); bt = ldi4(bfs_b, k);
    }
    // Walks the positions outward (inward): each step takes up to G of them,
    // none of them a child of another.  A lane's tables are loaded two steps
    // ahead and its data (load) one step ahead, from inside the step: body is
    // given the function that issues these loads, and calls it when it has
    // consumed its own.
    template <class D, class Load, class Body> TDJ void outward_steps(Load&& load, Body&& body) const {
        int4 e, bt, en, bn, e2 = {}, b2 = {};
        int j = own_up(0), s1, s2 = 0;
        tab(j, e, bt);
        D d;
        load(d, min(j, nb - 1), bt);
        s1 = min(G, bcast(e.z, 0));
        bool act = j < s1;
        tab(own_up(s1), en, bn);
#pragma unroll 1
        for (;;) {
            body(act, j, e, bt, d, [&] {
                s2 = min(s1 + G, bcast(en.z, s1));
                load(d, min(own_up(s1), nb - 1), bn);
                tab(own_up(s2), e2, b2);
            });
            if (s1 >= nb) break;
            j = own_up(s1); act = j < s2;
            e = en; bt = bn; en = e2; bn = b2; s1 = s2;
            grp_sync();
        }
        grp_sync();
    }
    template <class D, class Load, class Body> TDJ void inward_steps(Load&& load, Body&& body) const {
        int4 e, bt, en, bn, e2 = {}, b2 = {};
        int j = own_down(nb - 1), s1, s2 = 0;       // s1: the next step's positions end before it
        tab(j, e, bt);
        D d;
        load(d, max(j, 0), bt);
        s1 = max(nb - G, bcast(e.y, nb - 1) + 1);
        bool act = j >= s1;
        tab(own_down(s1 - 1), en, bn);
#pragma unroll 1
        for (;;) {
            body(act, j, e, bt, d, [&] {
                s2 = max(s1 - G, bcast(en.y, s1 - 1) + 1);
                load(d, max(own_down(s1 - 1), 0), bn);
                tab(own_down(s2 - 1), e2, b2);
            });
            if (s1 <= 0) break;
            j = own_down(s1 - 1); act = j >= s2;
            e = en; bt = bn; en = e2; bn = b2; s1 = s2;
            grp_sync();
        }
        grp_sync();
    }
    // q and u entries from (bt.y, bt.z) on, clamped to the vector.
    // (A tree of Welds has none: its loads read the record.)
    TDJ void ld_q(const double* q, int o, double* x) const {
        const double* p = nq > 0 ? q : S;
        const int last = max(nq - 1, 0);
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = p[min(o + k, last)];
    }
    TDJ void ld_u(const double* u, int o, double* x) const {
        const double* p = nu > 0 ? u : S;
        const int last = max(nu - 1, 0);
#pragma unroll
        for (int k = 0; k < 3; ++k) x[k] = p[min(o + k, last)];
    }
    static TDJ void mask_u(int ty, double* u) {
        const int d = mob_dof(ty);
#pragma unroll
        for (int k = 0; k < 3; ++k) u[k] = k < d ? u[k] : 0.0;
    }
    static TDJ void qdot(int ty, const double* q, const double* u, double* qd) {
        if (ty == BALL) quat_dot(q, d3{u[0], u[1], u[2]}, qd);
        else { qd[0] = u[0]; qd[1] = u[1]; qd[2] = u[2]; qd[3] = 0.0; }
    }

    // The parent's angular velocity in F axes (wF), trig cache (and rotation) of
    // position j into the record, its own angular velocity (and rotation) to its
    // children.  (wF is kept rather than w: recovered from w, a slow parent's
    // would carry the rounding of a fast body's.)
    TDJ void pass_on(int j, const int4& e, double* r, const d3& wF, const d3& w, const double* tc, const dm& R) const {
        double x[16] = {wF.x, wF.y, wF.z, tc[0], tc[1], tc[2], tc[3]};
#pragma unroll
        for (int k = 0; k < 9; ++k) x[7 + k] = HASF ? R.a[k] : 0.0;
        sto<HASF ? 16 : 8>(r, JG_W, x);
        if (e.w > 0) {
            fr(0, j) = w.x; fr(1, j) = w.y; fr(2, j) = w.z;
            if constexpr (HASF)
#pragma unroll
                for (int k = 0; k < 9; ++k) fr(3 + k, j) = R.a[k];
            // (a position's children follow each other)
            if (!near(e.z + e.w - 1, j)) {
                const double y[3] = {w.x, w.y, w.z};
                sto<3>(r, JG_WM, y);
            }
        }
    }
    TDJ void of_parent(int j, const int4& e, d3& w, dm& R) const {
        w = zero3<double>(); R = ident<double>();
        if (e.y < 0) return;
        double x[4], y[10];
        if (near(j, e.y)) {
#pragma unroll
            for (int k = 0; k < 3; ++k) x[k] = fr(k, e.y);
#pragma unroll
            for (int k = 0; k < kR; ++k) y[1 + k] = fr(3 + k, e.y);
        } else {
            const double* r = rec(e.y);
            ld<3>(r, JG_WM, x);
            if constexpr (HASF) ld<10>(r, JG_R - 1, y);
        }
        w = {x[0], x[1], x[2]};
        if constexpr (HASF)
#pragma unroll
            for (int k = 0; k < 9; ++k) R.a[k] = y[1 + k];
    }
    // X and w of the generic position j at (q, u) and its trig cache (w, R: the
    // parent's in, the position's out).
    template <class C>
    TDJ void turn(int ty, const C& K, const double* q, const double* u, double* tc, d3& wF, d3& w, dm& R) const {
        Gen J;
        Gen::trig(ty, q, tc); J.set(ty, q, tc, K[JC_PITCH]);
        wF = toF<IDF>(K, w);
        w = mulT(J.R, wF + J.wrel(u));
        if constexpr (HASF) {
            if constexpr (!IDF) { dm B; for (int k = 0; k < 9; ++k) B.a[k] = K[JC_R + k]; R = mul(R, B); }
            R = mul(R, J.R);
        }
    }
    template <class C> TDJ void turn_free(const C& K, const double* q, const double* u, double* tc, d3& w, dm& R) const {
        Jnt<FREE> J;
        tc[1] = tc[2] = tc[3] = 0.0;
        J.trig(q, tc); J.set(q, tc);
        w = out_w<FREE, IDF>(K, J, w, u);
        if constexpr (HASF) R = out_R<FREE, IDF>(K, J, R);
    }
    // The constants of a position (c), by JC_* and JC_PITCH.
    template <class K> TDJ void ld_con(const double* c, K& k, bool inertia) const {
        double x[18];
        ld<4>(c, JP_L, x);
        k[JC_L] = x[0]; k[JC_L + 1] = x[1]; k[JC_L + 2] = x[2]; k[JC_PITCH] = x[3];
        if (inertia) {
            ld<HASF ? 14 : 10>(c, JP_M, x + 4);
#pragma unroll
            for (int i = 0; i < 10; ++i) k[JC_M + i] = x[4 + i];
            if constexpr (HASF)
#pragma unroll
                for (int i = 0; i < 3; ++i) k[JC_B + i] = x[JP_B + i];
        }
        if constexpr (!IDF) {
            double y[10];
            ld<10>(c, JP_R, y);
#pragma unroll
            for (int i = 0; i < 9; ++i) k[JC_R + i] = y[i];
        }
    }

    // Trig caches, angular velocities (and rotations) at y.
    __device__ __forceinline__ void kin(const QU& y) const {
        struct D { double C[JC_STRIDE], q[4], u[3]; };
        outward_steps<D>([&](D& d, int j, const int4& bt) {
            ld_con(cons(j), d.C, false);
            ld_q(y.q, bt.y, d.q); ld_u(y.u, bt.z, d.u);
        }, [&](bool act, int j, const int4& e, const int4& bt, D& d, auto&& ahead) {
            double* r = rec(min(j, nb - 1));
            d3 w; dm R;
            of_parent(j, e, w, R);
            if (act && e.y < 0 && bt.x == FREE) {
                double q[4], u[6];
#pragma unroll
                for (int k = 0; k < 4; ++k) q[k] = y.q[bt.y + k];
#pragma unroll
                for (int k = 0; k < 6; ++k) u[k] = y.u[bt.z + k];
                double tc[4];
                turn_free(d.C, q, u, tc, w, R);
                pass_on(j, e, r, zero3<double>(), w, tc, R);
                act = false;
            }
            mask_u(bt.x, d.u);
            double tc[4];
            d3 wF;
            turn(bt.x, d.C, d.q, d.u, tc, wF, w, R);
            ahead();
            if (act) pass_on(j, e, r, wF, w, tc, R);
        });
    }

    // The inward sweep at y; true when some body's D was not positive definite.
    __device__ __forceinline__ bool inward(const QU& y) const {
        struct D { double C[JC_STRIDE], q[4], u[3], h[16], f[6]; };   // h: wF, trig cache, R
        bool bad = false;
        inward_steps<D>([&](D& d, int j, const int4& bt) {
            double* r = rec(j);
            ld_con(cons(j), d.C, true);
            ld_q(y.q, bt.y, d.q); ld_u(y.u, bt.z, d.u);
            ld<HASF ? 16 : 7>(r, JG_W, d.h);
            if constexpr (HASF) {
                const double* fb = fapp + 6*bt.w;
#pragma unroll
                for (int k = 0; k < 6; ++k) d.f[k] = fb[k];
            }
        }, [&](bool act, int j, const int4& e, const int4& bt, D& d, auto&& ahead) {
            double* r = rec(max(j, 0));
            art P = zero_art(); wf z{zero3<double>(), zero3<double>()};
            const int c1 = act ? e.z + e.w : 0;
#pragma unroll 1
            for (int c = e.z; c < c1; ++c) {
                double q[JG_PZ_N];
                if (near(c, j)) {
#pragma unroll
                    for (int k = 0; k < JG_PZ_N; ++k) q[k] = fr(k, c);
                } else {
                    ld<JG_PZ_N>(rec(c), JG_PZ, q);
                }
#pragma unroll
                for (int k = 0; k < 6; ++k) { P.M.a[k] += q[k]; P.J.a[k] += q[6 + k]; }
#pragma unroll
                for (int k = 0; k < 9; ++k) P.F[k] += q[12 + k];
                z.w = z.w + d3{q[21], q[22], q[23]};
                z.v = z.v + d3{q[24], q[25], q[26]};
            }
            grp_sync();
            const d3 wF = {d.h[0], d.h[1], d.h[2]};
            if constexpr (HASF) {
                dm R;
#pragma unroll
                for (int k = 0; k < 9; ++k) R.a[k] = d.h[JG_R + k];
                const d3 fm = mulT(R, d3{d.f[3], d.f[4], d.f[5]});
                z.w = z.w - (mulT(R, d3{d.f[0], d.f[1], d.f[2]}) + cross(d3{d.C[JC_B], d.C[JC_B + 1], d.C[JC_B + 2]}, fm));
                z.v = z.v - fm;
            }
            if (act && e.y < 0 && bt.x == FREE) {
                double q[7], u[6], g[6];
#pragma unroll
                for (int k = 0; k < 7; ++k) q[k] = y.q[bt.y + k];
#pragma unroll
                for (int k = 0; k < 6; ++k) u[k] = y.u[bt.z + k];
                Jnt<FREE> J;
                J.set(q, d.h + JG_TC);
                art P0 = P; wf z0 = z;
                const d3 w = out_w<FREE, IDF>(d.C, J, wF, u);
                bad |= in_body<FREE, IDF, false>(d.C, J, u, nullptr, P0, z0, w, wF, g, true);
                sto<6>(r, JG_G, g);
                act = false;
            }
            mask_u(bt.x, d.u);
            Gen J;
            J.set(bt.x, d.q, d.h + JG_TC, d.C[JC_PITCH]);
            double g[21];
            bad |= gen_in<IDF>(d.C, J, d.u, P, z, wF, g, ahead) && act;
            if (act) {
                sto<21>(r, JG_G, g);
                if (e.y >= 0) {
                    const double q[JG_PZ_N] = {P.M.a[0], P.M.a[1], P.M.a[2], P.M.a[3], P.M.a[4], P.M.a[5],
                                               P.J.a[0], P.J.a[1], P.J.a[2], P.J.a[3], P.J.a[4], P.J.a[5],
                                               P.F[0], P.F[1], P.F[2], P.F[3], P.F[4], P.F[5], P.F[6], P.F[7], P.F[8],
                                               z.w.x, z.w.y, z.w.z, z.v.x, z.v.y, z.v.z};
                    if (near(j, e.y)) {
#pragma unroll
                        for (int k = 0; k < JG_PZ_N; ++k) fr(k, j) = q[k];
                    } else {
                        sto<JG_PZ_N>(r, JG_PZ, q);
                    }
                }
            }
        });
        return bad;
    }

    // The outward sweep at y (after kin and inward).  NEXT: the state n.out
    // that the derivative leads to, and its own caches, angular velocities and
    // rotations; otherwise the derivative itself to f.
    template <bool NEXT> __device__ __forceinline__ void outward(const QU& y, const QUW& f, const Next& n) const {
        struct D { double C[JC_STRIDE], q[4], u[3], h[8], g[22]; };
        constexpr int A0 = NEXT ? 3 + kR : 0;       // A's place in the frontier
        outward_steps<D>([&](D& d, int j, const int4& bt) {
            double* r = rec(j);
            ld_con(cons(j), d.C, false);
            ld_q(y.q, bt.y, d.q); ld_u(y.u, bt.z, d.u);
            ld<7>(r, JG_W, d.h);
            ld<21>(r, JG_G, d.g);
        }, [&](bool act, int j, const int4& e, const int4& bt, D& d, auto&& ahead) {
            double* r = rec(min(j, nb - 1));
            double yq[21];
            if constexpr (NEXT) {
                // (used at the step's end)
                ld_q(n.y, bt.y, yq); ld_u(n.y + nq, bt.z, yq + 4);
                ld_q(n.f0, bt.y, yq + 7); ld_u(n.f0 + nq, bt.z, yq + 11);
                ld_q(n.v, bt.y, yq + 14); ld_u(n.v + nq, bt.z, yq + 18);
            }
            wf A{zero3<double>(), -grav};
            if (e.y >= 0) {
                if (near(j, e.y)) A = {{fr(A0, e.y), fr(A0 + 1, e.y), fr(A0 + 2, e.y)},
                                       {fr(A0 + 3, e.y), fr(A0 + 4, e.y), fr(A0 + 5, e.y)}};
                else {
                    double x[6];
                    ld<6>(rec(e.y), JG_A, x);
                    A = {{x[0], x[1], x[2]}, {x[3], x[4], x[5]}};
                }
            }
            auto hand_on = [&](const wf& A1) {
                if (e.w > 0) {
                    const double x[6] = {A1.w.x, A1.w.y, A1.w.z, A1.v.x, A1.v.y, A1.v.z};
#pragma unroll
                    for (int k = 0; k < 6; ++k) fr(A0 + k, j) = x[k];
                    // (a position's children follow each other)
                    if (!near(e.z + e.w - 1, j)) sto<6>(r, JG_A, x);
                }
            };
            if (act && e.y < 0 && bt.x == FREE) {
                double q[7], u[6], g[6], k1[13];
#pragma unroll
                for (int k = 0; k < 7; ++k) q[k] = y.q[bt.y + k];
#pragma unroll
                for (int k = 0; k < 6; ++k) { u[k] = y.u[bt.z + k]; g[k] = d.g[k]; }
                Jnt<FREE> J;
                J.set(q, d.h + JG_TC);
                wf A1 = A; d3 w1 = zero3<double>();
                out_body<FREE, IDF>(d.C, J, u, g, A1, w1, k1 + 7);
                hand_on(A1);
                quat_dot(q, d3{u[0], u[1], u[2]}, k1);
                k1[4] = u[3]; k1[5] = u[4]; k1[6] = u[5];
                if constexpr (NEXT) {
                    double x[13], s[13];
                    auto o = [&](int k) { return k < 7 ? bt.y + k : nq + bt.z + k - 7; };
#pragma unroll
                    for (int k = 0; k < 13; ++k) { x[k] = n.y[o(k)]; s[k] = n.c0*n.f0[o(k)] + n.cv*n.v[o(k)]; }
#pragma unroll
                    for (int k = 0; k < 13; ++k) if (!n.hold) x[k] += n.H*(s[k] + n.ck*k1[k]);
#pragma unroll
                    for (int k = 0; k < 13; ++k) {
                        n.out[o(k)] = x[k];
                        if (n.k) n.k[o(k)] = k1[k];
                        if (n.err) n.err[o(k)] = 0.2*fabs(x[k] - (k < 7 ? q[k] : u[k - 7]));
                    }
                    d3 w0 = zero3<double>(); dm R0 = ident<double>();
                    double tc[4];
                    turn_free(d.C, x, x + 7, tc, w0, R0);
                    pass_on(j, e, r, zero3<double>(), w0, tc, R0);
                } else {
                    if (f.q)
#pragma unroll
                        for (int k = 0; k < 7; ++k) f.q[bt.y + k] = k1[k];
#pragma unroll
                    for (int k = 0; k < 6; ++k) f.u[bt.z + k] = k1[7 + k];
                }
                act = false;
            }
            mask_u(bt.x, d.u);
            Gen J;
            J.set(bt.x, d.q, d.h + JG_TC, d.C[JC_PITCH]);
            double k1[7];
            qdot(bt.x, d.q, d.u, k1);
            gen_out<IDF>(d.C, J, d.u, d.g, A, d3{d.h[0], d.h[1], d.h[2]}, k1 + 4);
            const int nqb = mob_nq(bt.x), nub = J.d;
            if constexpr (NEXT) {
                double x[7], er[7];
#pragma unroll
                for (int k = 0; k < 7; ++k) {
                    x[k] = yq[k] + n.H*((n.c0*yq[7 + k] + n.cv*yq[14 + k]) + n.ck*k1[k]);
                    if (n.hold) x[k] = yq[k];
                    er[k] = 0.2*fabs(x[k] - (k < 4 ? d.q[k] : d.u[k - 4]));
                }
                double K[JC_STRIDE];
                for (int k = 0; k < JC_STRIDE; ++k) K[k] = d.C[k];
                ahead();
                if (act) {
                    hand_on(A);
                    auto put = [&](double* v, const double* y7) {
#pragma unroll
                        for (int k = 0; k < 4; ++k) if (k < nqb) v[bt.y + k] = y7[k];
#pragma unroll
                        for (int k = 0; k < 3; ++k) if (k < nub) v[nq + bt.z + k] = y7[4 + k];
                    };
                    put(n.out, x);
                    if (n.k) put(n.k, k1);
                    if (n.err) put(n.err, er);
                }
                mask_u(bt.x, x + 4);
                double tc[4];
                d3 wF, w; dm R;
                of_parent(j, e, w, R);
                turn(bt.x, K, x, x + 4, tc, wF, w, R);
                if (act) pass_on(j, e, r, wF, w, tc, R);
            } else {
                ahead();
                if (act) {
                    hand_on(A);
                    if (f.q)
#pragma unroll
                        for (int k = 0; k < 4; ++k) if (k < nqb) f.q[bt.y + k] = k1[k];
#pragma unroll
                    for (int k = 0; k < 3; ++k) if (k < nub) f.u[bt.z + k] = k1[4 + k];
                }
            }
        });
    }
    // f = (qdot, udot) of y; true when some body's D was not positive definite.
    __device__ __forceinline__ bool derivs(const QU& y, const QUW& f) const {
        kin(y);
        const bool bad = inward(y);
        outward<false>(y, f, Next{});
        return bad;
    }
};

} // namespace joint
} // namespace tdyn
