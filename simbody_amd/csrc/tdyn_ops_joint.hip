// Single-shot operators on batches of one serial chain, in joint frames
// (tdyn_joint.hpp): one lane per instance, the sweep state in registers.
//
// The record-based sweeps (k_op) write and read 0.7-1.6 kB per body between
// sweeps.  Here a sweep keeps 3 to 12 doubles per body for the next one (the
// body's angular velocity, G and DI*eps, or the force on it), the joint angles'
// sines are formed again, and rotations are recovered on the way back along the
// chain; the rest of the traffic is the arguments and the results themselves.
//
// Velocities and accelerations are not recovered from the tip's: a slow body's
// would carry the rounding of a fast outer one's.  So each body's force is
// formed on the way out, from the body's own acceleration, and kept.  (M v,
// the residual and the reactions with everything recovered: base torque of a
// two-link chain off by 7e-10 where the tip is 1e-8 of the link's mass and as
// much faster.  65,536 x 32 inverse dynamics: 180 us so, 202 as it is; M v 116
// and 178; realizeAcceleration 290 and 303.)
//
// What bounds it: at 65,536 chains the traffic (realizeAcceleration 1.26 GB at
// 4.2 TB/s, inverse dynamics 0.83 GB at 4.1, of the 4.9 a plain copy reaches;
// packed arguments at a lane stride are fetched several times), at a few chains
// the issue and the loads of single wavefronts (52 % of the cycles issuing, 45 %
// waiting).
#include "tdyn_joint.hpp"

namespace tdyn {
namespace joint {
namespace {

// One instance's part of a packed argument: base of the wavefront's first
// instance (scalar) and this lane's byte offset.
struct Pk {
    TD_GLOBAL double* b; unsigned o;
    TDJ Pk from(int r) const { return {b + r, o}; }
    TDJ TD_GLOBAL double& operator()(int k) const { return *(TD_GLOBAL double*)((TD_GLOBAL char*)(b + k) + o); }
    TDJ explicit operator bool() const { return b != nullptr; }
};
TDJ Pk packed(const double* p, size_t first, int n) {
    if (!p) return {nullptr, 0};
    return {(TD_GLOBAL double*)p + first * n, threadIdx.x * (unsigned)n * 8u};
}
// G rows of one wavefront in blocks of 64 lanes.
struct Blk {
    TD_GLOBAL double* b; unsigned o;
    TDJ Blk from(int r) const { return {b + (size_t)r * 64, o}; }
    TDJ TD_GLOBAL double& operator()(int k) const { return *(TD_GLOBAL double*)((TD_GLOBAL char*)(b + k * 64) + o); }
};
struct Tab { int y, q, u, g, gp; };        // (gp: the parent's G row)

// What a sweep needs of one body, loaded one body ahead.
struct In { double q[7], u[6], v[6], f[6], g[12], w[3]; };

enum : unsigned { LD_U = 1, LD_V = 2, LD_TAU = 4, LD_F = 8, LD_G = 16, LD_FM = 32, LD_W = 64 };
// (LD_FM: the force kept, put_force; LD_W: the parent's angular velocity, put_w)

template <bool IDF> struct Chain {
    cdptr prm, prm_g; const int4 *body_a, *body_j;
    int nb, nq, nu;
    Pk q, u, v, tau, F;         // arguments (v: udot or the vector of M v, J v)
    Pk ou, oq, ob, ob2;         // results
    Blk G;
    TDJ Tab tab(int b) const {
        const int4 a = ldi4(body_a, b - 1), j = ldi4(body_j, b - 1);
        return {a.y, a.z, a.w, j.y, j.w};
    }
    TDJ cdptr C(int b) const { return prm + (size_t)(b - 1) * PRM_STRIDE; }

    template <int T, unsigned W> TDJ void load(In& x, int b, const Tab& j) const {
        const Pk pq = q.from(j.q);
#pragma unroll
        for (int k = 0; k < Dim<T>::NQ; ++k) x.q[k] = pq(k);
        if constexpr ((W & LD_U) != 0) {
            const Pk p = u.from(j.u);
#pragma unroll
            for (int k = 0; k < Dim<T>::D; ++k) x.u[k] = p(k);
        }
        if constexpr ((W & LD_V) != 0) {
            const Pk p = v.from(j.u);
#pragma unroll
            for (int k = 0; k < Dim<T>::D; ++k) x.v[k] = v ? p(k) : 0.0;
        }
        if constexpr ((W & LD_TAU) != 0) {
            const Pk p = tau.from(j.u);
#pragma unroll
            for (int k = 0; k < Dim<T>::D; ++k) x.v[k] = tau ? p(k) : 0.0;
        }
        if constexpr ((W & LD_F) != 0) {
            if (F) {
                const Pk p = F.from(6*b);
#pragma unroll
                for (int k = 0; k < 6; ++k) x.f[k] = p(k);
            }
        }
        if constexpr ((W & LD_G) != 0) {
            const Blk g = G.from(j.g);
#pragma unroll
            for (int k = 0; k < Dim<T>::G; ++k) x.g[k] = g(k);
        }
        if constexpr ((W & LD_FM) != 0) {
            const Blk g = G.from(j.g);
#pragma unroll
            for (int k = 0; k < 6; ++k) x.g[k] = g(k);
        }
        if constexpr ((W & LD_W) != 0) {
            const Blk g = G.from(j.gp);
#pragma unroll
            for (int k = 0; k < 3; ++k) x.w[k] = g(k);
        }
    }
    // The angular velocity of body j into its G rows, where the sweep back
    // reads it before it writes G.
    TDJ void put_w(const Tab& j, const d3& w) const {
        const Blk g = G.from(j.g);
        g(0) = w.x; g(1) = w.y; g(2) = w.z;
    }
    // A force on body j (M axes) into its G rows, and out of them again.
    TDJ void put_force(const Tab& j, const wf& f) const {
        const Blk g = G.from(j.g);
        g(0) = f.w.x; g(1) = f.w.y; g(2) = f.w.z; g(3) = f.v.x; g(4) = f.v.y; g(5) = f.v.z;
    }
    static TDJ void add_kept(wf& f, const In& x) {
        f.w = f.w + d3{x.g[0], x.g[1], x.g[2]}; f.v = f.v + d3{x.g[3], x.g[4], x.g[5]};
    }
    template <unsigned W> TDJ void load_any(In& x, int b, const Tab& j) const {
        switch (j.y) {
        case PIN:       load<PIN, W>(x, b, j); break;
        case SLIDER:    load<SLIDER, W>(x, b, j); break;
        case UNIVERSAL: load<UNIVERSAL, W>(x, b, j); break;
        case BALL:      load<BALL, W>(x, b, j); break;
        default:        load<FREE, W>(x, b, j); break;
        }
    }
    // A sweep, base to tip (OUT) or back: fn(type, x, body, entry) per body,
    // the next body's values in flight meanwhile.
    template <bool OUT, unsigned W, class Fn> TDJ void sweep(const Fn& fn) const {
        In A, B;
        auto at = [&](int k) { return OUT ? k : nb + 1 - k; };
        Tab jA = tab(at(1)), jB = jA;
        load_any<W>(A, at(1), jA);
#pragma unroll 1
        for (int k = 1; k <= nb; k += 2) {
            if (k + 1 <= nb) { jB = tab(at(k + 1)); load_any<W>(B, at(k + 1), jB); }
            body(fn, A, at(k), jA);
            if (k + 1 > nb) break;
            if (k + 2 <= nb) { jA = tab(at(k + 2)); load_any<W>(A, at(k + 2), jA); }
            body(fn, B, at(k + 1), jB);
        }
    }
    template <int T> struct Type { static constexpr int t = T; };
    template <class Fn> TDJ void body(const Fn& fn, const In& x, int b, const Tab& j) const {
        switch (j.y) {
        case PIN:       fn(Type<PIN>(), x, b, j); break;
        case SLIDER:    fn(Type<SLIDER>(), x, b, j); break;
        case UNIVERSAL: fn(Type<UNIVERSAL>(), x, b, j); break;
        case BALL:      fn(Type<BALL>(), x, b, j); break;
        default:        fn(Type<FREE>(), x, b, j); break;
        }
    }
    template <int T> static TDJ Jnt<T> joint_of(const In& x) {
        double t[4];
        Jnt<T> J;
        J.trig(x.q, t); J.set(x.q, t);
        return J;
    }
    // body axes' rotation in Ground, and a body's force (Ground, at Bo) in M
    TDJ dm R_GB(const cdptr& c, const dm& R) const {
        if constexpr (IDF) return R;
        else { dm B; for (int i = 0; i < 9; ++i) B.a[i] = c[JC_RB + i]; return mul(R, B); }
    }
    static TDJ d3 Bo(const cdptr& c) { return {c[JC_B], c[JC_B + 1], c[JC_B + 2]}; }
    // Body b's own mass, first moment and inertia about Bo, M axes: from the
    // constants about Bo, as those about M have lost what the distance of the
    // joint adds (a last body of radius 0.001, its joint 3 away: 1e-10 of its
    // inertia).
    struct Own { double m; d3 mc; sym I; };
    TDJ Own own(int b) const {
        const cdptr g = prm_g + (size_t)(b - 1) * PRM_STRIDE, c = C(b);
        const double m = g[PRM_MASS];
        Own o{m, m*d3{g[PRM_COM], g[PRM_COM + 1], g[PRM_COM + 2]}, {}};
#pragma unroll
        for (int k = 0; k < 6; ++k) o.I.a[k] = m*g[PRM_G + k];
        if constexpr (!IDF) {
            dm B; for (int i = 0; i < 9; ++i) B.a[i] = c[JC_RB + i];
            o.mc = mul(B, o.mc); o.I = rot(B, o.I);
        }
        return o;
    }
    static TDJ wf force_M(const cdptr& c, const dm& R, const double* f) {
        const d3 fm = mulT(R, d3{f[3], f[4], f[5]});
        return {mulT(R, d3{f[0], f[1], f[2]}) + cross(Bo(c), fm), fm};
    }
    // (angular, linear at Bo) in Ground of (angular, linear at Mo) in M axes;
    // w: add the centripetal acceleration of Bo about Mo
    static TDJ void put_body(const Pk& o, const cdptr& c, const dm& R, const wf& A, const d3* w) {
        d3 v = A.v + cross(A.w, Bo(c));
        if (w) v = v + centripetal(*w, Bo(c));
        const d3 a = mul(R, A.w), l = mul(R, v);
        o(0) = a.x; o(1) = a.y; o(2) = a.z; o(3) = l.x; o(4) = l.y; o(5) = l.z;
    }
    static TDJ void put0(const Pk& o, int n) { for (int k = 0; k < n; ++k) o(k) = 0.0; }
};

// P - P H D^-1 H^T P about a point at b from M (M axes).
template <int T> TDJ void hinge_out(art& P, const Jnt<T>& J, const d3& b) {
    constexpr int N = Dim<T>::D;
    wf H[N], U[N];
    if constexpr (T == SLIDER) H[0] = {zero3<double>(), {1.0, 0.0, 0.0}};
    else {
        if constexpr (T == PIN) H[0].w = {0.0, 0.0, 1.0};
        else if constexpr (T == UNIVERSAL) { H[0].w = J.toB({1.0, 0.0, 0.0}); H[1].w = J.toB({0.0, 1.0, 0.0}); }
        else { H[0].w = {1.0, 0.0, 0.0}; H[1].w = {0.0, 1.0, 0.0}; H[2].w = {0.0, 0.0, 1.0}; }
        for (int k = 0; k < N; ++k) H[k].v = cross(H[k].w, b);
    }
    double D[N][N], DI[N][N];
#pragma unroll
    for (int k = 0; k < N; ++k) U[k] = {mulsym(P.J, H[k].w) + mulF(P.F, H[k].v), mulFt(P.F, H[k].w) + mulsym(P.M, H[k].v)};
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int k = 0; k < N; ++k) D[i][k] = dot(H[i].w, U[k].w) + dot(H[i].v, U[k].v);
    if constexpr (N == 1) DI[0][0] = 1.0 / D[0][0];
    else if constexpr (N == 2) {
        const double o = 1.0 / (D[0][0]*D[1][1] - D[0][1]*D[1][0]);
        DI[0][0] = o*D[1][1]; DI[1][1] = o*D[0][0]; DI[0][1] = DI[1][0] = -(o*D[0][1]);
    } else {
        const double c00 = D[1][1]*D[2][2] - D[1][2]*D[1][2], c01 = D[1][2]*D[0][2] - D[0][1]*D[2][2],
                     c02 = D[0][1]*D[1][2] - D[1][1]*D[0][2], o = 1.0 / (D[0][0]*c00 + D[0][1]*c01 + D[0][2]*c02);
        DI[0][0] = o*c00; DI[0][1] = DI[1][0] = o*c01; DI[0][2] = DI[2][0] = o*c02;
        DI[1][1] = o*(D[0][0]*D[2][2] - D[0][2]*D[0][2]);
        DI[1][2] = DI[2][1] = o*(D[0][1]*D[0][2] - D[0][0]*D[1][2]);
        DI[2][2] = o*(D[0][0]*D[1][1] - D[0][1]*D[0][1]);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        wf G{zero3<double>(), zero3<double>()};
#pragma unroll
        for (int k = 0; k < N; ++k) { G.w = G.w + DI[i][k]*U[k].w; G.v = G.v + DI[i][k]*U[k].v; }
        const double gw[3] = {G.w.x, G.w.y, G.w.z}, gv[3] = {G.v.x, G.v.y, G.v.z};
        const double uw[3] = {U[i].w.x, U[i].w.y, U[i].w.z}, uv[3] = {U[i].v.x, U[i].v.y, U[i].v.z};
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                P.F[3*r + c] -= gw[r]*uv[c];
                if (c >= r) { P.J.a[sidx(r, c)] -= gw[r]*uw[c]; P.M.a[sidx(r, c)] -= gv[r]*uv[c]; }
            }
    }
}

template <int OP, bool IDF>
__global__ void __launch_bounds__(64) k_cop(OpArgs a) {
    const int lane = blockIdx.x * 64 + threadIdx.x;
    if (lane >= a.n_inst) return;
    Chain<IDF> c;
    const int4 ta = ldi4(a.T.tree_a, 0);
    c.nb = ta.x; c.nq = ta.y; c.nu = ta.z;
    c.prm = cptr(a.T.prm_j); c.prm_g = cptr(a.T.prm); c.body_a = a.T.body_a; c.body_j = a.T.body_j;
    const size_t first = (size_t)blockIdx.x * 64;
    c.q = packed(a.q, first, c.nq); c.u = packed(a.u, first, c.nu);
    c.v = packed(a.udot_in, first, c.nu); c.tau = packed(a.fmob, first, c.nu);
    c.F = packed(a.fbody, first, 6*(c.nb + 1));
    c.ou = packed(a.out_u, first, c.nu); c.oq = packed(a.out_q, first, c.nq);
    c.G = {(TD_GLOBAL double*)a.scratch + first * a.g_rows, threadIdx.x * 8u};
    const cdptr gr = cptr(a.T.gravity);
    const d3 grav = {gr[0], gr[1], gr[2]};
    d3 w = zero3<double>();
    dm R = ident<double>();
    bool bad = false;

    if constexpr (OP == OP_FWD_SYS || OP == OP_FWD_GIVEN || OP == OP_MINV || OP == OP_REACT) {
        constexpr bool VEL = OP != OP_MINV, TAU = OP != OP_FWD_SYS, FB = OP != OP_MINV;
        const bool hasF = FB && c.F;
        if constexpr (VEL)
            c.template sweep<true, LD_U>([&](auto t, const In& x, int b, const Tab& j) {
                constexpr int T = decltype(t)::t;
                const Jnt<T> J = c.template joint_of<T>(x);
                w = out_w<T, IDF>(c.C(b), J, w, x.u);
                c.put_w(j, w);
                if (hasF) R = out_R<T, IDF>(c.C(b), J, R);
            });
        art P = zero_art(); wf z{zero3<double>(), zero3<double>()};
        c.template sweep<false, (VEL ? LD_U | LD_W : 0u) | (TAU ? LD_TAU : 0u) | (FB ? LD_F : 0u)>(
            [&](auto t, const In& x, int b, const Tab& j) {
                constexpr int T = decltype(t)::t;
                const cdptr C = c.C(b);
                const Jnt<T> J = c.template joint_of<T>(x);
                if (hasF) {
                    const wf f = c.force_M(C, R, x.f);
                    z.w = z.w - f.w; z.v = z.v - f.v;
                    R = in_R<T, IDF>(C, J, R);
                }
                double g[Dim<T>::G];
                const d3 wpar = {x.w[0], x.w[1], x.w[2]};
                bad |= in_body<T, IDF, TAU, VEL>(C, J, x.u, x.v, P, z, w, wpar, g, b == 1);
                w = wpar;
                const Blk G = c.G.from(j.g);
#pragma unroll
                for (int k = 0; k < Dim<T>::G; ++k) G(k) = g[k];
            });
        wf A{zero3<double>(), OP == OP_FWD_SYS ? -grav : zero3<double>()};
        w = zero3<double>(); R = ident<double>();
        const Pk ob = packed(a.out_body, first, 6*(c.nb + 1));
        const bool hasA = OP == OP_FWD_GIVEN && ob, hasR = hasA || OP == OP_REACT;
        c.template sweep<true, (VEL ? LD_U : 0u) | LD_G | (OP == OP_REACT ? LD_F : 0u)>([&](auto t, const In& x, int b, const Tab& j) {
            constexpr int T = decltype(t)::t;
            constexpr int D = Dim<T>::D, NQ = Dim<T>::NQ;
            const cdptr C = c.C(b);
            const Jnt<T> J = c.template joint_of<T>(x);
            double ud[D];
            out_body<T, IDF, VEL>(C, J, x.u, x.g, A, w, ud);
            if (c.ou) {
                const Pk o = c.ou.from(j.u);
#pragma unroll
                for (int k = 0; k < D; ++k) o(k) = ud[k];
            }
            if (hasR) R = out_R<T, IDF>(C, J, R);
            if constexpr (OP == OP_REACT) {
                // (G has been read)
                wf r = rigid_force<true>(C, A, w);
                if (hasF) { const wf e = c.force_M(C, R, x.f); r.w = r.w - e.w; r.v = r.v - e.v; }
                c.put_force(j, r);
            }
            if (hasA) c.put_body(ob.from(6*b), C, R, A, &w);
            if constexpr (OP == OP_FWD_SYS || OP == OP_FWD_GIVEN) {
                if (!c.oq) return;
                const Pk o = c.oq.from(j.q);
                double qd[NQ];
                const double* r = OP == OP_FWD_SYS ? x.u : ud;
                if constexpr (Dim<T>::quat) {
                    quat_dot(x.q, d3{r[0], r[1], r[2]}, qd);
                    if constexpr (OP == OP_FWD_GIVEN) {
                        const double s = -0.25 * (x.u[0]*x.u[0] + x.u[1]*x.u[1] + x.u[2]*x.u[2]);
#pragma unroll
                        for (int k = 0; k < 4; ++k) qd[k] += s*x.q[k];
                    }
                    if constexpr (T == FREE) { qd[4] = r[3]; qd[5] = r[4]; qd[6] = r[5]; }
                } else {
#pragma unroll
                    for (int k = 0; k < NQ; ++k) qd[k] = r[k];
                }
#pragma unroll
                for (int k = 0; k < NQ; ++k) o(k) = qd[k];
            }
        });
        if (hasA) c.put0(ob, 6);
        if constexpr (OP == OP_REACT) {
            // the force through each mobilizer at M, gathered tip to base
            wf f{zero3<double>(), zero3<double>()};
            c.template sweep<false, LD_FM>([&](auto t, const In& x, int b, const Tab& j) {
                constexpr int T = decltype(t)::t;
                const cdptr C = c.C(b);
                const Jnt<T> J = c.template joint_of<T>(x);
                c.add_kept(f, x);
                const d3 n = mul(R, f.w), l = mul(R, f.v);
                const Pk o = ob.from(6*b);
                o(0) = n.x; o(1) = n.y; o(2) = n.z; o(3) = l.x; o(4) = l.y; o(5) = l.z;
                f = in_force<T, IDF>(C, J, wf{J.fromB(f.w), J.fromB(f.v)}, arm<T, IDF>(C, J));
                R = in_R<T, IDF>(C, J, R);
            });
            c.put0(ob, 6);
        }
        if (a.status) a.status[lane] = bad ? 4 : 0;
    } else if constexpr (OP == OP_RESID || OP == OP_MULM || OP == OP_JAC || OP == OP_BACC || OP == OP_KIN) {
        constexpr bool VEL = OP == OP_RESID || OP == OP_BACC, OUTB = OP == OP_JAC || OP == OP_BACC || OP == OP_KIN;
        const bool hasF = OP == OP_RESID && c.F;
        wf A{zero3<double>(), zero3<double>()};
        d3 p = zero3<double>();
        double ke = 0, pe = 0;
        const Pk ob = packed(a.out_body, first, (OP == OP_KIN ? 12 : 6)*(c.nb + 1)),
                 ov = packed(a.out_body2, first, 6*(c.nb + 1));
        c.template sweep<true, (VEL || OP == OP_KIN ? LD_U : 0u) | (OP != OP_KIN ? LD_V : 0u) | (OP == OP_RESID ? LD_F : 0u)>(
            [&](auto t, const In& x, int b, const Tab& j) {
                constexpr int T = decltype(t)::t;
                const cdptr C = c.C(b);
                const Jnt<T> J = c.template joint_of<T>(x);
                if constexpr (OP == OP_KIN) p = p + mul(R, arm<T, IDF>(C, J));
                out_given<T, IDF, VEL>(C, J, x.u, OP == OP_KIN ? x.u : x.v, A, w);
                if (OUTB || hasF) R = out_R<T, IDF>(C, J, R);
                if constexpr (OP == OP_RESID || OP == OP_MULM) {
                    wf r = rigid_force<VEL>(C, A, w);
                    if (hasF) { const wf e = c.force_M(C, R, x.f); r.w = r.w - e.w; r.v = r.v - e.v; }
                    c.put_force(j, r);
                }
                if constexpr (OP == OP_JAC || OP == OP_BACC) c.put_body(ob.from(6*b), C, R, A, VEL ? &w : nullptr);
                if constexpr (OP == OP_KIN) {
                    // (about Bo, as the inertias below)
                    const auto o = c.own(b);
                    const d3 vb = A.v + cross(A.w, c.Bo(C));
                    ke += 0.5 * (dot(A.w, mulsym(o.I, A.w) + cross(o.mc, vb)) + dot(vb, o.m*vb + cross(A.w, o.mc)));
                    const d3 cm = {C[JC_C], C[JC_C + 1], C[JC_C + 2]};
                    pe -= dot(grav, C[JC_M]*p + mul(R, cm));
                    if (ob) {
                        const Pk o = ob.from(12*b);
                        const dm Rb = c.R_GB(C, R);
                        const d3 pb = p + mul(R, c.Bo(C));
                        for (int i = 0; i < 9; ++i) o(i) = Rb.a[i];
                        o(9) = pb.x; o(10) = pb.y; o(11) = pb.z;
                    }
                    if (ov) c.put_body(ov.from(6*b), C, R, A, nullptr);
                    if (c.oq) {
                        const Pk o = c.oq.from(j.q);
                        if constexpr (Dim<T>::quat) {
                            double qd[4];
                            quat_dot(x.q, d3{x.u[0], x.u[1], x.u[2]}, qd);
                            for (int k = 0; k < 4; ++k) o(k) = qd[k];
                            if constexpr (T == FREE) for (int k = 0; k < 3; ++k) o(4 + k) = x.u[3 + k];
                        } else {
#pragma unroll
                            for (int k = 0; k < Dim<T>::D; ++k) o(k) = x.u[k];
                        }
                    }
                }
            });
        if constexpr (OP == OP_JAC || OP == OP_BACC) c.put0(ob, 6);
        if constexpr (OP == OP_KIN) {
            if (ob) for (int i = 0; i < 12; ++i) ob(i) = (i == 0 || i == 4 || i == 8) ? 1.0 : 0.0;
            if (ov) c.put0(ov, 6);
            if (a.out_scalar) { a.out_scalar[2*(size_t)lane] = ke; a.out_scalar[2*(size_t)lane + 1] = pe; }
        }
        if constexpr (OP == OP_RESID || OP == OP_MULM) {
            wf f{zero3<double>(), zero3<double>()};
            c.template sweep<false, LD_FM>([&](auto t, const In& x, int b, const Tab& j) {
                constexpr int T = decltype(t)::t;
                const cdptr C = c.C(b);
                const Jnt<T> J = c.template joint_of<T>(x);
                c.add_kept(f, x);
                const wf fj{J.fromB(f.w), J.fromB(f.v)};
                double tt[Dim<T>::D];
                hinge_t<T>(J, fj, tt);
                const Pk o = c.ou.from(j.u), fm = c.tau.from(j.u);
#pragma unroll
                for (int k = 0; k < Dim<T>::D; ++k) o(k) = OP == OP_RESID && c.tau ? tt[k] - fm(k) : tt[k];
                f = in_force<T, IDF>(C, J, fj, arm<T, IDF>(C, J));
            });
        }
    } else {
        // rotations out, then back with what they re-express
        c.template sweep<true, 0u>([&](auto t, const In& x, int b, const Tab& j) {
            constexpr int T = decltype(t)::t;
            R = out_R<T, IDF>(c.C(b), c.template joint_of<T>(x), R);
        });
        if constexpr (OP == OP_JACT) {
            wf f{zero3<double>(), zero3<double>()};
            c.template sweep<false, LD_F>([&](auto t, const In& x, int b, const Tab& j) {
                constexpr int T = decltype(t)::t;
                const cdptr C = c.C(b);
                const Jnt<T> J = c.template joint_of<T>(x);
                const wf e = c.force_M(C, R, x.f);
                f.w = f.w + e.w; f.v = f.v + e.v;
                const wf fj{J.fromB(f.w), J.fromB(f.v)};
                double tt[Dim<T>::D];
                hinge_t<T>(J, fj, tt);
                const Pk o = c.ou.from(j.u);
#pragma unroll
                for (int k = 0; k < Dim<T>::D; ++k) o(k) = tt[k];
                f = in_force<T, IDF>(C, J, fj, arm<T, IDF>(C, J));
                R = in_R<T, IDF>(C, J, R);
            });
        } else if constexpr (OP == OP_ABI) {
            const Pk oP = packed(a.out_abi, first, 21*(c.nb + 1)), oPP = packed(a.out_abi2, first, 21*(c.nb + 1));
            art P = zero_art(); wf z{zero3<double>(), zero3<double>()};
            // blocks M, J (xx yy zz xy xz yz), F in Ground
            auto put = [&](const Pk& o, art X, const dm& Rg) {
                X.M = rot(Rg, X.M); X.J = rot(Rg, X.J); rot(Rg, X.F);
#pragma unroll
                for (int k = 0; k < 6; ++k) { o(k) = X.M.a[k]; o(6 + k) = X.J.a[k]; }
#pragma unroll
                for (int k = 0; k < 9; ++k) o(12 + k) = X.F[k];
            };
            c.template sweep<false, 0u>([&](auto t, const In& x, int b, const Tab& j) {
                constexpr int T = decltype(t)::t;
                const cdptr C = c.C(b);
                const Jnt<T> J = c.template joint_of<T>(x);
                {
                    // about Bo: the children's share moved there, and the body's own
                    const auto o = c.own(b);
                    art Q = P;
                    shift(Q, -c.Bo(C));
                    Q.M.a[0] += o.m; Q.M.a[1] += o.m; Q.M.a[2] += o.m;
#pragma unroll
                    for (int k = 0; k < 6; ++k) Q.J.a[k] += o.I.a[k];
                    Q.F[1] -= o.mc.z; Q.F[2] += o.mc.y; Q.F[3] += o.mc.z; Q.F[5] -= o.mc.x; Q.F[6] -= o.mc.y; Q.F[7] += o.mc.x;
                    put(oP.from(21*b), Q, R);
                    if (oPP) {
                        if constexpr (T == FREE) Q = zero_art(); else hinge_out<T>(Q, J, c.Bo(C));
                        put(oPP.from(21*b), Q, R);
                    }
                }
                double g[Dim<T>::G];
                art X = P; wf y = z;
                add_body(C, X);
                to_J<T>(J, X, y);
                bad |= eliminate<T, false>(X, y, nullptr, g);
                R = in_R<T, IDF>(C, J, R);
                to_F<T, false>(J, X, y);
                to_parent<T, IDF, false>(C, X, y, arm<T, IDF>(C, J));
                P = X;
            });
            for (int i = 0; i < 21; ++i) { oP(i) = 0.0; if (oPP) oPP(i) = 0.0; }
            if (a.status) a.status[lane] = bad ? 4 : 0;
        } else {
            // OP_CBI: composite inertias about M, carried as (m, m*com, I)
            const Pk ob = packed(a.out_body, first, 10*(c.nb + 1));
            double m = 0;
            d3 mc = zero3<double>();
            sym I = {{0, 0, 0, 0, 0, 0}};
            // about a point r before the origin
            auto move = [&](const d3& r) {
                const double rc = 2*dot(r, mc), rr = m*dot(r, r);
                I.a[0] += (rc + rr) - (2*r.x*mc.x + m*r.x*r.x);
                I.a[1] += (rc + rr) - (2*r.y*mc.y + m*r.y*r.y);
                I.a[2] += (rc + rr) - (2*r.z*mc.z + m*r.z*r.z);
                I.a[3] -= (r.x*mc.y + r.y*mc.x) + m*r.x*r.y;
                I.a[4] -= (r.x*mc.z + r.z*mc.x) + m*r.x*r.z;
                I.a[5] -= (r.y*mc.z + r.z*mc.y) + m*r.y*r.z;
                mc = mc + m*r;
            };
            c.template sweep<false, 0u>([&](auto t, const In& x, int b, const Tab& j) {
                constexpr int T = decltype(t)::t;
                const cdptr C = c.C(b);
                const Jnt<T> J = c.template joint_of<T>(x);
                {
                    // about Bo: the children's share moved there, and the body's own
                    const d3 k0 = mc; const sym I0 = I;
                    const auto own = c.own(b);
                    move(-c.Bo(C));
                    mc = mc + own.mc;
#pragma unroll
                    for (int k = 0; k < 6; ++k) I.a[k] += own.I.a[k];
                    const double mt = m + own.m, oo = 1.0/mt;
                    const d3 pc = mul(R, oo*mc);
                    const sym Ig = rot(R, I);
                    const Pk o = ob.from(10*b);
                    o(0) = mt; o(1) = pc.x; o(2) = pc.y; o(3) = pc.z;
#pragma unroll
                    for (int k = 0; k < 6; ++k) o(4 + k) = oo*Ig.a[k];
                    mc = k0; I = I0;
                }
                m += C[JC_M]; mc = mc + d3{C[JC_C], C[JC_C + 1], C[JC_C + 2]};
#pragma unroll
                for (int k = 0; k < 6; ++k) I.a[k] += C[JC_I + k];
                R = in_R<T, IDF>(C, J, R);
                const dm Rj = joint_rot<T>(J);
                mc = fromF<IDF>(C, mul(Rj, mc)); I = rot(Rj, I);
                if constexpr (!IDF) { dm Rc; for (int i = 0; i < 9; ++i) Rc.a[i] = C[JC_R + i]; I = rot(Rc, I); }
                move(arm<T, IDF>(C, J));
            });
            // Ground's entry is its infinite mass (RigidBodyNode_Weld.cpp:168-171)
            for (int i = 0; i < 10; ++i) ob(i) = i == 0 ? __builtin_inf() : (i >= 4 && i <= 6) ? 1.0 : 0.0;
        }
    }
}

template <int OP> void launch(const OpArgs& a, hipStream_t s) {
    const dim3 blk(64), grd((a.n_inst + 63) / 64);
    if (a.idf) k_cop<OP, true><<<grd, blk, 0, s>>>(a);
    else k_cop<OP, false><<<grd, blk, 0, s>>>(a);
}
} // namespace
} // namespace joint

bool launch_op_joint(OpKind k, const OpArgs& a, hipStream_t s) {
    using joint::launch;
    switch (k) {
    case OP_FWD_SYS:   launch<OP_FWD_SYS>(a, s); break;
    case OP_FWD_GIVEN: launch<OP_FWD_GIVEN>(a, s); break;
    case OP_MINV:      launch<OP_MINV>(a, s); break;
    case OP_REACT:     launch<OP_REACT>(a, s); break;
    case OP_RESID:     launch<OP_RESID>(a, s); break;
    case OP_MULM:      launch<OP_MULM>(a, s); break;
    case OP_JAC:       launch<OP_JAC>(a, s); break;
    case OP_BACC:      launch<OP_BACC>(a, s); break;
    case OP_KIN:       launch<OP_KIN>(a, s); break;
    case OP_JACT:      launch<OP_JACT>(a, s); break;
    case OP_ABI:       launch<OP_ABI>(a, s); break;
    case OP_CBI:       launch<OP_CBI>(a, s); break;
    default: return false;
    }
    return true;
}

} // namespace tdyn
