// Joint-frame constants of a body (tdyn_joint.hpp) from the PRM_* constants.
#pragma once
#include "tdyn_internal.hpp"

namespace tdyn {
namespace joint {

// The constants of a position in breadth-first blocks: arm, pitch, mass and inertia,
// offset of the body origin, R_MF last (not read where it is the identity).
enum { JP_L = 0, JP_PITCH = 3, JP_M = 4, JP_C = 5, JP_I = 8, JP_B = 14, JP_R = 18 };
// Field f of position j among nf, in pairs of a block of BW positions side by
// side.
__host__ __device__ inline int pair_at(int j, int nf, int f) {
    return (j / tgroup::BW) * (nf * tgroup::BW) + (f / 2) * (2 * tgroup::BW) + j % tgroup::BW * 2 + f % 2;
}

// Constant f of the body with PRM_* constants P and its parent's PP (null:
// Ground) in the order of the breadth-first blocks (JP_*).
__device__ inline double joint_const(const double* P, const double* PP, int f) {
    const int c = f < JP_PITCH ? JC_L + f : f == JP_PITCH ? (int)JC_PITCH : f < JP_B + 3 ? JC_M + f - JP_M
                : f >= JP_R && f < JP_R + 9 ? JC_R + f - JP_R : (int)JC_STRIDE;
    const double* p = P + PRM_P_BM;
    const double* k = P + PRM_COM;
    const double m = P[PRM_MASS];
    if (c < JC_L) {
        const int r = c / 3, j = c % 3;
        if (!PP) return P[PRM_R_PF + 3*r + j];
        return PP[PRM_R_MB + 3*r]*P[PRM_R_PF + j] + PP[PRM_R_MB + 3*r + 1]*P[PRM_R_PF + 3 + j] +
               PP[PRM_R_MB + 3*r + 2]*P[PRM_R_PF + 6 + j];
    }
    if (c < JC_M) {
        const int r = c - JC_L;
        if (!PP) return P[PRM_P_PF + r];
        double s = 0;
        for (int j = 0; j < 3; ++j) s += PP[PRM_R_MB + 3*r + j]*(P[PRM_P_PF + j] - PP[PRM_P_BM + j]);
        return s;
    }
    if (c == JC_M) return m;
    if (c < JC_I) {
        const int r = c - JC_C;
        double s = 0;
        for (int j = 0; j < 3; ++j) s += P[PRM_R_MB + 3*r + j]*(k[j] - p[j]);
        return m*s;
    }
    if (c < JC_B) {
        // unit inertia about M's origin: G + (p.p - 2 c.p) 1 - (p p^T - c p^T - p c^T), then to M axes
        double S[9];
        const double e = (p[0]*p[0] + p[1]*p[1] + p[2]*p[2]) - 2*(k[0]*p[0] + k[1]*p[1] + k[2]*p[2]);
        for (int r = 0; r < 3; ++r)
            for (int j = 0; j < 3; ++j)
                S[3*r + j] = (P[PRM_G + (r == j ? r : r + j == 1 ? 3 : r + j == 2 ? 4 : 5)] + (r == j ? e : 0.0)) -
                             (p[r]*p[j] - k[r]*p[j] - p[r]*k[j]);
        const int i = c - JC_I, r = i == 1 ? 1 : i == 2 ? 2 : i == 5 ? 1 : 0, j = i < 3 ? i : i == 3 ? 1 : 2;
        double s = 0;
        for (int x = 0; x < 3; ++x) {
            double t = 0;
            for (int y = 0; y < 3; ++y) t += S[3*x + y]*P[PRM_R_MB + 3*j + y];
            s += P[PRM_R_MB + 3*r + x]*t;
        }
        return m*s;
    }
    if (c < JC_B + 3) return P[PRM_P_MB + c - JC_B];
    return c == JC_PITCH ? P[PRM_PITCH] : 0.0;
}

} // namespace joint
} // namespace tdyn
