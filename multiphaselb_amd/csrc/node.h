// The time step of one node in the reference's own arithmetic: force, velocity, the MRT
// collisions and the heat source from values already in registers.  Shared by the
// per-routine kernels, the fused passes and the small-lattice kernel, so that all of them
// round alike; every expression keeps the reference's association order and the files
// that include this are built with -ffp-contract=off.
#pragma once

#include "kernels.h"
#include "physics.h"

namespace mplb {

// interForce.c:16-39 with interactionForce.c:47-79: psin[k] is psi at the downstream node
// x + c_k, psic the node's own; a node with a missing link feels no interaction force
template <class L, typename T>
__device__ inline void node_force(const EosParams& e, const T* psin, T psic, bool interior, T* Ff) {
    T F[3] = {T(0.0), T(0.0), T(0.0)};
    Ff[0] = Ff[1] = Ff[2] = T(0);
    if (!interior) return;
#pragma unroll
    for (int k = 1; k < L::Q; k++) {
        const T alpha = T(L::t.w[k]) * psin[k];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const int c = L::t.c[k][i];
            if (c == 1) F[i] += alpha;
            else if (c == -1) F[i] += -alpha;
        }
    }
    const T beta = -T(e.G) * psic;
#pragma unroll
    for (int i = 0; i < 3; i++) Ff[i] = F[i] * beta;
}

// total force of interForce.c:30-39
template <typename T>
__device__ inline void node_total_force(const EosParams& e, const T* Ff, T rho, T rho0, bool interior, T* Ft) {
#pragma unroll
    for (int j = 0; j < 3; j++) {
        T ft = Ff[j] + (rho - rho0) * T(e.g[j]);
        if (interior) ft += T(e.fext[j]);
        Ft[j] = ft;
    }
}

// liMRTSurfaceTension.c:11-132 (D2Q9) / xuMRTSurfaceTension.c:57-122 (D3Q15) of a node
// with every link present
template <class L, typename T>
__device__ inline void node_surface_tension(const EosParams& e, const ModelParams& mp, const T* psin, T psi, T* C) {
#pragma unroll
    for (int k = 0; k < L::Q; k++) C[k] = T(0);
    T Qt[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll
    for (int k = 1; k < L::Q; k++) {
        const T alpha = T(L::t.w[k]) * (psin[k] - psi);
#pragma unroll
        for (int i = 0; i < L::D; i++)
#pragma unroll
            for (int j = (L::D == 2 ? 0 : i); j < L::D; j++) {
                const int cc = L::t.c[k][i] * L::t.c[k][j];
                if (cc == 1) Qt[i][j] += alpha;
                else if (cc == -1) Qt[i][j] += -alpha;
            }
    }
    const T G = T(e.G), kap = T(mp.kappa);
#pragma unroll
    for (int i = 0; i < L::D; i++)
#pragma unroll
        for (int j = (L::D == 2 ? 0 : i); j < L::D; j++) Qt[i][j] = Qt[i][j] * T(0.5) * psi * G * kap;
    if (L::D == 2) {
        C[1] = T(1.5) * T(mp.Lambda[1]) * (Qt[0][0] + Qt[1][1]);
        C[2] = T(-1.5) * T(mp.Lambda[2]) * (Qt[0][0] + Qt[1][1]);
        C[7] = -T(mp.Lambda[8]) * (Qt[0][0] - Qt[1][1]);
        C[8] = -T(mp.Lambda[8]) * Qt[0][1];
    } else {
        C[1] = T(4.0) * T(mp.Lambda[1]) * (Qt[0][0] + Qt[1][1] + Qt[2][2]) / T(5.0);
        const T l10 = -T(mp.Lambda[10]);
        C[9] = l10 * (T(2) * Qt[0][0] - Qt[1][1] - Qt[2][2]);
        C[10] = l10 * (Qt[1][1] - Qt[2][2]);
        C[11] = l10 * Qt[0][1];
        C[12] = l10 * Qt[1][2];
        C[13] = l10 * Qt[0][2];
    }
}

// liMRTCollision.c:33-106 with liMRTForce.c:13-42 (D2Q9): F the total force, Fi the
// interaction force, C the surface-tension moments when mp.surf
template <class L, typename T>
__device__ inline void node_collide_limrt(const ModelParams& mp, T* fv, T rho, const T* U, const T* F, T Fi0, T Fi1,
                                          T psi, const T* C) {
    T m[L::Q], meq[L::Q], S[L::Q];
    T umag = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) umag += U[k] * U[k];
    meq[0] = rho;
    meq[1] = rho * (T(-2) + T(3) * umag);
    meq[2] = rho * (T(1) - T(3) * umag);
    meq[3] = rho * U[0];
    meq[4] = rho * (-U[0]);
    meq[5] = rho * U[1];
    meq[6] = rho * (-U[1]);
    meq[7] = rho * (U[0] * U[0] - U[1] * U[1]);
    meq[8] = rho * U[0] * U[1];
    moments<L, T>(fv, m);
    const T sigma = T(mp.sigma);
    const T L1 = T(mp.Lambda[1]), L2 = T(mp.Lambda[2]);
    S[0] = 0;
    S[1] = T(6) * (U[0] * F[0] + U[1] * F[1]) +
           T(12) * sigma * (Fi0 * Fi0 + Fi1 * Fi1) / (psi * psi * ((T(1) / L1) - T(0.5)));
    S[2] = T(-6) * (U[0] * F[0] + U[1] * F[1]) -
           T(12) * sigma * (Fi0 * Fi0 + Fi1 * Fi1) / (psi * psi * ((T(1) / L2) - T(0.5)));
    S[3] = F[0];
    S[4] = -F[0];
    S[5] = F[1];
    S[6] = -F[1];
    S[7] = T(2) * (U[0] * F[0] - U[1] * F[1]);
    S[8] = U[0] * F[1] + U[1] * F[0];
#pragma unroll
    for (int k = 0; k < L::Q; k++) {
        const T lam = T(mp.Lambda[k]);
        m[k] = m[k] - lam * (m[k] - meq[k]) + (T(1) - T(0.5) * lam) * S[k];
        if (mp.surf) m[k] = m[k] + C[k];
    }
    populations<L, T>(m, fv);
}

// xuMRTCollision.c:42-92 with xuMRTEquilibriumMS.c:23-51 and xuMRTForce.c:18-69 (D3Q15)
template <class L, typename T>
__device__ inline void node_collide_xumrt(const EosParams& e, const ModelParams& mp, T* fv, T rho, const T* U,
                                          const T* Fi, T psi, T rho0, const T* C) {
    T m[L::Q], meq[L::Q], S[L::Q];
    T umag = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) umag += U[k] * U[k];
    meq[0] = rho;
    meq[1] = rho * (T(-1.0) + umag);
    meq[2] = rho * (T(1.0) - T(5.0) * umag);
    meq[3] = rho * U[0];
    meq[4] = rho * T(-7.0) * U[0] / T(3.0);
    meq[5] = rho * U[1];
    meq[6] = rho * T(-7.0) * U[1] / T(3.0);
    meq[7] = rho * U[2];
    meq[8] = rho * T(-7.0) * U[2] / T(3.0);
    meq[9] = rho * (T(2.0) * U[0] * U[0] - U[1] * U[1] - U[2] * U[2]);
    meq[10] = rho * (U[1] * U[1] - U[2] * U[2]);
    meq[11] = rho * U[0] * U[1];
    meq[12] = rho * U[1] * U[2];
    meq[13] = rho * U[0] * U[2];
    meq[14] = 0;
    moments<L, T>(fv, m);
    T F[3];
#pragma unroll
    for (int j = 0; j < 3; j++) F[j] = Fi[j] + (rho - rho0) * T(e.g[j]);
    const T uDotF = U[0] * F[0] + U[1] * F[1] + U[2] * F[2];
    T fmag = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) fmag += F[k] * F[k];
    const T sigma = T(mp.sigma), L1 = T(mp.Lambda[1]);
    S[0] = 0;
    S[1] = T(2.0) * uDotF + (T(6.0) * sigma * fmag) / (psi * psi * ((T(1) / L1) - T(0.5)));
    S[2] = T(-10.0) * uDotF;
    S[3] = F[0];
    S[4] = T(-7.0) * F[0] / T(3.0);
    S[5] = F[1];
    S[6] = T(-7.0) * F[1] / T(3.0);
    S[7] = F[2];
    S[8] = T(-7.0) * F[2] / T(3.0);
    S[9] = T(4.0) * U[0] * F[0] - T(2.0) * U[1] * F[1] - T(2.0) * U[2] * F[2];
    S[10] = T(2.0) * U[1] * F[1] - T(2.0) * U[2] * F[2];
    S[11] = U[0] * F[1] + U[1] * F[0];
    S[12] = U[1] * F[2] + U[2] * F[1];
    S[13] = U[0] * F[2] + U[2] * F[0];
    S[14] = 0;
#pragma unroll
    for (int k = 0; k < L::Q; k++) {
        const T lam = T(mp.Lambda[k]);
        m[k] = m[k] - lam * (m[k] - meq[k]) + (T(1) - T(0.5) * lam) * S[k];
        if (mp.surf) m[k] = m[k] + C[k];
    }
    populations<L, T>(m, fv);
}

// liTempMRTCollision.c:31-84 with liTempMRTEquilibriumMS.c:20-41, liTempMRTSource.c:17-24
template <class L, typename T>
__device__ inline void node_collide_litemp(const ModelParams& mp, T* gv, T temp, const T* U, T ss) {
    T n[L::Q], neq[L::Q];
#pragma unroll
    for (int k = 0; k < L::Q; k++) neq[k] = T(0);
    neq[0] = temp;
    neq[1] = T(-2.0) * temp;
    neq[2] = T(2.0) * temp;
    neq[3] = temp * U[0];
    neq[4] = temp * (-U[0]);
    neq[5] = temp * U[1];
    neq[6] = temp * (-U[1]);
    moments<L, T>(gv, n);
    const T n4 = n[4], n6 = n[6];
#pragma unroll
    for (int k = 0; k < L::Q; k++) {
        const T lam = T(mp.Lambda[k]);
        const T gam = (k == 0) ? ss : T(0);
        n[k] = n[k] - lam * (n[k] - neq[k]) + gam;
    }
    n[3] = n[3] + (T(1) - T(mp.Lambda[3]) / T(2)) * T(mp.Lambda[4]) * n4;
    n[5] = n[5] + (T(1) - T(mp.Lambda[5]) / T(2)) * T(mp.Lambda[6]) * n6;
    populations<L, T>(n, gv);
}

// myMRTCollision.c:35-212 with myMRTEquilibriumMS.c:20-77 and sparseMatVecMult.c:11-28:
// Q = diag(Lambda) + Q34, Q56 (, Q78), Q_aux = I - Q/2; n <- n - Q (n - n_eq) + Q_aux Gamma.
template <class L, typename T>
__device__ inline void node_collide_my(const ModelParams& mp, T* gv, T temp, const T* U, T gam0) {
    T n[L::Q], neq[L::Q], aux1[L::Q], aux2[L::Q];
#pragma unroll
    for (int k = 0; k < L::Q; k++) neq[k] = T(0);
    neq[0] = temp;
    neq[1] = T(mp.alpha1) * temp;
    neq[2] = T(mp.alpha2) * temp;
    if (L::D == 2) {
        neq[3] = temp * U[0];
        neq[4] = temp * (-U[0]);
        neq[5] = temp * U[1];
        neq[6] = temp * (-U[1]);
    } else {
        neq[3] = temp * U[0];
        neq[4] = -(temp * U[0]);
        neq[5] = temp * U[1];
        neq[6] = -(temp * U[1]);
        neq[7] = temp * U[2];
        neq[8] = -(temp * U[2]);
    }
    moments<L, T>(gv, n);
    // relaxation matrix entries (myMRTCollision.c:39-127), computed as the reference does
    T Qd[L::Q], Qa[L::Q];
#pragma unroll
    for (int k = 0; k < L::Q; k++) {
        Qd[k] = T(mp.Lambda[k]);
        Qa[k] = T(1.0) + T(-0.5) * Qd[k];
    }
    const int npair = L::D == 2 ? 2 : 3;
    T Qo[3], Qao[3];
#pragma unroll
    for (int pr = 0; pr < 3; pr++) {
        const int a = 3 + 2 * pr, b = 4 + 2 * pr;
        Qo[pr] = Qd[b] * (Qd[a] / T(2.0) - T(1.0));
        Qao[pr] = T(-0.5) * Qo[pr];
    }
#pragma unroll
    for (int k = 0; k < L::Q; k++) aux2[k] = n[k] - neq[k];
#pragma unroll
    for (int k = 0; k < L::Q; k++) aux1[k] = Qd[k] * aux2[k];
#pragma unroll
    for (int pr = 0; pr < npair; pr++) aux1[3 + 2 * pr] = aux1[3 + 2 * pr] + Qo[pr] * aux2[4 + 2 * pr];
#pragma unroll
    for (int k = 0; k < L::Q; k++) aux2[k] = Qa[k] * (k == 0 ? gam0 : T(0));
#pragma unroll
    for (int pr = 0; pr < npair; pr++) aux2[3 + 2 * pr] = aux2[3 + 2 * pr] + Qao[pr] * T(0);
#pragma unroll
    for (int k = 0; k < L::Q; k++) n[k] = n[k] - aux1[k] + aux2[k];
    populations<L, T>(n, gv);
}

// macroVelocity.c:17-50 with liMRTVelocity.c:11-50 / xuMRTVelocity.c:19-50, component j
template <class L, typename T>
__device__ inline T node_velocity(const T* fv, T rho, T F, int j) {
    T lv = 0;
#pragma unroll
    for (int k = 0; k < L::Q; k++) {
        const int c = L::t.c[k][j];
        if (c == 1) lv += fv[k];
        else if (c == -1) lv += -fv[k];
    }
    return (lv + F * T(0.5)) / rho;
}

// sum of the populations in index order (macroDensity.c:19-60, myMRTTemperature.c:16-30)
template <class L, typename T>
__device__ inline T node_sum(const T* v) {
    T r = 0;
#pragma unroll
    for (int k = 0; k < L::Q; k++) r += v[k];
    return r;
}

// finiteDifference/{scalarGradient,invScalarGradient,vectorDivergence}.c along one axis:
// qa at x + e (ha: present), qb at x - e (hb), qi the node's own value
template <typename T>
__device__ inline T node_fd(T qa, bool ha, T qb, bool hb, T qi, bool inv) {
    if (ha && hb) {
        const T a = inv ? T(1.0) / qa : qa;
        const T b = inv ? T(1.0) / qb : qb;
        return T(0.5) * (a - b);
    }
    if (!ha && hb) {
        const T i = inv ? T(1.0) / qi : qi;
        const T b = inv ? T(1.0) / qb : qb;
        return i - b;
    }
    if (ha && !hb) {
        const T a = inv ? T(1.0) / qa : qa;
        const T i = inv ? T(1.0) / qi : qi;
        return a - i;
    }
    return T(0);
}

// heatSource.c:26-170 after the stencils: dot = grad T . grad 1/rho, divU; old T, new rho
template <class L, typename T>
__device__ inline T node_heat(const EosParams& e, const ModelParams& mp, T rho, T temp, T dot, T divU) {
    const T Cv = T(e.Cv);
    const T L3 = T(mp.Lambda[3]);
    T lambda;
    if (mp.model == M_MYMRT) {
        if (L::D == 2)
            lambda = rho * Cv * (T(1) / L3 - T(0.5)) * (T(4.0) + T(3.0) * T(mp.alpha1) + T(2.0) * T(mp.alpha2)) / T(6.0);
        else
            lambda = rho * Cv * (T(1) / L3 - T(0.5)) * (T(6.0) + T(11.0) * T(mp.alpha1) + T(mp.alpha2)) / T(9.0);
    } else {
        lambda = rho * Cv * (T(1) / L3 - T(0.5));
    }
    T dpdT = p_eos<T>(e, rho, T(1.1) * temp) - p_eos<T>(e, rho, T(0.9) * temp);
    dpdT = dpdT / (T(0.2) * temp);
    return -lambda * dot / Cv + divU * temp * (T(1.0) - dpdT / (rho * Cv));
}

// bounceBack.c:14-75 on a node's populations; miss[k]: link k has no upstream node
template <class L, typename T>
__device__ inline void node_bounce_back(T* v, const bool* miss) {
#pragma unroll
    for (int k = 0; k < L::Q; k++) {
        const int r = L::t.rev[k];
        if (miss[k]) {
            v[k] = v[r];
        } else if (!miss[r] && k >= 1 && k <= L::naxis) {
            v[k] = T(0.5) * v[k] + T(0.5) * v[r];
            v[r] = v[k];
        }
    }
}

// population k of the energy field's equilibrium (myMRTEquilibrium.c:5-95,
// liTempMRTEquilibrium.c:5-44)
template <class L, typename T>
__device__ inline T node_geq(const ModelParams& mp, int k, T temp, const T* U) {
    T geq[L::Q];
    if (mp.model == M_MYMRT) my_geq<L, T>(temp, U, T(mp.alpha1), T(mp.alpha2), geq);
    else litemp_geq<L, T>(temp, U, geq);
    return geq[k];
}

}  // namespace mplb
