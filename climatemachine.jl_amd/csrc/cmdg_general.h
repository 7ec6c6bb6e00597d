// cmdg_general.h -- DG kernels for general (curvilinear) hexahedral meshes: per-node
// metric terms, per-face-node normals and surface weights, vmap+ gathers.
//
// As in the brick kernels (cmdg_affine.h) the 6 Nfp face nodes of an element are tasks of
// their own, whose results reach the node lanes through LDS in the reference's face order, and
// on a small mesh (WIDE) the tasks have waves of their own.  On the node lanes a face node's
// up to three faces ran one after the other in both waves, with the fluxes of the whole volume
// phase held in registers (166 and 182 in the tendency and the gradient, now 126 and 94).
// The same operations in the same order, so the same bits.
// Bound by memory on a large mesh (per-node metric terms and per-face-node normals: about 250
// B a node in the gradient, 390 in the tendency), by the chain of dependent reads (neighbour
// index, its state and gradient flux) on one that fits the chip at once.  us a pass, gradient
// + tendency, before -> now: 24^3 Smagorinsky-Lilly 128 + 286 -> 100 + 214, with gravity 135 +
// 312 -> 138 + 261 (a task's theta_v costs what the faces' order gave), 14^3 27.8 + 52.6 ->
// 22.8 + 42.7, N = 3 24^3 69 + 132 -> 58 + 102.  A neighbour index read one task ahead
// lengthens the registers' lives by more than it hides (14 x 12 x 10 viscous right-hand side
// 35.7 against 36.9 us with it).  A task reads its own side from memory again; with nothing in
// cache (1 GiB written between calls) the right-hand side gains as much: 14 x 12 x 10 viscous
// 52.0 -> 48.6 us, 22^3 264 -> 246, Smagorinsky-Lilly 336 -> 263, with gravity 364 -> 325.  Of the
// meshes timed one lost, warm and cold: N = 3 18^3 viscous 59.0 -> 60.1 (5832 blocks are 1.6
// rounds of the 14 a CU that LDS lets run; 12^3 24.8 -> 23.3, 22^3 105.6 -> 101.7).
#pragma once
#include "cmdg_affine.h"

namespace cmdg {

// ------------------------------------------------------------------ gradient kernel
// Lifted jump M^-1 Mf (Phi(G*) - Phi(n G-)) of face node fn of face f of element e,
// CentralNumericalFluxGradient.
// OWN as in face_gradient_aff.
template <int Nq, bool BUOY, bool OWN>
__device__ __forceinline__ void face_gradient(const KParams &P, const KArrays &A, const double *__restrict__ Q,
                                              const double *__restrict__ aux, int64_t e, int f, int fn,
                                              const double (*sG)[Nq * Nq * Nq], double *jump) {
    constexpr int Np = Nq * Nq * Nq, Nfp = Nq * Nq, NGF = BUOY ? 10 : 9;
    const int64_t idx = fn + (int64_t)Nfp * (f + 6 * e);
    const double *sgp = A.sg + 5 * idx;
    const double nv[3] = {sgp[0], sgp[1], sgp[2]};
    const double sM = sgp[3], vMI = sgp[4];
    const int vn = face_node<Nq>(f, fn);
    const bool wall = A.bnd[f + 6 * e] != 0;
    const int32_t nb = wall ? (int32_t)(e * Np + vn) : A.nbr[idx];
    const int64_t ep = nb / Np;
    const int vp = nb - (int)ep * Np;
    double qp[5], Gm[5], Gp[5], Gs[3][5], nG[3][5];
#pragma unroll
    for (int s = 0; s < 5; ++s) qp[s] = Q[(int64_t)Np * (s + 5 * ep) + vp];
    const double Php = P.a_Phi >= 0 ? aux[(int64_t)Np * (P.naux * ep + P.a_Phi) + vp] : -0.0;
    const Aux a = load_aux(P, aux, Np, vn, e);
    if (OWN) {
        double q[5];
#pragma unroll
        for (int s = 0; s < 5; ++s) q[s] = Q[(int64_t)Np * (s + 5 * e) + vn];
        const Thermo tm = thermo(P, q, a.Phi);
        grad_arg<BUOY>(P, q, tm, BUOY ? theta_v(P, tm) : 0.0, Gm);
    } else {
#pragma unroll
        for (int s = 0; s < 5; ++s) Gm[s] = (s < 4 || BUOY) ? sG[s][vn] : 0.0;
    }
    const double thv = Gm[4];
    if (wall) {
        double qb[5];
        wall_state(qp, nv, 1.0, qb);
#pragma unroll
        for (int s = 0; s < 5; ++s) qp[s] = qb[s];
    }
    const Thermo tp = thermo(P, qp, Php);
    grad_arg<BUOY>(P, qp, tp, BUOY ? theta_v(P, tp) : 0.0, Gp);
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int s = 0; s < 5; ++s) {
            Gs[d][s] = wall ? nv[d] * Gp[s] : nv[d] * (Gp[s] + Gm[s]) * 0.5;
            nG[d][s] = nv[d] * Gm[s];
        }
    double gfs[10], gfm[10];
    grad_flux<BUOY>(Gs, a, thv, gfs);
    grad_flux<BUOY>(nG, a, thv, gfm);
    const double w = vMI * sM;
#pragma unroll
    for (int s = 0; s < NGF; ++s) jump[s] = w * (gfs[s] - gfm[s]);
}

// nuo: viscosity planes (Np, viscosity_planes, nelem).  BUOY as in k_gradient_aff.
template <int Nq, bool SMAG, bool BUOY, bool WIDE>
__global__ void __launch_bounds__((block_threads<Nq, WIDE>()))
k_gradient(KParams P, KArrays A, const double *__restrict__ Q, double *__restrict__ aux,
           double *__restrict__ gfo, double *__restrict__ nuo, double *__restrict__ Qcopy, int write_aux) {
    constexpr int Np = Nq * Nq * Nq, Nfp = Nq * Nq, NV = threads_for<Nq>();
    constexpr bool buoy = SMAG && BUOY;
    constexpr int NG = buoy ? 5 : 4, NJ = buoy ? 10 : 9, NGF = SMAG ? 10 : 9, NNU = viscosity_planes(SMAG, BUOY);
    __shared__ double sD[Nq * Nq];
    __shared__ double sG[NG][Np];
    __shared__ double sJ[NJ][6 * Nfp];
    const int64_t e = xcd_element(blockIdx.x, A.nelem);
    if (e >= A.nelem) return;
    const int n = threadIdx.x;
    if (n < Nq * Nq) sD[n] = A.D[n];
    const bool act = n < Np;
    const int i = n % Nq, j = (n / Nq) % Nq, k = n / (Nq * Nq);
    double thv = 1.0, rho = 0.0;
    Aux a;
    if (act) {
        double q[5], G[5];
        const double *qb = Q + (int64_t)Np * 5 * e + n;
#pragma unroll
        for (int s = 0; s < 5; ++s) q[s] = qb[Np * s];
        if (Qcopy) {
            double *qc = Qcopy + (int64_t)Np * 5 * e + n;
#pragma unroll
            for (int s = 0; s < 5; ++s) qc[Np * s] = q[s];
        }
        rho = q[0];
        a = load_aux(P, aux, Np, n, e);
        const Thermo t = thermo(P, q, a.Phi);
        if (buoy || (write_aux && P.a_theta_v >= 0)) thv = theta_v(P, t);
        if (write_aux) {
            double *ab = aux + (int64_t)Np * P.naux * e + n;
            if (P.a_theta_v >= 0) ab[(int64_t)Np * P.a_theta_v] = thv;
            if (P.a_air_T >= 0) ab[(int64_t)Np * P.a_air_T] = t.temp;
        }
        grad_arg<buoy>(P, q, t, thv, G);
#pragma unroll
        for (int s = 0; s < NG; ++s) sG[s][n] = G[s];
    }
    if (!WIDE) __syncthreads();
    for (int t = WIDE ? (n >= NV ? n - NV : 6 * Nfp) : n; t < 6 * Nfp; t += WIDE ? 6 * Nfp : NV) {
        double J[10];
        face_gradient<Nq, buoy, WIDE>(P, A, Q, aux, e, t / Nfp, t % Nfp, sG, J);
#pragma unroll
        for (int s = 0; s < NJ; ++s) sJ[s][t] = J[s];
    }
    __syncthreads();
    if (!act) return;

    const double *vg = A.vg + (int64_t)Np * NVG * e + n;
    double xi[9];
#pragma unroll
    for (int f = 0; f < 9; ++f) xi[f] = vg[Np * f];

    // horizontal pass, then vertical pass (DGModel_kernels.jl:1007-1127, 1235-1325):
    // the gradient-flux transform is applied to each pass and the results summed
    double gG[3][5], gV[3][5];
#pragma unroll
    for (int s = 0; s < 5; ++s)
#pragma unroll
        for (int d = 0; d < 3; ++d) gG[d][s] = gV[d][s] = 0.0;
#pragma unroll
    for (int s = 0; s < NG; ++s) {
        double g1 = 0.0, g2 = 0.0, g3 = -0.0;
#pragma unroll
        for (int m = 0; m < Nq; ++m) {
            g1 += sD[i + Nq * m] * sG[s][m + Nq * (j + Nq * k)];
            g2 += sD[j + Nq * m] * sG[s][i + Nq * (m + Nq * k)];
        }
#pragma unroll
        for (int m = 0; m < Nq; ++m) g3 += sD[k + Nq * m] * sG[s][i + Nq * (j + Nq * m)];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            double v = -0.0;
            v += xi[0 + 3 * d] * g1;
            v += xi[1 + 3 * d] * g2;
            gG[d][s] = v;
            gV[d][s] = -0.0 + xi[2 + 3 * d] * g3;
        }
    }

    double gf[10], gfv[10];
    grad_flux<buoy>(gG, a, thv, gf);
    grad_flux<buoy>(gV, a, thv, gfv);
#pragma unroll
    for (int s = 0; s < NJ; ++s) gf[s] += gfv[s];

    // the lifted jumps of this node's faces, in face order
#pragma unroll
    for (int dir = 0; dir < 3; ++dir) {
        int fn;
        const int f = node_face_dir<Nq>(i, j, k, dir, fn);
        if (f < 0) continue;
#pragma unroll
        for (int s = 0; s < NJ; ++s) gf[s] += sJ[s][f * Nfp + fn];
    }
    double *go = gfo + (int64_t)Np * NGF * e + n;
#pragma unroll
    for (int s = 0; s < NJ; ++s) go[Np * s] = gf[s];
    if (SMAG) {
        if (!buoy && write_aux) go[Np * 9] = 0.0;  // N^2
        double nu[3];
        viscosity<SMAG, BUOY>(P, rho, gf, a.gPhi, a.Delta, nu);
        double *no = nuo + (int64_t)Np * NNU * e + n;
#pragma unroll
        for (int s = 0; s < NNU; ++s) no[Np * s] = nu[s];
    }
}

// ------------------------------------------------------------------ tendency kernel
// One side of a face or one node: its fluxes from the state, static fields and gradient flux.
template <int Nq, bool SMAG>
__device__ __forceinline__ void node_flux2(const KParams &P, const double *__restrict__ gfi,
                                           const double *__restrict__ nui, int nnu, int64_t e, int n,
                                           const double q[5], double F2[3][5]) {
    constexpr int Np = Nq * Nq * Nq, NGF = SMAG ? 10 : 9;
    double gf[9], nu[3];
    const double *gb = gfi + (int64_t)Np * NGF * e + n;
#pragma unroll
    for (int s = 0; s < 9; ++s) gf[s] = gb[Np * s];
    if (SMAG) {
        const double *nb = nui + (int64_t)Np * nnu * e + n;
#pragma unroll
        for (int d = 0; d < 3; ++d) nu[d] = nb[Np * (nnu == 3 ? d : 0)];
    } else {
        const double gP[3] = {0.0, 0.0, 0.0};
        viscosity<false>(P, q[0], gf, gP, 0.0, nu);
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) flux2_row<SMAG>(P, q, gf, nu, d, F2[d]);
}

// Lifted numerical flux alpha M^-1 Mf F*.n of face node fn of face f of element e
// (NumericalFluxes.jl:219-340, 670-715); alpha = 1 in MODE 1.
template <int Nq, bool DIFF, bool SMAG, int MODE>
__device__ __forceinline__ void face_flux(const KParams &P, const KArrays &A, const double *__restrict__ Q,
                                          const double *__restrict__ gfi, const double *__restrict__ nui, int nnu,
                                          const double *__restrict__ aux, int64_t e, int f, int fn, double alpha,
                                          double out[5]) {
    constexpr int Np = Nq * Nq * Nq, Nfp = Nq * Nq;
    const int64_t idx = fn + (int64_t)Nfp * (f + 6 * e);
    const double *sgp = A.sg + 5 * idx;
    const double nv[3] = {sgp[0], sgp[1], sgp[2]};
    const double w = (MODE == 0 ? alpha * sgp[4] : sgp[4]) * sgp[3];  // alpha * vMI * sM
    const int vn = face_node<Nq>(f, fn);
    const bool wall = A.bnd[f + 6 * e] != 0;
    // at a wall the element itself stands in for the neighbour
    const int32_t nb = wall ? (int32_t)(e * Np + vn) : A.nbr[idx];
    const int64_t ep = nb / Np;
    const int vp = nb - (int)ep * Np;
    double q[5], qp[5];
#pragma unroll
    for (int s = 0; s < 5; ++s) {
        q[s] = Q[(int64_t)Np * (s + 5 * e) + vn];
        qp[s] = Q[(int64_t)Np * (s + 5 * ep) + vp];
    }
    const double h[3] = {nv[0] * 0.5, nv[1] * 0.5, nv[2] * 0.5};
    double f2[5];
    if (DIFF && !wall) {
        double Fm[3][5], Fp[3][5];
        node_flux2<Nq, SMAG>(P, gfi, nui, nnu, e, vn, q, Fm);
        node_flux2<Nq, SMAG>(P, gfi, nui, nnu, ep, vp, qp, Fp);
#pragma unroll
        for (int s = 0; s < 5; ++s)
            f2[s] = ((Fm[0][s] + Fp[0][s]) * h[0] + (Fm[1][s] + Fp[1][s]) * h[1]) + (Fm[2][s] + Fp[2][s]) * h[2];
    }
    __builtin_amdgcn_sched_barrier(0);  // the second-order part leaves five values
    const double *am = aux + (int64_t)Np * P.naux * e + vn, *ap = aux + (int64_t)Np * P.naux * ep + vp;
    const double Phim = P.a_Phi >= 0 ? am[(int64_t)Np * P.a_Phi] : -0.0, Phip = P.a_Phi >= 0 ? ap[(int64_t)Np * P.a_Phi] : -0.0;
    const double refm = P.a_ref_p >= 0 ? am[(int64_t)Np * P.a_ref_p] : 0.0, refp = P.a_ref_p >= 0 ? ap[(int64_t)Np * P.a_ref_p] : 0.0;
    if (wall) wall_state(q, nv, 2.0, qp);
    const Thermo tm = thermo(P, q, Phim), tp = thermo(P, qp, Phip);
    double Fm[3][5], Fp[3][5], flux[5];
    flux1(P, q, tm.p, refm, Fm);
    flux1(P, qp, tp.p, refp, Fp);
#pragma unroll
    for (int s = 0; s < 5; ++s)
        flux[s] = -0.0 + (((Fm[0][s] + Fp[0][s]) * h[0] + (Fm[1][s] + Fp[1][s]) * h[1]) + (Fm[2][s] + Fp[2][s]) * h[2]);
    if (P.rusanov) {
        const double rim = 1.0 / q[0], rip = 1.0 / qp[0];
        const double uNm = fabs((nv[0] * (rim * q[1]) + nv[1] * (rim * q[2])) + nv[2] * (rim * q[3]));
        const double uNp = fabs((nv[0] * (rip * qp[1]) + nv[1] * (rip * qp[2])) + nv[2] * (rip * qp[3]));
        const double mw = fmax(uNm + sqrt(P.gammaR * tm.temp), uNp + sqrt(P.gammaR * tp.temp));
#pragma unroll
        for (int s = 0; s < 5; ++s) flux[s] += (mw * (q[s] - qp[s])) * 0.5;
    }
    if (DIFF && !wall)
#pragma unroll
        for (int s = 0; s < 5; ++s) flux[s] += f2[s];
#pragma unroll
    for (int s = 0; s < 5; ++s) out[s] = w * flux[s];
}

// MODE 0: tend = alpha*RHS + beta*tend.   MODE 1: LSRK stage, tend is dQ:
//   dQ <- RHS + dQ; Qout = Qin + bdt*dQ; dQ *= rka.  In MODE 1 beta = 0 says dQ holds
//   zeros (the previous stage scaled it by rka = 0) and is not read; dq_store = 0 leaves
//   the scaled dQ unstored (this stage's rka is 0 and the next stage gets beta = 0).
template <int Nq, bool DIFF, bool SMAG, int MODE, bool WIDE>
__global__ void __launch_bounds__((block_threads<Nq, WIDE>()))
k_tendency(KParams P, KArrays A, const double *__restrict__ Q, const double *__restrict__ gfi,
           const double *__restrict__ nui, int nnu, double *__restrict__ aux, double *__restrict__ tend, double alpha,
           double beta, double *__restrict__ Qout, double rka, double bdt, int write_aux, int dq_store) {
    constexpr int Np = Nq * Nq * Nq, Nfp = Nq * Nq, NV = threads_for<Nq>();
    __shared__ double sD[Nq * Nq];
    __shared__ double sF[3][5][Np];
    __shared__ double sFl[5][6 * Nfp];  // lifted face fluxes
    const int64_t e = xcd_element(blockIdx.x, A.nelem);
    if (e >= A.nelem) return;
    const int n = threadIdx.x;
    if (n < Nq * Nq) sD[n] = A.D[n];
    const bool act = n < Np;
    const int i = n % Nq, j = (n / Nq) % Nq, k = n / (Nq * Nq);
    for (int t = WIDE ? (n >= NV ? n - NV : 6 * Nfp) : n; t < 6 * Nfp; t += WIDE ? 6 * Nfp : NV) {
        double fl5[5];
        face_flux<Nq, DIFF, SMAG, MODE>(P, A, Q, gfi, nui, nnu, aux, e, t / Nfp, t % Nfp, alpha, fl5);
#pragma unroll
        for (int s = 0; s < 5; ++s) sFl[s][t] = fl5[s];
    }

    double q[5], src[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    double MI = 0.0;
    if (act) {
        const double *qb = Q + (int64_t)Np * 5 * e + n;
#pragma unroll
        for (int s = 0; s < 5; ++s) q[s] = qb[Np * s];
        const Aux a = load_aux(P, aux, Np, n, e);
        const Thermo t = thermo(P, q, a.Phi);
        if (write_aux) {
            double *ab = aux + (int64_t)Np * P.naux * e + n;
            if (P.a_theta_v >= 0) ab[(int64_t)Np * P.a_theta_v] = theta_v(P, t);
            if (P.a_air_T >= 0) ab[(int64_t)Np * P.a_air_T] = t.temp;
        }
        double F[3][5];
        flux1(P, q, t.p, a.ref_p, F);
        if (DIFF) {
            double F2[3][5];
            node_flux2<Nq, SMAG>(P, gfi, nui, nnu, e, n, q, F2);
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
                for (int s = 0; s < 5; ++s) F[d][s] += F2[d][s];
        }
        const double *vg = A.vg + (int64_t)Np * NVG * e + n;
        const double M = vg[Np * 9];
        MI = vg[Np * 10];
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            const double x1 = vg[Np * ax], x2 = vg[Np * (ax + 3)], x3 = vg[Np * (ax + 6)];
#pragma unroll
            for (int s = 0; s < 5; ++s) sF[ax][s][n] = M * ((x1 * F[0][s] + x2 * F[1][s]) + x3 * F[2][s]);
        }
        if (P.gravity) {
            // Gravity() source (tendencies_momentum.jl:60-72)
            double drho = P.ref_src ? (q[0] - a.ref_rho) : q[0];
#pragma unroll
            for (int d = 0; d < 3; ++d) src[1 + d] = (-drho) * a.gPhi[d];
        }
    }
    __syncthreads();
    if (!act) return;

    // horizontal pass (written as alpha*T + beta*tendency), then vertical pass with
    // the source added at its own level (DGModel_kernels.jl:281-306, 453-545)
    double *tb = tend + (int64_t)Np * 5 * e + n;
    double T[5];
#pragma unroll
    for (int s = 0; s < 5; ++s) {
        double th = 0.0;
#pragma unroll
        for (int m = 0; m < Nq; ++m) {
            th += MI * sD[m + Nq * i] * sF[0][s][m + Nq * (j + Nq * k)];
            th += MI * sD[m + Nq * j] * sF[1][s][i + Nq * (m + Nq * k)];
        }
        double out;
        if (MODE == 0) out = (beta != 0.0) ? alpha * th + beta * tb[Np * s] : alpha * th;
        else out = (beta != 0.0) ? th + tb[Np * s] : th;
        double tv = 0.0;
#pragma unroll
        for (int m = 0; m < Nq; ++m) {
            tv += MI * sD[m + Nq * k] * sF[2][s][i + Nq * (j + Nq * m)];
            if (m == k) tv += src[s];
        }
        T[s] = (MODE == 0 ? alpha * tv : tv) + out;
    }

    // the face fluxes of this node's faces, in face order
#pragma unroll
    for (int dir = 0; dir < 3; ++dir) {
        int fn;
        const int f = node_face_dir<Nq>(i, j, k, dir, fn);
        if (f < 0) continue;
#pragma unroll
        for (int s = 0; s < 5; ++s) T[s] -= sFl[s][f * Nfp + fn];
    }

    if (MODE == 0) {
#pragma unroll
        for (int s = 0; s < 5; ++s) tb[Np * s] = T[s];
    } else {
        double *qo = Qout + (int64_t)Np * 5 * e + n;
#pragma unroll
        for (int s = 0; s < 5; ++s) {
            qo[Np * s] = q[s] + bdt * T[s];
            if (dq_store) tb[Np * s] = T[s] * rka;
        }
    }
}

}  // namespace cmdg
