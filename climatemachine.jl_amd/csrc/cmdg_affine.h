// cmdg_affine.h -- DG kernels for meshes of axis-aligned affine bricks.
//
// The context detects (bitwise, at cmdg_create) that every element's metric terms
// are a constant diagonal d xi / d x, that M = J * W[n] and sM = sJ_f * Wf[fn] with
// the tensor-product LGL weights, that face normals are +-e_d and that face
// neighbours are conforming (vmap+ = the opposite face of one element).  Geometry
// then shrinks from 11 doubles per node plus 5 per face node to 11 doubles and 6
// ints per element, and every product with an exactly-zero metric or normal
// component of the general formula is dropped; for finite data this changes no
// result bit.
//
// A face reads its neighbour's state and gradient flux straight from the neighbour's
// volume (25 values per face and variable; the kernels that update the state write it to
// another buffer than the one they read).  The static fields (Phi, p_ref), where the two
// sides differ, reach a face through a face trace written once at set-up: a face-major
// array (nelem, 6, nvar, Nfp) in which the 25 values a neighbour needs for one face and
// one variable are contiguous.
#pragma once
#include "cmdg_physics.h"

namespace cmdg {

// per-element record: xi11, xi22, xi33, J, sJ (6 faces), Delta
constexpr int AFF_GEO = 11;
// entries a face node
constexpr int TR_F2 = 4;  // a second-order flux row: states 1..4 (the mass entry is 0)
constexpr int TR_S = 2;   // Phi, p_ref

struct AffArrays {
    const double *geo;    // (nelem, AFF_GEO)
    const int32_t *nbe;   // (nelem, 6) neighbour element across face f, -1 at a wall
    const double *W;      // (Np)  (w_k w_j) w_i
    const double *Wf;     // (Nfp) w_b w_a for face node a + Nq b
    const double *D;      // (Nq, Nq)
    const double *str;    // (nelem, 6, TR_S, Nfp) static trace
    int32_t aux_cont;     // 1: Phi and p_ref agree bitwise on both sides of every interior face
    // Static auxiliary fields (Phi, grad Phi, rho_ref, p_ref, Delta): elements whose
    // static fields agree bitwise share one class, and the kernels read those fields
    // from the class's block of sa, (Np, naux, nclass) in the aux layout.  Without
    // classes, cls is null and sa is the aux array itself (class = element).
    const int32_t *cls;   // (nelem) class of each element, or null
    const double *sa;
    const float *gphi32;  // (Np, 3, nclass) grad Phi rounded to FP32 (mixed path; null without it)
};

// the class whose static fields element e reads
__device__ __forceinline__ int64_t static_class(const AffArrays &A, int64_t e) {
    return A.cls ? (int64_t)A.cls[e] : e;
}

// The elements one launch works on: the range first .. first + count - 1, or, with a
// list, list[0 .. count - 1].  Block b takes the element at position xcd_element(b, count):
// each XCD gets one contiguous run of the set.
struct ElemSet {
    const int32_t *list;
    int64_t first, count;
};
__device__ __forceinline__ int64_t set_element(const ElemSet &S, int64_t b) {
    const int64_t p = xcd_element(b, S.count);
    if (p >= S.count) return -1;
    return S.list ? (int64_t)S.list[p] : S.first + p;
}

template <int Nfp> __device__ __forceinline__ int64_t tri(int64_t e, int f, int v, int nv, int fn) {
    return ((e * 6 + f) * nv + v) * (int64_t)Nfp + fn;
}

// volume node of face node fn = a + Nq b of face f (the inverse of node_face_dir): the
// coordinate along the face's normal is 0 or N, the other two are (a, b) in order.
// Selects rather than a switch: the face tasks of one wave lie on up to three faces, and
// a switch over f branches once per face present.
template <int Nq> __device__ __forceinline__ int face_node(int f, int fn) {
    const int a = fn % Nq, b = fn / Nq, d = f >> 1, o = (f & 1) * (Nq - 1);
    const int i = d == 0 ? o : a;
    const int j = d == 1 ? o : (d == 0 ? a : b);
    const int k = d == 2 ? o : b;
    return i + Nq * (j + Nq * k);
}

// Face work is spread over all lanes of the workgroup: the 6 Nfp face nodes are
// tasks t = f Nfp + fn dealt round-robin (150 tasks on 128 lanes at N = 4 take 2 + 1
// wave-iterations, where one lane per volume node would run its up-to-3 faces in 3 +
// 3), each task's result goes to LDS, and each node then adds the results of its
// faces in face order (the reference's order).

// On a mesh too small to fill the chip (WIDE) a block has waves of their own for the face
// tasks, one lane a task, which run beside the volume waves instead of after them.
template <int Nq> constexpr int face_threads() { return (6 * Nq * Nq + 63) / 64 * 64; }
template <int Nq, bool WIDE> constexpr int block_threads() {
    return threads_for<Nq>() + (WIDE ? face_threads<Nq>() : 0);
}

// A static auxiliary field (Phi, p_ref) at volume node vn of element e, or dflt when
// the model has no such field.
template <int Nq>
__device__ __forceinline__ double own_aux(const KParams &P, const double *__restrict__ aux, int64_t e, int vn,
                                          int field, double dflt) {
    constexpr int Np = Nq * Nq * Nq;
    return field >= 0 ? aux[(int64_t)Np * (P.naux * e + field) + vn] : dflt;
}

// ------------------------------------------------------------------ gradient
// Lifted central jumps n (G* - G-) of face node fn of face f of element e
// (DGModel_kernels.jl:1471-1647, CentralNumericalFluxGradient NumericalFluxes.jl:67-123,
// walls: G* = n G(q_wall), bc_momentum.jl:24-43).  G- and theta_v- come from the element's
// own gradient arguments in LDS, q+ from the neighbour's volume state.  A normal along axis d
// fills row d of the gradient only, so four values carry the whole jump of the gradient
// flux: u_c and h_tot here, and with a gravitational potential the fifth, N^2's
// (row d of grad theta_v . grad Phi / theta_v); jump_gradient_flux spreads them.
// OWN: the element's own gradient argument is formed here from its state (the operations of
// its volume lanes, so their bits) instead of read from sG.
template <int Nq, bool SMAG, bool BUOY, bool OWN>
__device__ __forceinline__ void face_gradient_aff(const KParams &P, const AffArrays &A, int64_t e, int f, int fn,
                                                  int32_t ne, const double *__restrict__ Q,
                                                  const double (*sG)[Nq * Nq * Nq], double jump[5]) {
    constexpr int Np = Nq * Nq * Nq, Nfp = Nq * Nq;
    constexpr bool buoy = SMAG && BUOY;
    const int d = f >> 1, vn = face_node<Nq>(f, fn);
    const double nd = (f & 1) ? 1.0 : -1.0;
    const int64_t ce = static_class(A, e);
    double G[5], Gp[5], Gs[5], qm[5];
    if (OWN) {
#pragma unroll
        for (int s = 0; s < 5; ++s) qm[s] = Q[(int64_t)Np * (s + 5 * e) + vn];
        const Thermo t = thermo(P, qm, own_aux<Nq>(P, A.sa, ce, vn, P.a_Phi, -0.0));
        grad_arg<buoy>(P, qm, t, buoy ? theta_v(P, t) : 0.0, G);
    } else {
#pragma unroll
        for (int s = 0; s < 5; ++s) G[s] = (s < 4 || buoy) ? sG[s][vn] : 0.0;
    }
    if (ne >= 0) {
        const int fo = f ^ 1;
        // the neighbour's state at the shared node, from its volume (the gradient pass
        // writes no state, so every block reads the stage's state)
        double qp[5];
        const int64_t qb = (int64_t)Np * 5 * ne + face_node<Nq>(fo, fn);
#pragma unroll
        for (int s = 0; s < 5; ++s) qp[s] = Q[qb + Np * s];
        const double Php = A.aux_cont ? own_aux<Nq>(P, A.sa, ce, vn, P.a_Phi, -0.0) : A.str[tri<Nfp>(ne, fo, 0, TR_S, fn)];
        Thermo tp = thermo(P, qp, Php);
        grad_arg<buoy>(P, qp, tp, buoy ? theta_v(P, tp) : 0.0, Gp);
#pragma unroll
        for (int s = 0; s < 5; ++s) Gs[s] = nd * (Gp[s] + G[s]) * 0.5;
    } else {
        double q[5], qb[5];
#pragma unroll
        for (int s = 0; s < 5; ++s) q[s] = Q[(int64_t)Np * (s + 5 * e) + vn];
        const double Phi = own_aux<Nq>(P, A.sa, ce, vn, P.a_Phi, -0.0);
        const double nv[3] = {d == 0 ? nd : 0.0, d == 1 ? nd : 0.0, d == 2 ? nd : 0.0};
        wall_state(q, nv, 1.0, qb);
        Thermo tb = thermo(P, qb, Phi);
        grad_arg<buoy>(P, qb, tb, buoy ? theta_v(P, tb) : 0.0, Gp);
#pragma unroll
        for (int s = 0; s < 5; ++s) Gs[s] = nd * Gp[s];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) jump[s] = Gs[s] - nd * G[s];
    if (buoy) {
        const double gPd = A.sa[(int64_t)Np * (P.naux * ce + P.a_gPhi + d) + vn];
        jump[4] = (Gs[4] * gPd) / G[4] - ((nd * G[4]) * gPd) / G[4];
    }
}

// Adds w times the gradient-flux jump of a face along axis d (compile-time after unrolling)
// to gf: the transform of a gradient with row d alone.  Halving is exact, so these are the
// bits of transforming both sides and subtracting.
template <bool BUOY>
__device__ __forceinline__ void jump_gradient_flux(int d, double w, const double J[5], double *gf) {
    gf[d] += w * J[3];
    if (d == 0) {
        gf[3] += w * J[0];
        gf[4] += w * (J[1] * 0.5);
        gf[5] += w * (J[2] * 0.5);
    } else if (d == 1) {
        gf[4] += w * (J[0] * 0.5);
        gf[6] += w * J[1];
        gf[7] += w * (J[2] * 0.5);
    } else {
        gf[5] += w * (J[0] * 0.5);
        gf[7] += w * (J[1] * 0.5);
        gf[8] += w * J[2];
    }
    if (BUOY) gf[9] += w * J[4];
}

// Viscosity planes (Np, viscosity_planes, nelem) beside the FP64 gradient flux: nu_d of
// Smagorinsky-Lilly, 3 under a gravitational potential (the buoyancy correction makes it
// anisotropic), 1 without; none for a constant viscosity, which the tendency has at hand.
constexpr int viscosity_planes(bool smag, bool buoy) { return smag ? (buoy ? 3 : 1) : 0; }

// BUOY: as for k_gradient_mix, theta_v and its gradient are evaluated for N^2 only when
// the context has a gravitational potential.  Without one N^2 is zero, and its plane of the
// gradient flux (which no kernel reads) is written with the auxiliary refresh only, in the
// last pass of a call.
// Bound by memory: 40 B a node read, 80 written, and the neighbours' lines.  It writes no
// face trace: the tendency forms the neighbour's second-order row from the gradient flux
// and the viscosity planes (8 B a node), where a trace of rows took 38.4 B a node written
// here and read there; and a face's jump is the four or five values that differ from zero,
// 4.8-6 KB of LDS instead of 12.  48^3 Smagorinsky-Lilly: 697 -> 579 us a launch (the
// tendency 1005 -> 1017), 25^3 with gravity 120 -> 106 (151 -> 151), 33^3 constant
// viscosity 242 -> 199 (338 -> 366).  Register caps of 96 and 80 spill (15 and 37
// registers) and cost 763 and 1173 us at 48^3.
// The neighbours and the derivative matrix are read on every lane, not under a branch: its
// end waits for what it read (and stored to LDS) before the state is even asked for, two
// round trips a block.  In the tendency, likewise, every field of the node is asked for before
// anything is waited for.  us, gradient + tendency: 48^3 Smagorinsky-Lilly 582 + 972 -> 554 +
// 955, 33^3 constant viscosity 196 + 341 -> 183 + 334, 25^3 with gravity 107.8 + 147.9 ->
// 104.5 + 146.5.  Now, traced over warm calls: 555 + 937, 180 + 324, 105.6 + 143.0; the gradient
// moves 189 B a node at 48^3, 4.7 TB/s.  The face waves of a wide block read their own
// neighbour and fill the time (128 elements the same or 1 us a step slower so), so there the
// matrix stays under its branch.
template <int Nq, bool SMAG, bool BUOY, bool WIDE>
__global__ void __launch_bounds__((block_threads<Nq, WIDE>()))
k_gradient_aff(KParams P, AffArrays A, ElemSet ES, const double *__restrict__ Q, double *__restrict__ aux,
               double *__restrict__ gfo, double *__restrict__ nuo, double *__restrict__ Qcopy, int write_aux) {
    constexpr int Np = Nq * Nq * Nq, Nfp = Nq * Nq, NV = threads_for<Nq>();
    constexpr bool buoy = SMAG && BUOY;
    constexpr int NG = buoy ? 5 : 4, NGF = SMAG ? 10 : 9, NNU = viscosity_planes(SMAG, BUOY);
    __shared__ double sD[Nq * Nq];
    __shared__ double sG[NG][Np];
    __shared__ double sJ[NG][6 * Nfp];  // lifted jumps of the face nodes
    const int64_t e = set_element(ES, blockIdx.x);
    if (e < 0) return;
    __shared__ int32_t nb[6];  // the element's face neighbours
    const int n = threadIdx.x;
    int32_t nbn = 0;
    double Dn = 0.0;
    if (WIDE) {
        if (n < Nq * Nq) sD[n] = A.D[n];
    } else {  // on every lane (see above)
        nbn = A.nbe[6 * e + min(n, 5)];
        Dn = A.D[min(n, Nq * Nq - 1)];
    }
    const bool act = n < Np;
    const int i = n % Nq, j = (n / Nq) % Nq, k = n / (Nq * Nq);
    const double *ge = A.geo + (int64_t)AFF_GEO * e;
    double rho = 0.0, thv = 1.0;
    Aux a;
    if (act) {
        const double *qb = Q + (int64_t)Np * 5 * e + n;
        double q[5], G[5];
#pragma unroll
        for (int s = 0; s < 5; ++s) q[s] = qb[Np * s];
        if (Qcopy)  // the step's working copy of the state: written once, next read a pass later
#pragma unroll
            for (int s = 0; s < 5; ++s) __builtin_nontemporal_store(q[s], Qcopy + (int64_t)Np * (s + 5 * e) + n);
        rho = q[0];
        a = load_aux(P, A.sa, Np, n, static_class(A, e));
        Thermo t = thermo(P, q, a.Phi);
        // theta_v enters N^2 = grad theta_v . grad Phi / theta_v only, zero without a
        // gravitational potential (grad Phi = 0): then it is evaluated only for the aux
        // refresh
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
    if (!WIDE && n < 6) nb[n] = nbn;
    if (!WIDE && n < Nq * Nq) sD[n] = Dn;
    // lifted central jumps of all face nodes, spread over every lane (WIDE: over the face
    // waves, meanwhile)
    if (WIDE) {
        const int t = n - NV;
        if (t >= 0 && t < 6 * Nfp) {
            double J[5];
            face_gradient_aff<Nq, SMAG, BUOY, true>(P, A, e, t / Nfp, t % Nfp, A.nbe[6 * e + t / Nfp], Q, sG, J);
#pragma unroll
            for (int s = 0; s < NG; ++s) sJ[s][t] = J[s];
        }
    } else {
        __syncthreads();
        for (int t = n; t < 6 * Nfp; t += NV) {
            double J[5];
            face_gradient_aff<Nq, SMAG, BUOY, false>(P, A, e, t / Nfp, t % Nfp, nb[t / Nfp], Q, sG, J);
#pragma unroll
            for (int s = 0; s < NG; ++s) sJ[s][t] = J[s];
        }
    }
    __syncthreads();

    if (act) {
        // horizontal pass then vertical pass, transform applied to each and summed
        const double xi0 = ge[0], xi1 = ge[1], xi2 = ge[2];
        double gf[10], gH[3][5], gV[3][5];
#pragma unroll
        for (int s = 0; s < 5; ++s) {
            double g1 = 0.0, g2 = 0.0, g3 = -0.0;
            if (s < NG) {
#pragma unroll
                for (int m = 0; m < Nq; ++m) {
                    g1 += sD[i + Nq * m] * sG[s][m + Nq * (j + Nq * k)];
                    g2 += sD[j + Nq * m] * sG[s][i + Nq * (m + Nq * k)];
                }
#pragma unroll
                for (int m = 0; m < Nq; ++m) g3 += sD[k + Nq * m] * sG[s][i + Nq * (j + Nq * m)];
            }
            gH[0][s] = xi0 * g1;
            gH[1][s] = xi1 * g2;
            gH[2][s] = 0.0;
            gV[0][s] = 0.0;
            gV[1][s] = 0.0;
            gV[2][s] = xi2 * g3;
        }
        double tmp[10];
        grad_flux<buoy>(gH, a, thv, gf);
        grad_flux<buoy>(gV, a, thv, tmp);
#pragma unroll
        for (int s = 0; s < (buoy ? 10 : 9); ++s) gf[s] += tmp[s];
        // the lifted jumps of this node's faces, in face order: M^-1 Mf (...)
        const double MI = 1.0 / (ge[3] * A.W[n]);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            int fn;
            const int f = node_face_dir<Nq>(i, j, k, d, fn);
            if (f < 0) continue;
            const double w = MI * (ge[4 + f] * A.Wf[fn]);
            double J[5];
#pragma unroll
            for (int s = 0; s < NG; ++s) J[s] = sJ[s][f * Nfp + fn];
            jump_gradient_flux<buoy>(d, w, J, gf);
        }
        double *go = gfo + (int64_t)Np * NGF * e + n;
#pragma unroll
        for (int s = 0; s < (buoy ? 10 : 9); ++s) go[Np * s] = gf[s];
        if (SMAG) {
            if (!buoy && write_aux) go[Np * 9] = 0.0;  // N^2
            double nu[3];
            viscosity<SMAG, BUOY>(P, rho, gf, a.gPhi, ge[10], nu);
            double *no = nuo + (int64_t)Np * NNU * e + n;
#pragma unroll
            for (int s = 0; s < NNU; ++s) no[Np * s] = nu[s];
        }
    }
}

// ------------------------------------------------------------------ tendency
// Numerical flux (first + second order, Rusanov or central) at face node fn of face
// f of element e, seen from e (normal +-e_d): NumericalFluxes.jl:219-340, 670-715,
// walls bc_momentum.jl:24-49 / bc_energy.jl:10-17 (zero second-order flux).
// The neighbour's second-order row is formed here from its gradient flux and viscosity at
// the shared node (the strain-rate row, d h_tot / d x_d, nu_d; WithDivergence the two other
// diagonal entries): the operations, and so the bits, of the neighbour's own row.
// OWN: the element's own side is read from memory and its second-order row formed here too
// (its volume lanes' bits again); otherwise its state is staged in sQ and the row is f2own.
template <int Nq, bool DIFF, int NNU, bool OWN>
__device__ __forceinline__ void face_flux_aff(const KParams &P, const AffArrays &A, int64_t e, int64_t ce, int f,
                                              int fn, int32_t ne, const double (*sQ)[Nq * Nq * Nq], const double *__restrict__ Q,
                                              const double *__restrict__ gfi, const double *__restrict__ nui,
                                              const double *f2own, double flux[5]) {
    constexpr bool SMAG = NNU > 0;
    constexpr int NGF = SMAG ? 10 : 9;
    constexpr int Np = Nq * Nq * Nq, Nfp = Nq * Nq;
    const int d = f >> 1, vn = face_node<Nq>(f, fn);
    const double nd = (f & 1) ? 1.0 : -1.0;
    const double h = nd * 0.5;
    const bool wall = ne < 0;
    const int fo = f ^ 1;
    // the own state at the face's volume node; the neighbour's from its volume
    double q[5], qp[5];
#pragma unroll
    for (int s = 0; s < 5; ++s) q[s] = OWN ? Q[(int64_t)Np * (s + 5 * e) + vn] : sQ[s][vn];
    const double Phi = own_aux<Nq>(P, A.sa, ce, vn, P.a_Phi, -0.0);
    const double ref_p = own_aux<Nq>(P, A.sa, ce, vn, P.a_ref_p, 0.0);
    double Php = Phi, refpp = ref_p;
    // the neighbour's strain-rate row, trace, viscosity and enthalpy gradient, loaded with
    // its state
    double S0 = 0.0, S1 = 0.0, S2 = 0.0, trS = 0.0, nud = 0.0, gd = 0.0;
    if (!wall) {
        const double *qb = Q + (int64_t)Np * 5 * ne + face_node<Nq>(fo, fn);
#pragma unroll
        for (int s = 0; s < 5; ++s) qp[s] = qb[Np * s];
        if (DIFF) {
            const int vp = face_node<Nq>(fo, fn);
            const double *gn = gfi + (int64_t)Np * NGF * ne + vp;
            S0 = gn[Np * pick3(d, 3, 4, 5)];
            S1 = gn[Np * pick3(d, 4, 6, 7)];
            S2 = gn[Np * pick3(d, 5, 7, 8)];
            gd = gn[Np * d];
            if (SMAG) nud = nui[(int64_t)Np * (NNU * (int64_t)ne + (NNU == 3 ? d : 0)) + vp];
            else if (P.with_div) trS = (gn[Np * 3] + gn[Np * 6]) + gn[Np * 8];
        }
        if (!A.aux_cont) {
            Php = A.str[tri<Nfp>(ne, fo, 0, TR_S, fn)];
            refpp = A.str[tri<Nfp>(ne, fo, 1, TR_S, fn)];
        }
    } else {
        const double nv[3] = {d == 0 ? nd : 0.0, d == 1 ? nd : 0.0, d == 2 ? nd : 0.0};
        wall_state(q, nv, 2.0, qp);
    }
    // the second-order part first: it leaves four values of the neighbour's six
    double f2[TR_F2];
    if (DIFF && !wall) {
        double F2p[5];
        if (!SMAG) {
            const double g0[1] = {0.0}, gP[3] = {0.0, 0.0, 0.0};
            double nu[3];
            viscosity<false>(P, qp[0], g0, gP, 0.0, nu);
            nud = nu[0];
        }
        flux2_row_parts<SMAG>(P, qp, S0, S1, S2, trS, nud, gd, d, F2p);
        double F2m[5];
        if (OWN) {
            const double *gm = gfi + (int64_t)Np * NGF * e + vn;
            const double g0[1] = {0.0}, gP[3] = {0.0, 0.0, 0.0};
            double nu[3];
            if (SMAG) nu[0] = nui[(int64_t)Np * (NNU * e + (NNU == 3 ? d : 0)) + vn];
            else viscosity<false>(P, q[0], g0, gP, 0.0, nu);
            const double tr = !SMAG && P.with_div ? (gm[Np * 3] + gm[Np * 6]) + gm[Np * 8] : 0.0;
            flux2_row_parts<SMAG>(P, q, gm[Np * pick3(d, 3, 4, 5)], gm[Np * pick3(d, 4, 6, 7)],
                                  gm[Np * pick3(d, 5, 7, 8)], tr, nu[0], gm[Np * d], d, F2m);
        }
#pragma unroll
        for (int v = 0; v < TR_F2; ++v) f2[v] = ((OWN ? F2m[1 + v] : f2own[v]) + F2p[1 + v]) * h;
    }
    __builtin_amdgcn_sched_barrier(0);
    const Thermo tm = thermo(P, q, Phi);
    const Thermo tp = thermo(P, qp, Php);
    const double rim = 1.0 / q[0], rip = 1.0 / qp[0];
    const double u[3] = {div_by(q[1], q[0], rim), div_by(q[2], q[0], rim), div_by(q[3], q[0], rim)};
    const double up[3] = {div_by(qp[1], qp[0], rip), div_by(qp[2], qp[0], rip), div_by(qp[3], qp[0], rip)};
    double Fm[5], Fp[5];
    flux1_row(q, u, tm.p, P.ref_sub ? (tm.p - ref_p) : tm.p, d, Fm);
    flux1_row(qp, up, tp.p, P.ref_sub ? (tp.p - refpp) : tp.p, d, Fp);
#pragma unroll
    for (int s = 0; s < 5; ++s) flux[s] = (Fm[s] + Fp[s]) * h;
    if (P.rusanov) {
        const double qmd = pick3(d, q[1], q[2], q[3]);
        const double qpd = pick3(d, qp[1], qp[2], qp[3]);
        const double wm = fabs(nd * (rim * qmd)) + sqrt(P.gammaR * tm.temp);
        const double wp = fabs(nd * (rip * qpd)) + sqrt(P.gammaR * tp.temp);
        const double mw = fmax(wm, wp);
#pragma unroll
        for (int s = 0; s < 5; ++s) flux[s] += (mw * (q[s] - qp[s])) * 0.5;
    }
    if (DIFF && !wall)
#pragma unroll
        for (int v = 0; v < TR_F2; ++v) flux[1 + v] += f2[v];
}

// MODE 0: tend = alpha*RHS + beta*tend.   MODE 1: LSRK stage (tend is dQ):
//   dQ <- RHS + dQ; Qout = Qin + bdt*dQ; dQ *= rka.  Qout is another buffer than Q:
//   blocks read their neighbours' volume state.  MODE 1 takes alpha = 1 and beta = 1,
//   or beta = 0 when dQ holds zeros (the previous stage scaled it by rka = 0): it is then
//   not read; dq_store = 0 leaves the scaled dQ unstored (this stage's rka is 0 and the
//   next stage is launched with beta = 0).
// NNU: viscosity planes of nui (Smagorinsky-Lilly; 0: a constant viscosity).
// What bounds it: nothing alone.  At 48^3 (Smagorinsky-Lilly) the lines that miss L2 are 319 B
// a node read and 80 written, 5.9 TB/s; VALU issues in 48 % of the cycles, LDS in 29 %; each
// wave waits 63 % of its life, so waves are what helps.  The horizontal fluxes share
// one LDS space with the vertical ones and the staged state that follow them, and a face
// node's own row shares its slot with the flux (16.2 KB a block; three directions at once
// took 20.0), which with the second-order part of a face taken first (94 registers, 110-122
// before) lets 5 waves a SIMD run instead of 4.  48^3: 1017 -> 965 us a launch, 33^3 constant
// viscosity 366 -> 341, 25^3 with gravity 150.5 -> 147.5 (now, with what the gradient pass's note
// adds, 937, 324 and 143).  Fewer blocks a CU (LDS padding, 4 waves): 8 / 7 / 6 / 5 give 1010 / 1065 / 1150 / 1475 us; nine spilled registers 1332.  Face
// tasks first, both sides read from memory instead of LDS, cut the missed lines to 213 B and
// cost 1069 us: the added vector-memory instructions weigh more.
// At Nq = 4 five waves spill.
template <int Nq, bool DIFF, int NNU, int MODE, bool WIDE>
__global__ void __launch_bounds__((block_threads<Nq, WIDE>()))
__attribute__((amdgpu_waves_per_eu(WIDE ? 1 : Nq == 5 ? 5 : 4)))
k_tendency_aff(KParams P, AffArrays A, ElemSet ES, const double *__restrict__ Q,
               const double *__restrict__ gfi, const double *__restrict__ nui, double *__restrict__ aux,
               double *__restrict__ tend, double alpha, double beta, double *__restrict__ Qout, double rka,
               double bdt, int write_aux, int dq_store) {
    constexpr int Np = Nq * Nq * Nq, Nfp = Nq * Nq, NV = threads_for<Nq>();
    constexpr bool SMAG = NNU > 0;
    constexpr int NGF = SMAG ? 10 : 9;
    __shared__ double sD[Nq * Nq];
    // M(xi_a F) of the two horizontal directions; then, once every lane has its horizontal
    // divergence, of the vertical one (in [0]) and the element's state for the face tasks
    // (in [1])
    __shared__ double sF[2][5][Np];
    double(*sQ)[Np] = sF[1];
    // per face node: this element's second-order row, then the face flux in its place
    __shared__ double sFl[6 * Nfp][5];
    const int64_t e = set_element(ES, blockIdx.x);
    if (e < 0) return;
    __shared__ int32_t nb[6];  // the element's face neighbours
    const int n = threadIdx.x;
    int32_t nbn = 0;
    double Dn = 0.0;
    if (WIDE) {
        if (n < Nq * Nq) sD[n] = A.D[n];
    } else {  // on every lane (see above)
        nbn = A.nbe[6 * e + min(n, 5)];
        Dn = A.D[min(n, Nq * Nq - 1)];
    }
    const bool act = n < Np;
    const int i = n % Nq, j = (n / Nq) % Nq, k = n / (Nq * Nq);
    const double *ge = A.geo + (int64_t)AFF_GEO * e;

    const int64_t ce = static_class(A, e);
    double q[5], gf[9], u[3], nu[3], Fv[5], MI = 0.0;
    if (WIDE) {
        const int t = n - NV;
        if (t >= 0 && t < 6 * Nfp) {
            double fl5[5];
            face_flux_aff<Nq, DIFF, NNU, true>(P, A, e, ce, t / Nfp, t % Nfp, A.nbe[6 * e + t / Nfp], nullptr, Q, gfi,
                                               nui, nullptr, fl5);
#pragma unroll
            for (int s = 0; s < 5; ++s) sFl[t][s] = fl5[s];
        }
    }
    if (act) {
        const double *qb = Q + (int64_t)Np * 5 * e + n;
#pragma unroll
        for (int s = 0; s < 5; ++s) q[s] = qb[Np * s];
        // all of the node's fields before the first is waited for: the branch below would
        // hold the rest back (WIDE: the other waves fill the time, the registers count more)
        if (DIFF && !WIDE) {
            const double *gb = gfi + (int64_t)Np * NGF * e + n;
#pragma unroll
            for (int s = 0; s < 9; ++s) gf[s] = gb[Np * s];
            if (SMAG) {
                const double *nb_ = nui + (int64_t)Np * NNU * e + n;
#pragma unroll
                for (int d = 0; d < 3; ++d) nu[d] = nb_[Np * (NNU == 3 ? d : 0)];
            }
        }
        const double Wn = A.W[n];
        const Thermo t = thermo(P, q, own_aux<Nq>(P, A.sa, ce, n, P.a_Phi, -0.0));
        if (write_aux) {
            double *ab = aux + (int64_t)Np * P.naux * e + n;
            if (P.a_theta_v >= 0) ab[(int64_t)Np * P.a_theta_v] = theta_v(P, t);
            if (P.a_air_T >= 0) ab[(int64_t)Np * P.a_air_T] = t.temp;
        }
        const double p = t.p;
        const double pm = P.ref_sub ? (p - own_aux<Nq>(P, A.sa, ce, n, P.a_ref_p, 0.0)) : p;
        const double rinv = 1.0 / q[0];
        u[0] = div_by(q[1], q[0], rinv);
        u[1] = div_by(q[2], q[0], rinv);
        u[2] = div_by(q[3], q[0], rinv);
        if (DIFF && WIDE) {
            const double *gb = gfi + (int64_t)Np * NGF * e + n;
#pragma unroll
            for (int s = 0; s < 9; ++s) gf[s] = gb[Np * s];
            if (SMAG) {
                const double *nb_ = nui + (int64_t)Np * NNU * e + n;
#pragma unroll
                for (int d = 0; d < 3; ++d) nu[d] = nb_[Np * (NNU == 3 ? d : 0)];
            }
        }
        if (DIFF && !SMAG) {
            const double gP[3] = {0.0, 0.0, 0.0};
            viscosity<false>(P, q[0], gf, gP, 0.0, nu);
        }
        const double M = ge[3] * Wn;
        MI = 1.0 / M;
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            double F[5], F2[5];
            flux1_row(q, u, p, pm, ax, F);
            if (DIFF) {
                flux2_row<SMAG>(P, q, gf, nu, ax, F2);
                int fn;
                const int f = node_face_dir<Nq>(i, j, k, ax, fn);
                if (!WIDE && f >= 0)
#pragma unroll
                    for (int v = 0; v < TR_F2; ++v) sFl[f * Nfp + fn][v] = F2[1 + v];
#pragma unroll
                for (int s = 0; s < 5; ++s) F[s] += F2[s];
            }
            const double x = ge[ax];
#pragma unroll
            for (int s = 0; s < 5; ++s) {
                const double v = M * (x * F[s]);
                if (ax < 2) sF[ax][s][n] = v;
                else Fv[s] = v;
            }
        }
    }
    if (!WIDE && n < 6) nb[n] = nbn;
    if (!WIDE && n < Nq * Nq) sD[n] = Dn;
    __syncthreads();
    // horizontal divergence of this node, into registers
    double T[5];
    if (act) {
        const double *tb = tend + (int64_t)Np * 5 * e + n;
#pragma unroll
        for (int s = 0; s < 5; ++s) {
            double th = 0.0;
#pragma unroll
            for (int m = 0; m < Nq; ++m) {
                th += MI * sD[m + Nq * i] * sF[0][s][m + Nq * (j + Nq * k)];
                th += MI * sD[m + Nq * j] * sF[1][s][i + Nq * (m + Nq * k)];
            }
            // MODE 1 is called with alpha = beta = 1 (exact products).  The branch on
            // beta also bounds the scheduler: without it every LDS read of the five
            // variables is hoisted ahead of the arithmetic (224 VGPRs against 119,
            // occupancy 2 against 4 waves per SIMD).
            T[s] =
                (beta != 0.0) ? alpha * th + beta * (MODE == 1 ? __builtin_nontemporal_load(tb + Np * s) : tb[Np * s])
                              : alpha * th;
        }
    }
    __syncthreads();
    if (act) {
#pragma unroll
        for (int s = 0; s < 5; ++s) {
            sF[0][s][n] = Fv[s];
            sQ[s][n] = q[s];
        }
    }
    __syncthreads();
    // vertical divergence and source
    if (act) {
        double src[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        if (P.gravity) {
            // Gravity() source (tendencies_momentum.jl:60-72), its static fields read again
            // (a class's block stays in cache) rather than held across the barriers
            const Aux a = load_aux(P, A.sa, Np, n, ce);
            const double drho = P.ref_src ? (sQ[0][n] - a.ref_rho) : sQ[0][n];
#pragma unroll
            for (int d = 0; d < 3; ++d) src[1 + d] = (-drho) * a.gPhi[d];
        }
#pragma unroll
        for (int s = 0; s < 5; ++s) {
            double tv = 0.0;
#pragma unroll
            for (int m = 0; m < Nq; ++m) {
                tv += MI * sD[m + Nq * k] * sF[0][s][i + Nq * (j + Nq * m)];
                if (m == k) tv += src[s];
            }
            T[s] = (MODE == 0 ? alpha * tv : tv) + T[s];
        }
    }
    // numerical fluxes of all face nodes, spread over every lane
    if (!WIDE) {
        for (int t = n; t < 6 * Nfp; t += NV) {
            double own[TR_F2], fl5[5];
            if (DIFF)
#pragma unroll
                for (int v = 0; v < TR_F2; ++v) own[v] = sFl[t][v];
            face_flux_aff<Nq, DIFF, NNU, false>(P, A, e, ce, t / Nfp, t % Nfp, nb[t / Nfp], sQ, Q, gfi, nui, own, fl5);
#pragma unroll
            for (int s = 0; s < 5; ++s) sFl[t][s] = fl5[s];
        }
        __syncthreads();
    }

    if (act) {
        // the face fluxes of this node's faces, in face order
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            int fn;
            const int f = node_face_dir<Nq>(i, j, k, d, fn);
            if (f < 0) continue;
            const double w = (MODE == 0 ? alpha * MI : MI) * (ge[4 + f] * A.Wf[fn]);
#pragma unroll
            for (int s = 0; s < 5; ++s) T[s] -= w * sFl[f * Nfp + fn][s];
        }
        double *tb = tend + (int64_t)Np * 5 * e + n;
        if (MODE == 0) {
#pragma unroll
            for (int s = 0; s < 5; ++s) tb[Np * s] = T[s];
        } else {
            // the stage's state from its LDS copy (sQ is intact after the face tasks); dQ,
            // Q' and dQ' pass through once, so they go nontemporal as in k_tendency_mix (here
            // without a measurable change: 96^3 plain FP64 41.07 GDOF/s with and without)
            double *qo = Qout + (int64_t)Np * 5 * e + n;
#pragma unroll
            for (int s = 0; s < 5; ++s) {
                __builtin_nontemporal_store(sQ[s][n] + bdt * T[s], qo + Np * s);
                if (dq_store) __builtin_nontemporal_store(T[s] * rka, tb + Np * s);
            }
        }
    }
}

}  // namespace cmdg
