// cmdg_learn.h -- kernels that build and train the learned closure and measure it:
// the FP64 velocity gradient of the DG gradient pass, the 2:1 element-agglomeration
// filter, training samples of the subgrid stress, the MLP loss gradient and Adam
// step, and DG -> equispaced interpolation for kinetic-energy spectra.
#pragma once
#include "cmdg_affine.h"
#include "cmdg_closure.h"

namespace cmdg {

// ------------------------------------------------------------------ velocity gradient
// du_c/dx_d at (n, 3c + d, e), FP64, formed as in the gradient pass: the volume
// derivative of u = rho u / rho plus the lifted central jump M^-1 Mf n (u* - u-),
// u* = (u+ + u-)/2 between elements, u* = u(q_wall) (normal momentum removed) on walls
// (DGModel_kernels.jl:1007-1127, 1471-1647; bc_momentum.jl:24-43).
template <int Nq>
__global__ void __launch_bounds__(threads_for<Nq>())
k_velgrad_aff(AffArrays A, int64_t nelem, const double *__restrict__ Q, double *__restrict__ Gu) {
    constexpr int Np = Nq * Nq * Nq;
    __shared__ double sD[Nq * Nq];
    __shared__ double sU[3][Np];
    const int64_t e = xcd_element(blockIdx.x, nelem);
    if (e >= nelem) return;
    const int n = threadIdx.x;
    if (n < Nq * Nq) sD[n] = A.D[n];
    const bool act = n < Np;
    const int i = n % Nq, j = (n / Nq) % Nq, k = n / (Nq * Nq);
    double u[3] = {0.0, 0.0, 0.0};
    if (act) {
        const double *qb = Q + (int64_t)Np * 5 * e + n;
        const double rinv = 1.0 / qb[0];
        for (int c = 0; c < 3; ++c) {
            u[c] = rinv * qb[Np * (1 + c)];
            sU[c][n] = u[c];
        }
    }
    __syncthreads();
    if (!act) return;
    const double *ge = A.geo + (int64_t)AFF_GEO * e;
    double g[3][3];
    for (int c = 0; c < 3; ++c) {
        double g1 = 0.0, g2 = 0.0, g3 = 0.0;
        for (int m = 0; m < Nq; ++m) {
            g1 += sD[i + Nq * m] * sU[c][m + Nq * (j + Nq * k)];
            g2 += sD[j + Nq * m] * sU[c][i + Nq * (m + Nq * k)];
            g3 += sD[k + Nq * m] * sU[c][i + Nq * (j + Nq * m)];
        }
        g[0][c] = ge[0] * g1;
        g[1][c] = ge[1] * g2;
        g[2][c] = ge[2] * g3;
    }
    const double MI = 1.0 / (ge[3] * A.W[n]);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        int fn;
        const int f = node_face_dir<Nq>(i, j, k, d, fn);
        if (f < 0) continue;
        const double w = MI * (ge[4 + f] * A.Wf[fn]) * ((f & 1) ? 1.0 : -1.0);
        const int32_t ne = A.nbe[6 * e + f];
        double jump[3];
        if (ne >= 0) {
            const double *qp = Q + (int64_t)Np * 5 * ne + face_node<Nq>(f ^ 1, fn);
            const double rp = 1.0 / qp[0];
            for (int s = 0; s < 3; ++s) jump[s] = 0.5 * (rp * qp[Np * (1 + s)] - u[s]);
        } else {
            for (int s = 0; s < 3; ++s) jump[s] = 0.0;
            jump[d] = -u[d];
        }
        for (int s = 0; s < 3; ++s) g[d][s] += w * jump[s];
    }
    double *o = Gu + (int64_t)Np * 9 * e + n;
    for (int cc = 0; cc < 3; ++cc)
        for (int d = 0; d < 3; ++d) o[(int64_t)Np * (3 * cc + d)] = g[d][cc];
}

// ------------------------------------------------------------------ 2:1 filter
// Coarse element ec is the union of 8 fine elements children[8 ec + (hx + 2 hy + 4 hz)],
// h = 0 for the lower half of the coarse element along that axis.  The coarse nodal
// values are the L2 projection (exact mass matrix) of the fine DG field onto the
// coarse polynomial space, a tensor product of the 1-D projections
// proj[h][i][a] (coarse node i, fine node a).  Fields filtered: rho, rho u (3), rho e
// and the second moments rho u_a u_b (11, 12, 13, 22, 23, 33) -> out (Np, 11, ncoarse).
constexpr int NMOM = 11;
struct FilterProj {
    double p[2][5][5];
};

// One axis at a time (70 products a node and field, 8 x 5 + 4 x 5 + 2 x 5, instead of
// 8 x 125): along x the two children of a pair into X, along y two pairs into Y, along z two
// halves into the result, each partial sum in registers and passed on through LDS, a row of Nq nodes padded
// to an even number so that two are read at once.  The children of the next pair are loaded
// while this one is contracted.  48^3 fine elements: 2176 -> 199 us traced warm (705 MB, 148 us at the
// copy rate); the sums are shorter, and closer to 64-bit exact, than the triple loop's.
template <int Nq>
__global__ void __launch_bounds__(threads_for<Nq>())
k_box_filter(const double *__restrict__ Qf, const int32_t *__restrict__ children, int64_t ncoarse, FilterProj PR,
             double *__restrict__ out) {
#pragma clang fp contract(fast)
    constexpr int Np = Nq * Nq * Nq, RW = (Nq + 1) / 2 * 2;  // padded row along x
    __shared__ double sM[NMOM][Nq * Nq * RW];                // moments of a child, then X or Y (Np of them)
    __shared__ double sP[2][Nq][Nq];
    const int64_t ec = blockIdx.x;
    if (ec >= ncoarse) return;
    const int n = threadIdx.x;
    const bool act = n < Np;
    const int i = n % Nq, j = (n / Nq) % Nq, k = n / (Nq * Nq);
    if (n < 2 * Nq * Nq) sP[n / (Nq * Nq)][(n / Nq) % Nq][n % Nq] = PR.p[n / (Nq * Nq)][(n / Nq) % Nq][n % Nq];
    const int32_t *ch = children + 8 * ec;
    double q[2][5];
    auto fetch = [&](int pair) {
        if (act)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const double *qb = Qf + (int64_t)Np * 5 * ch[2 * pair + h] + n;
#pragma unroll
                for (int s = 0; s < 5; ++s) q[h][s] = qb[Np * s];
            }
    };
    fetch(0);
    double zacc[NMOM] = {};
#pragma unroll 1
    for (int hz = 0; hz < 2; ++hz) {
        double yacc[NMOM] = {};
#pragma unroll 1
        for (int hy = 0; hy < 2; ++hy) {
            double xacc[NMOM] = {};
#pragma unroll
            for (int hx = 0; hx < 2; ++hx) {
                __syncthreads();
                if (act) {
                    const double r = q[hx][0], m1 = q[hx][1], m2 = q[hx][2], m3 = q[hx][3];
                    const double ri = 1.0 / r;
                    const int w = i + RW * (j + Nq * k);
                    sM[0][w] = r;
                    sM[1][w] = m1;
                    sM[2][w] = m2;
                    sM[3][w] = m3;
                    sM[4][w] = q[hx][4];
                    sM[5][w] = m1 * m1 * ri;
                    sM[6][w] = m1 * m2 * ri;
                    sM[7][w] = m1 * m3 * ri;
                    sM[8][w] = m2 * m2 * ri;
                    sM[9][w] = m2 * m3 * ri;
                    sM[10][w] = m3 * m3 * ri;
                }
                __syncthreads();
                if (hx == 1 && !(hz && hy)) fetch(2 * hz + hy + 1);
                if (act) {
                    double p[Nq];
#pragma unroll
                    for (int a = 0; a < Nq; ++a) p[a] = sP[hx][i][a];
#pragma unroll
                    for (int f = 0; f < NMOM; ++f) {
                        const double *row = &sM[f][RW * (j + Nq * k)];
#pragma unroll
                        for (int a = 0; a < Nq; ++a) xacc[f] += p[a] * row[a];
                    }
                }
            }
            __syncthreads();
            if (act)
#pragma unroll
                for (int f = 0; f < NMOM; ++f) sM[f][n] = xacc[f];
            __syncthreads();
            if (act) {
                double p[Nq];
#pragma unroll
                for (int b = 0; b < Nq; ++b) p[b] = sP[hy][j][b];
#pragma unroll
                for (int f = 0; f < NMOM; ++f)
#pragma unroll
                    for (int b = 0; b < Nq; ++b) yacc[f] += p[b] * sM[f][i + Nq * (b + Nq * k)];
            }
        }
        __syncthreads();
        if (act)
#pragma unroll
            for (int f = 0; f < NMOM; ++f) sM[f][n] = yacc[f];
        __syncthreads();
        if (act) {
            double p[Nq];
#pragma unroll
            for (int c = 0; c < Nq; ++c) p[c] = sP[hz][k][c];
#pragma unroll
            for (int f = 0; f < NMOM; ++f)
#pragma unroll
                for (int c = 0; c < Nq; ++c) zacc[f] += p[c] * sM[f][i + Nq * (j + Nq * c)];
        }
    }
    if (act)
#pragma unroll
        for (int f = 0; f < NMOM; ++f) out[(int64_t)Np * (f + NMOM * ec) + n] = zacc[f];
}

// ------------------------------------------------------------------ training samples
// One sample per coarse node from the filtered moments M (Np, 11, E) and the coarse
// velocity gradient Gu (Np, 9, E):
//   u = (rho u)/rho,  tau_ab = (rho u_a u_b)/rho - u_a u_b   (subgrid stress),
//   S = sym(Gu), S^d its deviator, |S| = sqrt(2 S:S), k = Delta^2 |S|,
//   T = tau^d - 2 (nu_mol - nu_floor) S^d   (what nu_0 - nu_floor must supply),
//   a = 2 k S^d;  with the network's coefficient c the model's deviatoric stress is
//   -c a - 2 nu_floor S^d, so the squared error is c^2 P + 2 c Q + R with P = a:a,
//   Q = a:T, R = T:T.
// Row layout (SoA, leading dimension ld): rows 0-8 du_c/dx_d at 3c + d, row 9
// Delta, rows 10-12 P, Q, R.
constexpr int SAMPLE_W = 13;

__global__ void k_closure_samples(const double *__restrict__ M, const double *__restrict__ Gu, int64_t nelem, int Np,
                                  double Delta, double nu_mol, double nu_floor, float *__restrict__ out, int64_t ld,
                                  int64_t offset) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nelem * Np) return;
    const int64_t e = t / Np;
    const int n = (int)(t - e * Np);
    const double *mb = M + (int64_t)Np * NMOM * e + n;
    const double *gb = Gu + (int64_t)Np * 9 * e + n;
    const double r = mb[0], ri = 1.0 / r;
    const double u[3] = {mb[Np] * ri, mb[2 * Np] * ri, mb[3 * Np] * ri};
    const int mi[3][3] = {{5, 6, 7}, {6, 8, 9}, {7, 9, 10}};
    double tau[3][3], G[3][3], S[3][3];
    for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) {
            tau[a][b] = mb[(int64_t)Np * mi[a][b]] * ri - u[a] * u[b];
            G[a][b] = gb[(int64_t)Np * (3 * a + b)];
        }
    for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) S[a][b] = 0.5 * (G[a][b] + G[b][a]);
    const double trS = (S[0][0] + S[1][1] + S[2][2]) / 3.0, trT = (tau[0][0] + tau[1][1] + tau[2][2]) / 3.0;
    double SS = 0.0;
    for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) SS += S[a][b] * S[a][b];
    const double c = Delta * Delta * sqrt(2.0 * SS);
    double P = 0.0, Qv = 0.0, R = 0.0;
    for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) {
            const double Sd = S[a][b] - (a == b ? trS : 0.0);
            const double T = (tau[a][b] - (a == b ? trT : 0.0)) - 2.0 * (nu_mol - nu_floor) * Sd;
            const double av = 2.0 * c * Sd;
            P += av * av;
            Qv += av * T;
            R += T * T;
        }
    float *o = out + offset + (int64_t)(t);
    for (int q = 0; q < 9; ++q) o[ld * q] = (float)G[q / 3][q % 3];
    o[ld * 9] = (float)Delta;
    o[ld * 10] = (float)P;
    o[ld * 11] = (float)Qv;
    o[ld * 12] = (float)R;
}

// Replaces P, Q, R of each sample by their mean over the sample's element (the local
// average of the dynamic procedure): the optimum coefficient of a node is then the
// element's least-squares coefficient -sum Q / sum P, not the noisy pointwise one.
__global__ void __launch_bounds__(128) k_element_average_pqr(float *__restrict__ out, int64_t ld, int64_t offset,
                                                             int Np) {
    __shared__ double red[3][128];
    const int64_t e = blockIdx.x;
    const int n = threadIdx.x;
    float *o = out + offset + e * Np;
    for (int r = 0; r < 3; ++r) red[r][n] = n < Np ? (double)o[ld * (10 + r) + n] : 0.0;
    __syncthreads();
    for (int w = 64; w > 0; w >>= 1) {
        if (n < w)
            for (int r = 0; r < 3; ++r) red[r][n] += red[r][n + w];
        __syncthreads();
    }
    if (n < Np)
        for (int r = 0; r < 3; ++r) o[ld * (10 + r) + n] = (float)(red[r][0] / Np);
}

// ------------------------------------------------------------------ training
// FP32 master parameters, flat: W1 [32][10] at 0, b1 at 320, W2 [32][32] at 352,
// b2 at 1376, W3 [32] at 1408, b3 at 1440.
constexpr int MP_W1 = 0, MP_B1 = 320, MP_W2 = 352, MP_B2 = 1376, MP_W3 = 1408, MP_B3 = 1440, MLP_NPARAM = 1441;
constexpr int GRAD_W = MLP_NPARAM + 1;  // + loss
// A row of partial gradients is one workgroup's.  The caller's workspace holds a row for
// every TRAIN_TB samples; a batch above 16384 fills TRAIN_ROWS of them, one a CU, whose waves
// take several tiles each, until a row holds ROW_SAMPLES samples (a batch of 65536), and from
// there on a row for every ROW_SAMPLES: what is summed in FP32 before the rows' FP64 sum does
// not grow with the batch.
constexpr int TRAIN_TB = 64, TRAIN_ROWS = 256, ROW_SAMPLES = 256;
constexpr int TRAIN_NT = 256, TRAIN_TILE = 16;  // threads a workgroup; samples a wave's tile
inline int64_t train_rows(int64_t batch) {
    const int64_t nb = (batch + TRAIN_TB - 1) / TRAIN_TB, full = (batch + ROW_SAMPLES - 1) / ROW_SAMPLES;
    return nb < TRAIN_ROWS ? nb : full < TRAIN_ROWS ? TRAIN_ROWS : full;
}

__device__ __forceinline__ float silu_fwd(float a, float &dsilu) {
#pragma clang fp contract(fast)
    const float s = 1.0f / (1.0f + expf(-a));
    dsilu = s * (1.0f + a * (1.0f - s));
    return a * s;
}

// The loss sum and its gradient with respect to every parameter over a workgroup's samples,
// written to partial[blockIdx][GRAD_W].  Forward as the inference (FP32 here, with the same
// input normalisation and output clamp), loss
// sum_s (c^2 P + 2 c Q + R) * inv_norm, c = clamp(y, MLP_CMIN, MLP_CMAX).
//
// Every product is a contraction, so it runs on FP32 MFMA (16x16x4: lane l holds
// A[l%16][l/16], B[l/16][l%16] and D[4(l/16)..+3][l%16]; FP32 products and sums).  A wave
// takes tiles of 16 samples as columns, features as rows: lane (g = l/16, s = l%16) holds
// features 16m + 4g + r of sample s.  The sum over the features of the next layer may take
// them in any order, so chunk (m, r) of it takes the features 16m + 4g + r, g = 0..3, that
// the lanes already hold in register (m, r); only the weights are laid out to match.  The
// weight gradients contract over samples, for which each matrix is transposed once through
// the wave's LDS.  b1 rides along as the weight of an eleventh input that is 1.
// 65536 rows of a 2^21-sample table: 187 -> 25 us traced warm (one lane a sample with its activations in
// 170 registers ran one wave a SIMD, its weight-gradient loops 64 serial LDS reads long).
// What is left is the gather (13 words of a sample lie in 13 lines): rows in order take 15.
// 256 rows of partials, one workgroup a CU, are faster than 512 or 1024 from 32768 samples on
// (27 against 31 and 33 us for the two launches at 65536), and equal below.  Above 65536 a row
// keeps to 256 samples: 268 us at 2^20, 1016 at 2^22, where 256 rows of any length took 250 and
// 949 but summed up to 16384 samples a row in FP32 (one repeated tile of samples: 4e-5 off).
__global__ void __launch_bounds__(TRAIN_NT)
k_mlp_grad(const float *__restrict__ params, const float *__restrict__ shift, const float *__restrict__ scale,
           const float *__restrict__ samples, int64_t ld, const int64_t *__restrict__ idx, int64_t batch,
           float inv_norm, float *__restrict__ partial) {
#pragma clang fp contract(fast)
    constexpr int NW = TRAIN_NT / 64, LD = TRAIN_TILE + 1;     // a padded row of 16 samples
    constexpr int R_D2 = 0, R_H1 = 32, R_D1 = 64, R_X = 96, ROWS = 112;
    static_assert(ROWS * LD >= GRAD_W, "a wave's slab holds its gradient row at the end");
    __shared__ float slab[NW][ROWS * LD];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, s = lane & 15, g = lane >> 4;
    float *W = slab[wave];

    // weights as MFMA operands, biases and w3 in the features' layout
    float A1[2][3], A2[2][2][4], A2t[2][2][4], B2[2][4], W3[2][4];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const int k = 4 * c + g, o = 16 * m + s;
            A1[m][c] = k < MLP_IN ? params[MP_W1 + MLP_IN * o + k] : (k == MLP_IN ? params[MP_B1 + o] : 0.0f);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                A2[m][q][r] = params[MP_W2 + MLP_H * (16 * m + s) + 16 * q + 4 * g + r];
                A2t[m][q][r] = params[MP_W2 + MLP_H * (16 * q + 4 * g + r) + 16 * m + s];
            }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            B2[m][r] = params[MP_B2 + 16 * m + 4 * g + r];
            W3[m][r] = params[MP_W3 + 16 * m + 4 * g + r];
        }
    }
    const float b3 = params[MP_B3];
    float sh[3], sc[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const int k = 4 * c + g;
        sh[c] = k < MLP_IN ? shift[k] : 0.0f;
        sc[c] = k < MLP_IN ? scale[k] : 0.0f;
    }

    mlp_f32x4 G2[2][2] = {}, G1[2] = {};  // dW2 and dW1 (with db1) of the wave's samples
    float g3[2][4] = {}, gb2[2][4] = {}, gb3 = 0.0f, loss = 0.0f;

    // the four words of a sample that this lane reads: inputs g, 4 + g, 8 + g and row 10 + g
    const int64_t ntile = (batch + TRAIN_TILE - 1) / TRAIN_TILE, stride = (int64_t)gridDim.x * NW;
    float raw[4];
    bool valid;
    auto fetch = [&](int64_t tile) {
        const int64_t i = tile * TRAIN_TILE + s;
        valid = tile < ntile && i < batch;
        raw[0] = raw[1] = raw[2] = raw[3] = 0.0f;
        if (valid) {
            const float *p = samples + (idx ? idx[i] : i);
            raw[0] = p[ld * g];
            raw[1] = p[ld * (4 + g)];
            if (g < 2) raw[2] = p[ld * (8 + g)];
            if (g < 3) raw[3] = p[ld * (10 + g)];
        }
    };
    int64_t tile = (int64_t)blockIdx.x * NW + wave;
    fetch(tile);
    for (; tile < ntile; tile += stride) {
        const bool live = valid;
        float x[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) x[c] = live ? (raw[c] - sh[c]) * sc[c] : 0.0f;
        if (g == 2) x[2] = 1.0f;  // input 10
        const float pqr = raw[3];
        const float P = __shfl(pqr, s), Qv = __shfl(pqr, 16 + s), R = __shfl(pqr, 32 + s);
        fetch(tile + stride);

        float h1[2][4], a1d[2][4], a2d[2][4], y = 0.0f;
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            mlp_f32x4 a = {};
#pragma unroll
            for (int c = 0; c < 3; ++c) a = __builtin_amdgcn_mfma_f32_16x16x4f32(A1[m][c], x[c], a, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) h1[m][r] = silu_fwd(a[r], a1d[m][r]);
        }
        float h2[2][4];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            mlp_f32x4 a = {B2[m][0], B2[m][1], B2[m][2], B2[m][3]};
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    a = __builtin_amdgcn_mfma_f32_16x16x4f32(A2[m][q][r], h1[q][r], a, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                h2[m][r] = silu_fwd(a[r], a2d[m][r]);
                y += W3[m][r] * h2[m][r];
            }
        }
        y += __shfl_xor(y, 16);
        y += __shfl_xor(y, 32);
        y += b3;
        float dy = 0.0f;
        if (live) {
            const bool clamped = y > MLP_CMAX || y < MLP_CMIN;
            const float c = fminf(fmaxf(y, MLP_CMIN), MLP_CMAX);
            loss += (c * c * P + 2.0f * c * Qv + R) * inv_norm;
            dy = clamped ? 0.0f : (2.0f * c * P + 2.0f * Qv) * inv_norm;
        }
        gb3 += dy;
        float d2[2][4];
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                d2[m][r] = dy * W3[m][r] * a2d[m][r];
                g3[m][r] += dy * h2[m][r];
                gb2[m][r] += d2[m][r];
                const int f = 16 * m + 4 * g + r;
                W[(R_D2 + f) * LD + s] = d2[m][r];
                W[(R_H1 + f) * LD + s] = h1[m][r];
            }
#pragma unroll
        for (int c = 0; c < 3; ++c) W[(R_X + 4 * c + g) * LD + s] = x[c];
        W[(R_X + 12 + g) * LD + s] = 0.0f;
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            mlp_f32x4 a = {};
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    a = __builtin_amdgcn_mfma_f32_16x16x4f32(A2t[m][q][r], d2[q][r], a, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) W[(R_D1 + 16 * m + 4 * g + r) * LD + s] = a[r] * a1d[m][r];
        }
        // the slab is the wave's own: LDS serves one wave's accesses in order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float u2[2], u1[2], v2[2];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                u2[m] = W[(R_D2 + 16 * m + s) * LD + 4 * c + g];
                u1[m] = W[(R_D1 + 16 * m + s) * LD + 4 * c + g];
                v2[m] = W[(R_H1 + 16 * m + s) * LD + 4 * c + g];
            }
            const float v1 = W[(R_X + s) * LD + 4 * c + g];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                G1[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(u1[m], v1, G1[m], 0, 0, 0);
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    G2[m][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(u2[m], v2[q], G2[m][q], 0, 0, 0);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    // the wave's gradient row into its slab, then the workgroup's sum in wave order
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int o = 16 * m + 4 * g + r;
            if (s < MLP_IN) W[MP_W1 + MLP_IN * o + s] = G1[m][r];
            if (s == MLP_IN) W[MP_B1 + o] = G1[m][r];
#pragma unroll
            for (int q = 0; q < 2; ++q) W[MP_W2 + MLP_H * o + 16 * q + s] = G2[m][q][r];
            float v3 = g3[m][r], vb = gb2[m][r];
#pragma unroll
            for (int w = 1; w < 16; w <<= 1) {
                v3 += __shfl_xor(v3, w);
                vb += __shfl_xor(vb, w);
            }
            if (s == 0) {
                W[MP_W3 + o] = v3;
                W[MP_B2 + o] = vb;
            }
        }
#pragma unroll
    for (int w = 1; w < 16; w <<= 1) {
        gb3 += __shfl_xor(gb3, w);
        loss += __shfl_xor(loss, w);
    }
    if (lane == 0) {
        W[MP_B3] = gb3;
        W[MLP_NPARAM] = loss;
    }
    __syncthreads();
    float *pb = partial + (int64_t)blockIdx.x * GRAD_W;
    for (int q = threadIdx.x; q < GRAD_W; q += TRAIN_NT) {
        float acc = slab[0][q];
#pragma unroll
        for (int w = 1; w < NW; ++w) acc += slab[w][q];
        pb[q] = acc;
    }
}

// grad[q] = sum over the rows of partial[b][q] in FP64, in a fixed order (deterministic): 16
// columns a workgroup, 16 lanes a column, each every 16th row, then those 16 in order.  The
// last entry is the loss.  (One lane a column took 250 us over 1024 rows: six workgroups,
// one load after the other.)
constexpr int REDUCE_C = 16;
__global__ void __launch_bounds__(256) k_grad_reduce(const float *__restrict__ partial, int64_t nb,
                                                     float *__restrict__ grad) {
    __shared__ double red[16][REDUCE_C + 1];
    const int c = threadIdx.x % REDUCE_C, r = threadIdx.x / REDUCE_C;
    const int q = blockIdx.x * REDUCE_C + c;
    double acc = 0.0;
    if (q < GRAD_W) {
#pragma unroll 8
        for (int64_t b = r; b < nb; b += 16) acc += (double)partial[b * GRAD_W + q];
    }
    red[r][c] = acc;
    __syncthreads();
    if (r == 0 && q < GRAD_W) {
#pragma unroll
        for (int k = 1; k < 16; ++k) acc += red[k][c];
        grad[q] = (float)acc;
    }
}

__global__ void k_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, int64_t n, float lr, float b1, float b2, float eps, float c1, float c2) {
#pragma clang fp contract(fast)
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const float gq = g[q];
    const float mq = b1 * m[q] + (1.0f - b1) * gq;
    const float vq = b2 * v[q] + (1.0f - b2) * gq * gq;
    m[q] = mq;
    v[q] = vq;
    p[q] -= lr * (mq / c1) / (sqrtf(vq / c2) + eps);
}

// ------------------------------------------------------------------ spectra
// Velocity u = (rho u)/rho of element e interpolated to p^3 equispaced points
// xi_m = -1 + (2m + 1)/p per axis (cell centres), written to
// out[c][iz p + mz][iy p + my][ix p + mx] for the element's brick index (ix, iy, iz)
// (InterpolationBrick semantics, src/Numerics/Mesh/Interpolation.jl:66-571, onto a
// uniform grid).  L[m][i] = l_i(xi_m).
struct InterpMat {
    double L[8][5];
};

// One axis at a time through LDS.  Where the elements fill the uniform grid (their number is
// its points over p^3) the workgroups walk them with x fastest, as a stacked brick stores them
// (z fastest, then x, then y), so that one XCD's L2 completes the lines of out, of which an
// element writes p words; any order is right, the position comes from eijk.
// 40^3 elements, p = 4: 177 -> 77 us traced warm (354 MB, 74 us at the copy rate); with p at run time
// the index arithmetic held it at 141.
constexpr int interp_threads(int p) { return p <= 3 ? 64 : p <= 5 ? 128 : 256; }
template <int Nq, int p>
__global__ void __launch_bounds__(interp_threads(p))
k_interp_equispaced(const double *__restrict__ Q, const int32_t *__restrict__ eijk, int64_t nelem, InterpMat IM,
                    int64_t nxt, int64_t nyt, int64_t nzt, double *__restrict__ out) {
#pragma clang fp contract(fast)
    constexpr int Np = Nq * Nq * Nq, nt = interp_threads(p);
    // u (3 Np), then the values interpolated along x and y [c][k][my][mx]
    __shared__ double sA[3 * (p * p * Nq > Np ? p * p * Nq : Np)];
    __shared__ double sB[3 * p * Nq * Nq];  // along x: [c][k][j][mx]
    __shared__ double sL[p * Nq];
    const int t = threadIdx.x;
    int64_t e = xcd_element(blockIdx.x, nelem);
    if (e >= nelem) return;
    const int64_t nx = nxt / p, ny = nyt / p, nz = nzt / p;
    if (nx * ny * nz == nelem) {
        const int64_t ix = e % nx, r = e / nx;
        e = (r % nz) + nz * (ix + nx * (r / nz));
    }
    if (t < p * Nq) sL[t] = IM.L[t / Nq][t % Nq];
#pragma unroll
    for (int n = t; n < Np; n += nt) {
        const double *qb = Q + (int64_t)Np * 5 * e + n;
        const double ri = 1.0 / qb[0];
#pragma unroll
        for (int c = 0; c < 3; ++c) sA[c * Np + n] = qb[Np * (1 + c)] * ri;
    }
    const int X0 = eijk[3 * e], Y0 = eijk[3 * e + 1], Z0 = eijk[3 * e + 2];
    __syncthreads();
#pragma unroll
    for (int w = t; w < 3 * Nq * Nq * p; w += nt) {
        const int mx = w % p, row = w / p;  // row = (c Nq + k) Nq + j
        double v = 0.0;
#pragma unroll
        for (int a = 0; a < Nq; ++a) v += sL[mx * Nq + a] * sA[row * Nq + a];
        sB[w] = v;
    }
    __syncthreads();
#pragma unroll
    for (int w = t; w < 3 * Nq * p * p; w += nt) {
        const int mx = w % p, my = (w / p) % p, ck = w / (p * p);
        double v = 0.0;
#pragma unroll
        for (int b = 0; b < Nq; ++b) v += sL[my * Nq + b] * sB[(ck * Nq + b) * p + mx];
        sA[w] = v;
    }
    __syncthreads();
#pragma unroll
    for (int w = t; w < 3 * p * p * p; w += nt) {
        const int xy = w % (p * p), mz = (w / (p * p)) % p, c = w / (p * p * p);
        double v = 0.0;
#pragma unroll
        for (int k = 0; k < Nq; ++k) v += sL[mz * Nq + k] * sA[(c * Nq + k) * p * p + xy];
        const int64_t X = (int64_t)X0 * p + xy % p, Y = (int64_t)Y0 * p + xy / p, Z = (int64_t)Z0 * p + mz;
        out[((c * nzt + Z) * nyt + Y) * nxt + X] = v;
    }
}

}  // namespace cmdg
