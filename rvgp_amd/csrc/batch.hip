// Batched independent GP fits on one shared manifold: F vector fields, each
// with its own training subset (of any size) and its own hyperparameters,
// fitted together.  The single-fit path (GPflow's GPR reached from
// RVGP/main.py:87-95) runs F times in the reference; here every fit of a
// step runs inside one kernel launch.
//
// Weight-space form (exact for any subset size): with the intrinsic
// eigenvector rows U_i (d x k) of the training nodes of fit f,
//     G_f = sum_i U_i^T U_i      b_f = sum_i U_i^T c_i,   c_i = T_i^T y_i
// equal Phi^T Phi and Phi^T y over the ambient rows Phi_i = T_i U_i (the
// gauge T_i has orthonormal columns), so the ambient design matrix is never
// formed.  Per optimiser step and fit:
//     A = G + s2 diag(S)^-1 = L L^T,  X = L^-1,  diag(A^-1)_j = |X e_j|^2,
//     w = X^T (X b),  then the NLML / adjoint of gp.hip's weight-space
//     finish and one Adam update of the fit's 4 unconstrained parameters.
//
// Kernels:
//   batch_gram_kernel<BT, WT>  upper BT x BT tiles of every G_f on the matrix
//                              cores (v_mfma_f64_16x16x4f64), U rows gathered
//                              through the fit's node list into LDS (FP32
//                              input is widened to FP64 in LDS); XCD-aware
//                              block order keeps one fit's tiles on one XCD.
//   batch_rhs_kernel           b_f and y^T y per fit.
//   batch_step_kernel<NB>      one workgroup per fit (persistent over fits):
//                              filter, A, right-looking blocked Cholesky of
//                              [A | I] that yields L and L^-1 together
//                              (diagonal block in registers of one wave,
//                              panel staged in LDS, trailing update of both
//                              halves on the matrix cores), solves, NLML,
//                              adjoint and Adam.
#include "common.h"

#pragma clang fp contract(fast)

namespace rvgp {

typedef double dbl4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ Gram
template <typename T>
__device__ __forceinline__ double as_f64(T v) { return (double)v; }

constexpr int GBK = 16;  // gathered rows per LDS stage

template <int BT, int WT, typename TIn>
__global__ __launch_bounds__((BT / WT) * (BT / WT) * 64) void batch_gram_kernel(
    int F, int k, int d, const TIn* __restrict__ U, int ldu, const int* __restrict__ off,
    const int* __restrict__ nodes, int ntiles, int T, double* __restrict__ G) {
    constexpr int NW = (BT / WT) * (BT / WT);
    constexpr int NTH = NW * 64;
    constexpr int MT = WT / 16;  // MFMA tiles per wave side
    __shared__ double As[GBK][BT + 1];
    __shared__ double Bs[GBK][BT + 1];
    __shared__ int rows[GBK];

    // XCD-aware order: blocks are dealt round-robin to the 8 XCDs, so logical
    // block q = (L mod 8) * (total / 8) + L / 8 keeps consecutive q -- the
    // tiles of one fit -- on one XCD and its L2
    const int total = ntiles * F;
    int q = blockIdx.x;
    if (total % 8 == 0) q = (blockIdx.x % 8) * (total / 8) + blockIdx.x / 8;
    const int f = q / ntiles;
    int t = q - f * ntiles;
    // tile t -> (ti, tj), ti <= tj, row-major over the upper triangle
    int ti = 0;
    while (t >= T - ti) { t -= T - ti; ++ti; }
    const int tj = ti + t;
    const bool diag = ti == tj;
    const int m0 = ti * BT, n0 = tj * BT;
    const int r0 = off[f] * d, r1 = off[f + 1] * d;

    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wm = (w / (BT / WT)) * WT, wn = (w % (BT / WT)) * WT;
    dbl4 acc[MT][MT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = dbl4{0, 0, 0, 0};

    for (int k0 = r0; k0 < r1; k0 += GBK) {
        if (tid < GBK) {
            const int r = k0 + tid;
            rows[tid] = r < r1 ? nodes[r / d] * d + (r % d) : -1;
        }
        __syncthreads();
        for (int e = tid; e < GBK * BT; e += NTH) {
            const int kk = e / BT, mm = e - kk * BT;
            const int ur = rows[kk];
            double va = 0.0, vb = 0.0;
            if (ur >= 0) {
                const TIn* up = U + (size_t)ur * ldu;
                if (m0 + mm < k) va = as_f64(up[m0 + mm]);
                if (!diag && n0 + mm < k) vb = as_f64(up[n0 + mm]);
            }
            As[kk][mm] = va;
            if (!diag) Bs[kk][mm] = vb;
        }
        __syncthreads();
        const double(*Bp)[BT + 1] = diag ? As : Bs;
#pragma unroll
        for (int ks = 0; ks < GBK; ks += 4) {
            const int kr = ks + (lane >> 4);
            double a[MT], b[MT];
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                a[i] = As[kr][wm + i * 16 + (lane & 15)];
                b[i] = Bp[kr][wn + i * 16 + (lane & 15)];
            }
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    // f64 MFMA output: lane holds column lane%16, rows lane/16 + 4 r
    double* Gf = G + (size_t)f * k * k;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gm = m0 + wm + i * 16 + (lane >> 4) + 4 * r;
                const int gn = n0 + wn + j * 16 + (lane & 15);
                if (gm < k && gn < k) {
                    Gf[(size_t)gm * k + gn] = acc[i][j][r];
                    if (!diag) Gf[(size_t)gn * k + gm] = acc[i][j][r];
                }
            }
}

// b_f[j] = sum over the fit's rows of U[row][j] c[row]; yy_f = sum of the
// fit's per-node |y_i|^2.  grid (ceil(k / 64), F): wave w of 16 takes the nodes
// w, w + 16, ... of 64 columns, so that a fit's rows are in flight together (a
// thread per column walked them one by one: 128 fits of 50 to 1500 nodes,
// 637 -> 64 us).
constexpr int kRhsWaves = 16;

__global__ __launch_bounds__(64 * kRhsWaves) void batch_rhs_kernel(int F, int k, int d,
                                                                   const double* __restrict__ U, int ldu,
                                                                   const int* __restrict__ off,
                                                                   const int* __restrict__ nodes,
                                                                   const double* __restrict__ c,
                                                                   const double* __restrict__ ynorm2,
                                                                   double* __restrict__ b,
                                                                   double* __restrict__ yy) {
    __shared__ double sh[kRhsWaves][64];
    const int f = blockIdx.y, lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = blockIdx.x * 64 + lane;
    const int t0 = off[f], t1 = off[f + 1];
    double s0 = 0.0, s1 = 0.0;
    if (j < k) {
#pragma unroll 4
        for (int t = t0 + wv; t < t1; t += kRhsWaves) {
            const double* up = U + (size_t)nodes[t] * d * ldu + j;
            const double* cp = c + (size_t)t * d;
            for (int p = 0; p < d; ++p) {
                if (p & 1) s1 = fma(up[(size_t)p * ldu], cp[p], s1);
                else s0 = fma(up[(size_t)p * ldu], cp[p], s0);
            }
        }
    }
    sh[wv][lane] = s0 + s1;
    __syncthreads();
    if (wv == 0 && j < k) {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < kRhsWaves; ++q) s += sh[q][lane];
        b[(size_t)f * k + j] = s;
    }
    if (blockIdx.x == 0) {
        double s = 0.0;
        for (int t = t0 + threadIdx.x; t < t1; t += 64 * kRhsWaves) s += ynorm2[t];
        s = wave_sum(s);
        __syncthreads();
        if (lane == 0) sh[0][wv] = s;
        __syncthreads();
        if (threadIdx.x == 0) {
            double v = 0.0;
#pragma unroll
            for (int q = 0; q < kRhsWaves; ++q) v += sh[0][q];
            yy[f] = v;
        }
    }
}

// ------------------------------------------------------------------ step
// Threads per fit workgroup (ST = 512 or 1024, a template parameter chosen
// by the autotuner): more waves hide more of each panel step's memory
// latency; fewer leave more registers per thread.
template <int ST>
__device__ double wg_sum(double v, double* sh) {
    v = wave_sum(v);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[w] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < ST / 64; ++i) s += sh[i];
    return s;
}

// Lanes 0-3 of a fit: gradients to `out`, one Adam step of their parameter.
// sig = dtheta/du = sigmoid(u); p1, p2 = b1, b2 to the power of the new step.
__device__ __forceinline__ void step_finish(int tid, int f, double gth, double nlml, double sig,
                                            double* uf, const int* trainable, double* m1, double* m2,
                                            double* tstep, double step, int do_adam, double lr,
                                            double b1, double b2, double p1, double p2, double eps,
                                            double* out) {
    const double gu = gth * sig;
    double* o = out + 9 * (size_t)f;
    if (tid == 0) o[0] = nlml;
    o[1 + tid] = gth;
    o[5 + tid] = gu;
    if (do_adam) {
        // Adam on the fit's own state; its step counter is read by
        // lanes 0-3 before lane 0 stores the increment
        if (trainable[tid]) {
            double* mf = m1 + 4 * (size_t)f;
            double* vf = m2 + 4 * (size_t)f;
            mf[tid] = b1 * mf[tid] + (1.0 - b1) * gu;
            vf[tid] = b2 * vf[tid] + (1.0 - b2) * gu * gu;
            const double mh = mf[tid] / (1.0 - p1);
            const double vh = vf[tid] / (1.0 - p2);
            uf[tid] -= lr * mh / (sqrt(vh) + eps);
        }
        __builtin_amdgcn_wave_barrier();
        if (tid == 0) tstep[f] = step;
    }
}

// Per-fit workspace: W = [A | X] (k x 2k, row-major) then vectors
// S, dS (3k), gS, ainv, t, w, Gw (9k doubles).
__host__ __device__ inline size_t step_ws_doubles(int k) { return 2 * (size_t)k * k + 9 * (size_t)k; }

template <int NB, int ST>
__global__ __launch_bounds__(ST) void batch_step_kernel(
    int F, int k, int typ, const double* __restrict__ lam, double n_rows,
    const double* __restrict__ G, const double* __restrict__ bvec, const double* __restrict__ yy,
    const double* __restrict__ Mrows, const double* __restrict__ lower, double* __restrict__ u,
    const int* __restrict__ trainable, double* __restrict__ m1, double* __restrict__ m2,
    double* __restrict__ tstep, int do_adam, double lr, double b1, double b2, double eps,
    double* __restrict__ ws, double* __restrict__ out, int* __restrict__ status) {
    extern __shared__ double lds[];
    // LDS: Ld[NB][NB + 1] (diagonal factor), P[k][NB + 1] (panel rows)
    double* Ld = lds;
    double* P = lds + NB * (NB + 1);
    __shared__ double sh[ST / 64];
    __shared__ double th[8];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int ldw = 2 * k;

    for (int f = blockIdx.x; f < F; f += gridDim.x) {
        const double* Gf = G + (size_t)f * k * k;
        const double* bf = bvec + (size_t)f * k;
        double* W = ws + (size_t)f * step_ws_doubles(k);
        double* S = W + 2 * (size_t)k * k;
        double* dS = S + k;
        double* gS = dS + 3 * k;
        double* ainv = gS + k;
        double* tv = ainv + k;
        double* wv_ = tv + k;
        double* Gw = wv_ + k;
        double* uf = u + 4 * (size_t)f;

        // ---- theta = softplus(u) + lower
        if (tid < 4) {
            const double x = uf[tid];
            const double sp = x > 0 ? x + log1p(exp(-x)) : log1p(exp(x));
            th[tid] = sp + lower[tid];
        }
        __syncthreads();
        const double nu = th[0], kappa = th[1], sf = th[2], s2 = th[3];

        // ---- spectral filter S and dS/d(nu, kappa, sigma_f) (kernels.py:41-53)
        const double shf = 2.0 * nu / (kappa * kappa);
        double sr = 0.0, snu = 0.0, ska = 0.0;
        for (int j = tid; j < k; j += ST) {
            double r, dn, dk;
            if (typ == 0) {
                const double base = lam[j] + shf;
                r = pow(base, -nu);
                dn = -log(base) - nu * (2.0 / (kappa * kappa)) / base;
                dk = 4.0 * nu * nu / (kappa * kappa * kappa * base);
            } else {
                r = exp(-0.5 * lam[j] * kappa * kappa);
                dn = 0.0;
                dk = -lam[j] * kappa;
            }
            sr += r;
            snu += r * dn;
            ska += r * dk;
        }
        sr = wg_sum<ST>(sr, sh);
        snu = wg_sum<ST>(snu, sh) / sr;
        ska = wg_sum<ST>(ska, sh) / sr;
        for (int j = tid; j < k; j += ST) {
            double r, dn, dk;
            if (typ == 0) {
                const double base = lam[j] + shf;
                r = pow(base, -nu);
                dn = -log(base) - nu * (2.0 / (kappa * kappa)) / base;
                dk = 4.0 * nu * nu / (kappa * kappa * kappa * base);
            } else {
                r = exp(-0.5 * lam[j] * kappa * kappa);
                dn = 0.0;
                dk = -lam[j] * kappa;
            }
            const double s = sf * n_rows * r / sr;
            S[j] = s;
            dS[j] = s * (dn - snu);
            dS[k + j] = s * (dk - ska);
            dS[2 * k + j] = s / sf;
        }
        __syncthreads();

        // ---- W = [G + diag(s2 / S) | I]
        for (size_t e = tid; e < (size_t)k * ldw; e += ST) {
            const int i = (int)(e / ldw), j = (int)(e - (size_t)i * ldw);
            double v;
            if (j < k) v = Gf[(size_t)i * k + j] + (i == j ? s2 / S[i] : 0.0);
            else v = (j - k == i) ? 1.0 : 0.0;
            W[e] = v;
        }
        __syncthreads();

        // ---- blocked right-looking Cholesky of A, applied to X at once
        int bad = 0;
        for (int j0 = 0; j0 < k; j0 += NB) {
            const int jb = min(NB, k - j0);
            const int t0 = j0 + jb;  // first trailing row
            // (1) diagonal block: lane i holds row i in registers
            if (wv == 0) {
                double row[NB];
                const int i = lane;
#pragma unroll
                for (int c = 0; c < NB; ++c)
                    row[c] = (i < jb && c <= i) ? W[(size_t)(j0 + i) * ldw + j0 + c] : 0.0;
#pragma unroll
                for (int c = 0; c < NB; ++c) {
                    if (c < jb) {
                        double piv = bcast(row[c], c);
                        if (!(piv > 0.0)) {  // not positive definite (or NaN)
                            bad = 1;
                            piv = 1.0;
                        }
                        const double dc = sqrt(piv);
                        const double lic = i > c ? row[c] / dc : (i == c ? dc : 0.0);
                        row[c] = lic;
#pragma unroll
                        for (int l = c + 1; l < NB; ++l) {
                            const double llc = __shfl(lic, l, 64);  // L[l][c] (VGPR)
                            if (l <= i && l < jb) row[l] -= lic * llc;
                        }
                    }
                }
                if (i < NB) {
#pragma unroll
                    for (int c = 0; c < NB; ++c) {
                        Ld[i * (NB + 1) + c] = (c <= i && i < jb) ? row[c] : 0.0;
                        if (c <= i && i < jb) W[(size_t)(j0 + i) * ldw + j0 + c] = row[c];
                    }
                }
            }
            __syncthreads();
            // (2) panel rows i >= t0: L[i, J] = A[i, J] L_JJ^-T (row solve),
            //     and rows J of X: X[J, :t0] = L_JJ^-1 X[J, :t0] (column solve)
            const int nrow = k - t0, ncol = t0;
            for (int e = tid; e < nrow + ncol; e += ST) {
                double x[NB];
                if (e < nrow) {
                    const int i = t0 + e;
                    double* wr = W + (size_t)i * ldw + j0;
#pragma unroll
                    for (int c = 0; c < NB; ++c) x[c] = c < jb ? wr[c] : 0.0;
#pragma unroll
                    for (int c = 0; c < NB; ++c) {
                        if (c < jb) {
                            double s = x[c];
#pragma unroll
                            for (int l = 0; l < c; ++l) s -= x[l] * Ld[c * (NB + 1) + l];
                            x[c] = s / Ld[c * (NB + 1) + c];
                        }
                    }
#pragma unroll
                    for (int c = 0; c < NB; ++c) {
                        const double v = c < jb ? x[c] : 0.0;
                        if (c < jb) wr[c] = v;
                        P[e * (NB + 1) + c] = v;
                    }
                } else {
                    const int cc = e - nrow;  // column of X
                    double* xc = W + (size_t)j0 * ldw + k + cc;
#pragma unroll
                    for (int r = 0; r < NB; ++r) x[r] = r < jb ? xc[(size_t)r * ldw] : 0.0;
#pragma unroll
                    for (int r = 0; r < NB; ++r) {
                        if (r < jb) {
                            double s = x[r];
#pragma unroll
                            for (int l = 0; l < r; ++l) s -= Ld[r * (NB + 1) + l] * x[l];
                            x[r] = s / Ld[r * (NB + 1) + r];
                        }
                    }
#pragma unroll
                    for (int r = 0; r < NB; ++r)
                        if (r < jb) xc[(size_t)r * ldw] = x[r];
                }
            }
            __syncthreads();
            // (3) trailing update on the matrix cores, 16 x 16 tiles:
            //     A[i, j] -= P_i . P_j   (t0 <= j <= i: lower tiles)
            //     X[i, c] -= P_i . X[J, c]  (c < t0)
            // A wave takes TG tiles at a time and issues all their loads of
            // the old values before the products, so TG round trips to the
            // cache overlap instead of following one another.
            const int TR = (nrow + 15) / 16, TC = (ncol + 15) / 16;
            const int nA = TR * (TR + 1) / 2, ntile = nA + TR * TC;
            constexpr int TG = 4;
            for (int base = wv * TG; base < ntile; base += (ST / 64) * TG) {
                int tis[TG], tjs[TG];
                dbl4 cv[TG];
#pragma unroll
                for (int g = 0; g < TG; ++g) {
                    const int tI = base + g;
                    int ti = -1, tj = 0;
                    if (tI < nA) {
                        // lower-triangle tile index -> (ti, tj), tj <= ti
                        ti = (int)((sqrt(8.0 * tI + 1.0) - 1.0) * 0.5);
                        while ((ti + 1) * (ti + 2) / 2 <= tI) ++ti;
                        while (ti * (ti + 1) / 2 > tI) --ti;
                        tj = tI - ti * (ti + 1) / 2;
                    } else if (tI < ntile) {
                        const int q = tI - nA;
                        ti = q / TC;
                        tj = TR + q - (q / TC) * TC;  // X tiles: tj >= TR marks them
                    }
                    tis[g] = ti;
                    tjs[g] = tj;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int row = ti * 16 + (lane >> 4) + 4 * r;
                        double v = 0.0;
                        if (ti >= 0 && row < nrow) {
                            if (tj < TR) {
                                const int col = tj * 16 + (lane & 15);
                                if (col <= row) v = W[(size_t)(t0 + row) * ldw + t0 + col];
                            } else {
                                const int col = (tj - TR) * 16 + (lane & 15);
                                if (col < ncol) v = W[(size_t)(t0 + row) * ldw + k + col];
                            }
                        }
                        cv[g][r] = v;
                    }
                }
#pragma unroll
                for (int g = 0; g < TG; ++g) {
                    const int ti = tis[g], tj = tjs[g];
                    if (ti < 0) continue;
                    dbl4 acc = dbl4{0, 0, 0, 0};
                    const int ar = ti * 16 + (lane & 15);  // panel row of the A fragment
#pragma unroll
                    for (int ks = 0; ks < NB; ks += 4) {
                        const int kc = ks + (lane >> 4);
                        const double a = (ar < nrow && kc < jb) ? P[ar * (NB + 1) + kc] : 0.0;
                        double b;
                        if (tj < TR) {
                            const int br = tj * 16 + (lane & 15);
                            b = (br < nrow && kc < jb) ? P[br * (NB + 1) + kc] : 0.0;
                        } else {
                            const int bc = (tj - TR) * 16 + (lane & 15);
                            b = (bc < ncol && kc < jb) ? W[(size_t)(j0 + kc) * ldw + k + bc] : 0.0;
                        }
                        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int row = ti * 16 + (lane >> 4) + 4 * r;
                        if (row >= nrow) continue;
                        const double v = cv[g][r] - acc[r];
                        if (tj < TR) {
                            const int col = tj * 16 + (lane & 15);
                            if (col <= row) W[(size_t)(t0 + row) * ldw + t0 + col] = v;
                        } else {
                            const int col = (tj - TR) * 16 + (lane & 15);
                            if (col < ncol) W[(size_t)(t0 + row) * ldw + k + col] = v;
                        }
                    }
                }
            }
            __syncthreads();
        }
        bad = (int)wave_max((double)bad);
        if (wv == 0 && lane == 0 && status) status[f] = bad ? RVGP_ST_NOT_SPD : RVGP_ST_OK;

        // ---- one coalesced pass over the rows of X = L^-1 (a wave per row):
        //      t = X b, and the column norms diag(A^-1)_c = sum_i X[i][c]^2
        //      accumulated per wave in LDS (the panel's space), then summed
        //      in wave order
        double* part = P;  // (ST / 64) x k partial sums
        for (int e = tid; e < (ST / 64) * k; e += ST) part[e] = 0.0;
        __syncthreads();
        for (int i = wv; i < k; i += ST / 64) {
            double s = 0.0;
            const double* xr = W + (size_t)i * ldw + k;
            for (int c = lane; c <= i; c += 64) {
                const double x = xr[c];
                s += x * bf[c];
                part[wv * k + c] += x * x;
            }
            s = wave_sum(s);
            if (lane == 0) tv[i] = s;
        }
        __syncthreads();
        for (int c = tid; c < k; c += ST) {
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < ST / 64; ++q) {
                s += part[q * k + c];
                part[q * k + c] = 0.0;
            }
            ainv[c] = s;
        }
        __syncthreads();
        // ---- w = X^T t, the same row pass
        for (int i = wv; i < k; i += ST / 64) {
            const double ti = tv[i];
            const double* xr = W + (size_t)i * ldw + k;
            for (int c = lane; c <= i; c += 64) part[wv * k + c] += xr[c] * ti;
        }
        __syncthreads();
        for (int c = tid; c < k; c += ST) {
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < ST / 64; ++q) s += part[q * k + c];
            wv_[c] = s;
        }
        __syncthreads();
        // ---- Gw = G w
        for (int i = wv; i < k; i += ST / 64) {
            double s = 0.0;
            for (int c = lane; c < k; c += 64) s += Gf[(size_t)i * k + c] * wv_[c];
            s = wave_sum(s);
            if (lane == 0) Gw[i] = s;
        }
        __syncthreads();

        // ---- NLML and adjoint (gp.hip weight-space finish, one right-hand side)
        const double Mf = Mrows[f];
        double bw = 0.0, wGw = 0.0, ld = 0.0, lS = 0.0, tr = 0.0;
        for (int j = tid; j < k; j += ST) {
            const double sj = S[j], wj = wv_[j];
            bw += bf[j] * wj;
            wGw += wj * Gw[j];
            ld += log(W[(size_t)j * ldw + j]);
            lS += log(sj);
            tr += ainv[j] / sj;
            gS[j] = 0.5 * (1.0 / sj - s2 * ainv[j] / (sj * sj) - wj * wj / (sj * sj));
        }
        bw = wg_sum<ST>(bw, sh);
        wGw = wg_sum<ST>(wGw, sh);
        ld = wg_sum<ST>(ld, sh);
        lS = wg_sum<ST>(lS, sh);
        tr = wg_sum<ST>(tr, sh);
        const double y2 = yy[f];
        const double nlml = 0.5 * (y2 - bw) / s2 + 0.5 * ((Mf - k) * log(s2) + lS + 2.0 * ld) +
                            0.5 * Mf * log(6.283185307179586);
        const double res2 = y2 - 2.0 * bw + wGw;
        const double gs2 = 0.5 * ((Mf - k) / s2 + tr - res2 / (s2 * s2));
        __syncthreads();
        double g0 = 0.0, g1 = 0.0, g2 = 0.0;
        for (int j = tid; j < k; j += ST) {
            g0 += gS[j] * dS[j];
            g1 += gS[j] * dS[k + j];
            g2 += gS[j] * dS[2 * k + j];
        }
        g0 = wg_sum<ST>(g0, sh);
        g1 = wg_sum<ST>(g1, sh);
        g2 = wg_sum<ST>(g2, sh);
        if (tid < 4) {
            const double gth = tid == 0 ? g0 : tid == 1 ? g1 : tid == 2 ? g2 : gs2;
            const double step = do_adam ? tstep[f] + 1.0 : 0.0;
            const double p1 = do_adam ? pow(b1, step) : 0.0, p2 = do_adam ? pow(b2, step) : 0.0;
            step_finish(tid, f, gth, nlml, 1.0 / (1.0 + exp(-uf[tid])), uf, trainable, m1, m2, tstep,
                        step, do_adam, lr, b1, b2, p1, p2, eps, out);
        }
        __syncthreads();
    }
}

// ------------------------------------------------------- step, A in LDS
// The same step with the factor in LDS, for fits of up to kLdsTiles 16-column
// blocks (k <= 160, 155 KB), `steps` of them in one launch.  G comes from memory
// (from a launch's second step on from L2); the last step leaves L and X = L^-1
// there for the predictions.  The 16 x 16 tiles of the lower triangle hold A
// right of the eliminated columns and X left of them, in place: step J turns its
// column of tiles into the panel P (kept aside) and then into X's.  Phase b
// solves the panel's rows and X's columns against L_JJ, one to a thread; phase c
// updates all tiles below on the matrix cores, while wave 0 updates the next
// diagonal tile first and factors it beside the products.  Two barriers a block.
// What bounds it is the chain of 16 pivots a block (3 us a block with the solve);
// a step of its own pays as much again for fetching instructions that it runs
// once, so each logarithm, power and exponential has one place, different threads
// bringing different arguments.  128 fits of k = 120: 232 -> 72 us a step of its
// own, 45 us in a launch of 50.  Past k = 160 the kernel above, from memory, is
// the only one.
constexpr int kLdsTiles = 10;
constexpr int kLdsST = 512;
constexpr int kTS = 16 * 17;  // doubles of a tile, rows padded to 17

// Sums of N values over the workgroup, in every thread.
template <int ST, int N>
__device__ __forceinline__ void wg_sum_n(double (&v)[N], double* sh) {
#pragma unroll
    for (int q = 0; q < N; ++q) v[q] = wave_sum_dpp(v[q]);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int q = 0; q < N; ++q) sh[(threadIdx.x >> 6) * N + q] = v[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < N; ++q) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < ST / 64; ++i) s += sh[i * N + q];
        v[q] = s;
    }
}

// One wave factors the 16 x 16 tile T = L L^T: lane i holds row i (every
// 16-lane row the same) and eliminates without square roots (a pivot's reciprocal by the hardware
// estimate and one cubic step is all that the next column waits for); the
// columns are scaled at the end, every lane taking one pivot's inverse square
// root.  L goes to Ld with 1 / L_ii in the padding column, L_ii to diag.
// Returns whether a pivot was not positive.
__device__ __forceinline__ int factor16(const double* T, double* Ld, double* diag, int lane) {
    const int i = lane & 15;
    double row[16], mine = 1.0;
    int bad = 0;
#pragma unroll
    for (int c = 0; c < 16; ++c) row[c] = T[i * 17 + c];
#pragma unroll
    for (int c = 0; c < 16; ++c) {
        double piv = row_bcast(row[c], c);
        const bool good = piv > 0.0;  // not positive definite (or NaN) otherwise
        bad |= !good;
        piv = good ? piv : 1.0;
        mine = i == c ? piv : mine;
        double r = __builtin_amdgcn_rcp(piv);
        const double e = fma(-piv, r, 1.0);
        r = fma(r, fma(e, e, e), r);
        const double m = row[c] * r;
#pragma unroll
        for (int l = c + 1; l < 16; ++l) row[l] = fma(-m, row_bcast(row[c], l), row[l]);
    }
    double r = __builtin_amdgcn_rsq(mine);
    double e = fma(-mine * r, r, 1.0);
    r = fma(r * e, fma(0.375, e, 0.5), r);
    double d = mine * r;
    d = fma(fma(-d, d, mine), 0.5 * r, d);
#pragma unroll
    for (int c = 0; c < 16; ++c) {
        const double rc = row_bcast(r, c);
        row[c] = i > c ? row[c] * rc : (i == c ? d : 0.0);
    }
    if (lane < 16) {
#pragma unroll
        for (int c = 0; c < 16; ++c) Ld[i * 17 + c] = row[c];
        Ld[i * 17 + 16] = r;
        diag[i] = d;
    }
    return bad;
}

// NQ: rows of G that a thread holds, at least ceil(k / PT).
template <int NQ>
__global__ __launch_bounds__(kLdsST) void batch_step_lds_kernel(
    int F, int k, int typ, const double* __restrict__ lam, double n_rows,
    const double* __restrict__ G, const double* __restrict__ bvec, const double* __restrict__ yy,
    const double* __restrict__ Mrows, const double* __restrict__ lower, double* __restrict__ u,
    const int* __restrict__ trainable, double* __restrict__ m1, double* __restrict__ m2,
    double* __restrict__ tstep, int do_adam, int steps, double lr, double b1, double b2, double eps,
    double* __restrict__ ws, double* __restrict__ out, int* __restrict__ status) {
    constexpr int ST = kLdsST;
    extern __shared__ double lds[];
    const int NT = (k + 15) >> 4, KP = 16 * NT, ntile = NT * (NT + 1) / 2;
    double* T = lds;                    // NT (NT + 1) / 2 tiles
    double* P = T + ntile * kTS;        // NT panel tiles; partial sums at the end
    double* Ld = P + NT * kTS;          // the diagonal factor
    double* S = Ld + kTS;               // KP doubles each from here
    double* bf = S + KP;
    double* diag = bf + KP;
    double* ainv = diag + KP;
    double* tv = ainv + KP;
    double* wl = tv + KP;
    __shared__ double sh[8 * (ST / 64)];
    __shared__ double th[4], pw[2], ls2;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m16 = lane & 15, kq = lane >> 4;
    // PT threads a row or column of the matrix: thread pp of column pc
    const int PT = min(ST / KP, NT), pc0 = tid % KP, pp0 = tid / KP;
    auto tile = [&](int ti, int tj) { return T + (ti * (ti + 1) / 2 + tj) * kTS; };

    for (int f = blockIdx.x; f < F; f += gridDim.x) {
        // opaque to the loop over fits and at each use: NQ kept addresses would spill
        int pc = pc0, pp = pp0;
        asm volatile("" : "+v"(pc), "+v"(pp));
        const double* Gf = G + (size_t)f * k * k;
        double* uf = u + 4 * (size_t)f;
        double* W = ws + (size_t)f * step_ws_doubles(k);  // [L | X] and the vectors, written only
        double* wsv = W + 2 * (size_t)k * k;
        const int ldw = 2 * k;

        // G by columns, thread pp the rows pp, pp + PT, ...; twice a step, each time
        // ahead of its use (held over the factorisation it would spill)
        double g[NQ];
        auto load_g = [&]() {
            asm volatile("" : "+v"(pc), "+v"(pp));
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int i = pp + PT * q;
                g[q] = i < k && pc < k && pp < PT ? Gf[(size_t)i * k + pc] : 0.0;
            }
        };
        const double done = do_adam ? tstep[f] : 0.0;
        for (int it = 0; it < steps; ++it) {
            const bool final = it + 1 == steps;  // the step that [L | X] and the vectors are left of
            load_g();
            // ---- theta = softplus(u) + lower, sigmoid(u)
            double sig = 0.0;
            const double step = done + it + 1.0;
            if (tid < 4) {
                const double x = uf[tid];
                const double e = exp(-fabs(x));
                sig = (x < 0.0 ? e : 1.0) / (1.0 + e);
                th[tid] = fmax(x, 0.0) + log1p(e) + lower[tid];
            }
            __syncthreads();
            const double nu = th[0], kappa = th[1], sf = th[2], s2 = th[3];

            // ---- spectral filter S (kernels.py:41-53; k <= ST), Adam's powers
            const bool adam = do_adam && tid >= ST - 2;
            double base = 1.0, r = 0.0;
            if (typ == 0 && tid < k) base = lam[tid] + 2.0 * nu / (kappa * kappa);
            if ((typ == 0 && tid < k) || adam)
                r = pow(adam ? (tid == ST - 1 ? b2 : b1) : base, adam ? step : -nu);
            if (adam) {
                pw[tid - (ST - 2)] = r;
                r = 0.0;
            }
            if (typ != 0 && tid < k) r = exp(-0.5 * lam[tid] * kappa * kappa);
            double sr[1] = {r};
            wg_sum_n<ST, 1>(sr, sh);
            if (tid < KP) {
                S[tid] = tid < k ? sf * n_rows * r / sr[0] : 1.0;
                bf[tid] = tid < k ? bvec[(size_t)f * k + tid] : 0.0;
            }
            __syncthreads();

            // ---- the lower tiles of G + diag(s2 / S), the identity past k
            asm volatile("" : "+v"(pc), "+v"(pp));
            if (pp < PT) {
                const double dd = pc < k ? s2 / S[pc] : 1.0;
                double* row = tile(pc >> 4, 0) + (pc & 15) * 17;  // G is symmetric
#pragma unroll
                for (int q = 0; q < NQ; ++q) {
                    const int i = pp + PT * q;
                    if (i <= (pc | 15)) row[(i >> 4) * kTS + (i & 15)] = g[q] + (i == pc ? dd : 0.0);
                }
            }
            __syncthreads();

            // ---- blocked Cholesky of A and X = L^-1, in place
            int bad = 0;
            for (int J = -1; J < NT; ++J) {
                if (J >= 0) {
                    // (b) panel rows P_i = A[i, J] L_JJ^-T, X[J, :] = L_JJ^-1 X[J, :]
                    const int nrow = 16 * (NT - J - 1), ncol = 16 * (J + 1), off = (nrow + 63) & ~63;
                    const bool isrow = tid < nrow, iscol = tid >= off && tid - off < ncol;
                    // lane i of each 16 holds row i of L_JJ and 1 / L_ii: broadcasts in
                    // the wave, as LDS would be the bound (136 reads a wave)
                    double lr[16];
                    const double rl = Ld[m16 * 17 + 16];
#pragma unroll
                    for (int c = 0; c < 16; ++c) lr[c] = Ld[m16 * 17 + c];
                    if (isrow || iscol) {
                        const int e = isrow ? tid : tid - off, eb = e >> 4, em = e & 15;
                        double* src = isrow ? tile(J + 1 + eb, J) + em * 17 : tile(J, eb) + em;
                        const int st = isrow ? 1 : 17;
                        const bool unit = iscol && eb == J;
                        double x[16];
#pragma unroll
                        for (int c = 0; c < 16; ++c) x[c] = unit ? (c == em ? 1.0 : 0.0) : src[c * st];
#pragma unroll
                        for (int c = 0; c < 16; ++c) {
                            x[c] *= row_bcast(rl, c);
#pragma unroll
                            for (int l = c + 1; l < 16; ++l) x[l] = fma(-x[c], row_bcast(lr[c], l), x[l]);
                        }
                        double* dst = isrow ? P + eb * kTS + em * 17 : src;
#pragma unroll
                        for (int c = 0; c < 16; ++c) dst[c * st] = x[c];
                    } else if (final && tid >= ST - 256) {  // past every row and column: L_JJ to memory
                        const int i = (tid >> 4) & 15, c = tid & 15, gi = 16 * J + i;
                        if (gi < k && c <= i) W[(size_t)gi * ldw + 16 * J + c] = Ld[i * 17 + c];
                    }
                    __syncthreads();
                    if (J + 1 == NT) break;
                }
                // (c) C[i, c] -= P_i Q_c for every tile of the rows below: Q_c = P_c^T
                //     right of the panel, X[J, c] left of it; C starts at 0 in its column
                const int q0 = (J + 1) * (J + 2) / 2;  // tile (J + 1, 0)
                auto update = [&](int q, int ti, int tj) {
                    double* C = T + q * kTS;
                    const double* Pi = P + (ti - J - 1) * kTS;
                    const bool right = tj > J;
                    const double* Q = right ? P + (tj - J - 1) * kTS : tile(J, tj);
                    dbl4 acc = dbl4{0, 0, 0, 0}, acc2 = acc;
                    if (tj != J) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[e] = C[(kq + 4 * e) * 17 + m16];
                    }
                    double av[4], bv[4];
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const int kc = 4 * s + kq;
                        av[s] = -Pi[m16 * 17 + kc];
                        bv[s] = Q[right ? m16 * 17 + kc : kc * 17 + m16];
                    }
                    // two chains of two products
                    acc2 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[0], bv[0], acc2, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[1], bv[1], acc, 0, 0, 0);
                    acc2 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[2], bv[2], acc2, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[3], bv[3], acc, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) C[(kq + 4 * e) * 17 + m16] = acc[e] + acc2[e];
                };
                if (wv == 0) {
                    if (J >= 0) update(q0 + J + 1, J + 1, J + 1);
                    // the tile's stores and loads are this wave's own, in order
                    bad |= factor16(tile(J + 1, J + 1), Ld, diag + 16 * (J + 1), lane);
                } else if (J >= 0) {
                    int ti = J + 1, tj = wv - 1;
                    for (int q = q0 + wv - 1; q < ntile; q += ST / 64 - 1, tj += ST / 64 - 1) {
                        while (tj > ti) tj -= ++ti;
                        if (q != q0 + J + 1) update(q, ti, tj);
                    }
                    for (int i = 4 * (wv - 1) + kq; final && i < 16 * (NT - J - 1); i += ST / 16 - 4) {  // P to memory
                        const int gi = 16 * (J + 1) + i;
                        if (gi < k) W[(size_t)gi * ldw + 16 * J + m16] = P[(i >> 4) * kTS + (i & 15) * 17 + m16];
                    }
                }
                __syncthreads();
            }
            if (tid == 0 && status) status[f] = bad ? RVGP_ST_NOT_SPD : RVGP_ST_OK;

            load_g();
            // ---- t = X b, diag(A^-1)_c = sum_i X[i][c]^2, w = X^T t, tile by tile
            //      (X is zero above its diagonal)
            double* pt = P;  // PT x KP partial sums, twice: at most P (PT <= NT, PT KP <= ST)
            double* pa = P + (size_t)PT * KP;
            const int mt = pc >> 4, mr = pc & 15;
            if (pp < PT) {
                double st = 0.0, sa = 0.0;
                for (int tj = pp; tj <= mt; tj += PT) {
                    const double* X = tile(mt, tj) + mr * 17;
#pragma unroll
                    for (int c = 0; c < 16; ++c) st = fma(X[c], bf[16 * tj + c], st);
                }
                for (int ti = mt + pp; ti < NT; ti += PT) {
                    const double* X = tile(ti, mt) + mr;
#pragma unroll
                    for (int e = 0; e < 16; ++e) sa = fma(X[e * 17], X[e * 17], sa);
                }
                pt[pp * KP + pc] = st;
                pa[pp * KP + pc] = sa;
            }
            for (int ti = wv; final && ti < NT; ti += ST / 64) {  // X to memory, zero above its diagonal
                for (int tj = 0; tj < NT; ++tj) {
                    const int c = 16 * tj + m16;
                    const double* X = tile(ti, min(ti, tj)) + kq * 17 + m16;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int i = 16 * ti + kq + 4 * e;
                        if (i < k && c < k) W[(size_t)i * ldw + k + c] = tj <= ti ? X[4 * e * 17] : 0.0;
                    }
                }
            }
            __syncthreads();
            if (tid < KP) {
                double st = 0.0, sa = 0.0;
                for (int q = 0; q < PT; ++q) {
                    st += pt[q * KP + tid];
                    sa += pa[q * KP + tid];
                }
                tv[tid] = st;
                ainv[tid] = sa;
            }
            __syncthreads();
            if (pp < PT) {
                double sw = 0.0;
                for (int ti = mt + pp; ti < NT; ti += PT) {
                    const double* X = tile(ti, mt) + mr;
#pragma unroll
                    for (int e = 0; e < 16; ++e) sw = fma(X[e * 17], tv[16 * ti + e], sw);
                }
                pt[pp * KP + pc] = sw;
            }
            __syncthreads();
            // ---- the logarithms of A's diagonal factor, S and the filter's base;
            //      the tiles are free by now
            double* lb = T;  // 3 x KP
            if (tid < KP) {
                double sw = 0.0;
                for (int q = 0; q < PT; ++q) sw += pt[q * KP + tid];
                wl[tid] = sw;
            }
            {
                const int part = tid / KP, at = tid % KP;
                const bool last = tid == ST - 1;  // 3 KP < ST
                if (part < 3 || last) {
                    double arg = last ? s2 : part == 0 ? base : part == 1 ? diag[at] : S[at];
                    arg = log(arg);
                    if (last) ls2 = arg;
                    else lb[tid] = arg;
                }
            }
            __syncthreads();
            // ---- G w by columns (G is symmetric)
            asm volatile("" : "+v"(pc), "+v"(pp));
            if (pp < PT) {
                double s = 0.0;
#pragma unroll
                for (int q = 0; q < NQ; ++q) s = fma(g[q], wl[min(pp + PT * q, KP - 1)], s);
                pa[pp * KP + pc] = s;
            }
            __syncthreads();

            // ---- NLML and adjoint (gp.hip weight-space finish, one right-hand side)
            double v[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
            double gs = 0.0, dn = 0.0, dk = 0.0, sj = 1.0, gw = 0.0;
            if (tid < k) {
                for (int q = 0; q < PT; ++q) gw += pa[q * KP + tid];
                const double wj = wl[tid], aj = ainv[tid];
                sj = S[tid];
                if (typ == 0) {
                    dn = -lb[tid] - nu * (2.0 / (kappa * kappa)) / base;
                    dk = 4.0 * nu * nu / (kappa * kappa * kappa * base);
                } else {
                    dk = -lam[tid] * kappa;
                }
                gs = 0.5 * (1.0 / sj - s2 * aj / (sj * sj) - wj * wj / (sj * sj));
                v[0] = bf[tid] * wj;
                v[1] = wj * gw;
                v[2] = lb[KP + tid];
                v[3] = lb[2 * KP + tid];
                v[4] = aj / sj;
                v[5] = r * dn;
                v[6] = r * dk;
                v[7] = gs * (sj / sf);
            }
            wg_sum_n<ST, 8>(v, sh);
            double gr[2] = {0.0, 0.0};
            if (tid < k) {
                const double d0 = sj * (dn - v[5] / sr[0]), d1 = sj * (dk - v[6] / sr[0]);
                gr[0] = gs * d0;
                gr[1] = gs * d1;
                const double vec[9] = {sj, d0, d1, sj / sf, gs, ainv[tid], tv[tid], wl[tid], gw};
                if (final) {
#pragma unroll
                    for (int q = 0; q < 9; ++q) wsv[q * k + tid] = vec[q];
                }
            }
            wg_sum_n<ST, 2>(gr, sh);
            if (tid < 4) {
                const double y2 = yy[f], Mf = Mrows[f];
                const double nlml = 0.5 * (y2 - v[0]) / s2 + 0.5 * ((Mf - k) * ls2 + v[3] + 2.0 * v[2]) +
                                    0.5 * Mf * 1.8378770664093454836;  // log(2 pi)
                const double res2 = y2 - 2.0 * v[0] + v[1];
                const double gs2 = 0.5 * ((Mf - k) / s2 + v[4] - res2 / (s2 * s2));
                const double gth = tid == 0 ? gr[0] : tid == 1 ? gr[1] : tid == 2 ? v[7] : gs2;
                step_finish(tid, f, gth, nlml, sig, uf, trainable, m1, m2, tstep, step, do_adam, lr, b1, b2,
                            pw[0], pw[1], eps, out);
            }
            __syncthreads();
        }
    }
}

template <int NB, int ST>
static size_t step_lds_bytes(int k) {
    // Ld, then the panel P (k x (NB + 1)), whose space also holds the
    // per-wave partial sums (ST / 64) x k of the final row passes
    const size_t pn = (size_t)k * (NB + 1) > (size_t)(ST / 64) * k ? (size_t)k * (NB + 1)
                                                                    : (size_t)(ST / 64) * k;
    return sizeof(double) * ((size_t)NB * (NB + 1) + pn);
}

template <int NB, int ST>
static int launch_step(int grid, int F, int k, int typ, const double* lam, double n_rows,
                       const double* G, const double* b, const double* yy, const double* M,
                       const double* lower, double* u, const int* trainable, double* m1,
                       double* m2, double* t, int do_adam, int steps, double lr, double b1,
                       double b2, double eps, double* ws, double* out, int* status, hipStream_t s) {
    const size_t lds = step_lds_bytes<NB, ST>(k);
    // 160 KiB of LDS per workgroup, less 1 KiB kept for the static arrays
    constexpr size_t kMaxDyn = 160 * 1024 - 1024;
    RVGP_CHECK_ARG(lds <= kMaxDyn, "rvgp_batch_step: k = %d needs %zu bytes of LDS with panel "
                                   "width %d (at most %zu); use a narrower panel",
                   k, lds, NB, kMaxDyn);
    // the LDS opt-in is raised to the 160 KiB maximum once per panel width
    // (not per launch: the launch may be under HIP graph capture)
    static bool opted_in = false;
    if (!opted_in) {
        RVGP_CHECK_HIP(hipFuncSetAttribute((const void*)batch_step_kernel<NB, ST>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxDyn));
        opted_in = true;
    }
    for (int i = 0; i < steps; ++i) {
        hipLaunchKernelGGL((batch_step_kernel<NB, ST>), dim3(grid), dim3(ST), lds, s, F, k, typ, lam, n_rows,
                           G, b, yy, M, lower, u, trainable, m1, m2, t, do_adam, lr, b1, b2, eps, ws,
                           out, status);
        RVGP_LAUNCH_CHECK();
    }
    return RVGP_OK;
}

// Panels of 16 with the factor in LDS where it fits (one workgroup shape); the
// launch above otherwise (k > 160) and for panels of 32.
template <int ST>
static int launch_step16(int grid, int F, int k, int typ, const double* lam, double n_rows,
                         const double* G, const double* b, const double* yy, const double* M,
                         const double* lower, double* u, const int* trainable, double* m1,
                         double* m2, double* t, int do_adam, int steps, double lr, double b1,
                         double b2, double eps, double* ws, double* out, int* status, hipStream_t s) {
    const int NT = (k + 15) / 16;
    if (NT > kLdsTiles)
        return launch_step<16, ST>(grid, F, k, typ, lam, n_rows, G, b, yy, M, lower, u, trainable, m1,
                                   m2, t, do_adam, steps, lr, b1, b2, eps, ws, out, status, s);
    constexpr auto bytes = [](int nt) {
        return (int)sizeof(double) * ((nt * (nt + 1) / 2 + nt + 1) * kTS + 6 * 16 * nt);
    };
    static_assert(bytes(kLdsTiles) <= 160 * 1024 - 2048, "LDS");
    // 128 columns leave 4 threads each, 160 leave 3: 32 or 54 rows a thread
    const auto kern = NT <= 8 ? batch_step_lds_kernel<32> : batch_step_lds_kernel<54>;
    static bool opted_in = false;  // once, as above
    if (!opted_in) {
        for (const auto fn : {batch_step_lds_kernel<32>, batch_step_lds_kernel<54>})
            RVGP_CHECK_HIP(hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                               bytes(kLdsTiles)));
        opted_in = true;
    }
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kLdsST), bytes(NT), s, F, k, typ, lam, n_rows, G, b, yy, M,
                       lower, u, trainable, m1, m2, t, do_adam, steps, lr, b1, b2, eps, ws, out, status);
    RVGP_LAUNCH_CHECK();
    return RVGP_OK;
}

template <int BT, int WT, typename TIn>
static int launch_gram(int F, int k, int d, const TIn* U, int ldu, const int* off,
                       const int* nodes, double* G, hipStream_t s) {
    const int T = (k + BT - 1) / BT;
    const int ntiles = T * (T + 1) / 2;
    const size_t total = (size_t)ntiles * F;
    RVGP_CHECK_ARG(total < (1u << 31), "rvgp_batch_gram: too many tiles");
    hipLaunchKernelGGL((batch_gram_kernel<BT, WT, TIn>), dim3((unsigned)total),
                       dim3((BT / WT) * (BT / WT) * 64), 0, s, F, k, d, U, ldu, off, nodes, ntiles,
                       T, G);
    RVGP_LAUNCH_CHECK();
    return RVGP_OK;
}

}  // namespace rvgp

using namespace rvgp;

extern "C" int rvgp_batch_gram(int f64, int F, int k, int d, const void* U, int ldu,
                               const int* node_off, const int* nodes, int tile, double* G,
                               void* stream) {
    RVGP_CHECK_ARG(F >= 1 && k >= 1 && d >= 1 && ldu >= k, "rvgp_batch_gram: bad sizes");
    hipStream_t s = as_stream(stream);
    if (f64) {
        const double* u = static_cast<const double*>(U);
        if (tile == 32) return launch_gram<32, 16, double>(F, k, d, u, ldu, node_off, nodes, G, s);
        if (tile == 64) return launch_gram<64, 32, double>(F, k, d, u, ldu, node_off, nodes, G, s);
        if (tile == 128) return launch_gram<128, 64, double>(F, k, d, u, ldu, node_off, nodes, G, s);
    } else {
        const float* u = static_cast<const float*>(U);
        if (tile == 32) return launch_gram<32, 16, float>(F, k, d, u, ldu, node_off, nodes, G, s);
        if (tile == 64) return launch_gram<64, 32, float>(F, k, d, u, ldu, node_off, nodes, G, s);
        if (tile == 128) return launch_gram<128, 64, float>(F, k, d, u, ldu, node_off, nodes, G, s);
    }
    RVGP_CHECK_ARG(false, "rvgp_batch_gram: tile must be 32, 64 or 128 (got %d)", tile);
    return RVGP_EINVAL;
}

extern "C" int rvgp_batch_rhs(int F, int k, int d, const double* U, int ldu, const int* node_off,
                              const int* nodes, const double* c, const double* ynorm2, double* b,
                              double* yy, void* stream) {
    RVGP_CHECK_ARG(F >= 1 && k >= 1 && d >= 1 && ldu >= k, "rvgp_batch_rhs: bad sizes");
    hipLaunchKernelGGL(batch_rhs_kernel, dim3(cdiv(k, 64), F), dim3(64 * kRhsWaves), 0, as_stream(stream), F, k,
                       d, U, ldu, node_off, nodes, c, ynorm2, b, yy);
    RVGP_LAUNCH_CHECK();
    return RVGP_OK;
}

extern "C" size_t rvgp_batch_step_ws_bytes(int F, int k) {
    return sizeof(double) * (size_t)(F > 0 ? F : 0) * step_ws_doubles(k > 0 ? k : 0);
}

extern "C" int rvgp_batch_steps(int F, int k, int typ, const double* evals, double n_rows,
                               const double* G, const double* b, const double* yy,
                               const double* M, const double* lower, double* u,
                               const int* trainable, double* m1, double* m2, double* t,
                               int do_adam, int steps, double lr, double b1, double b2, double eps,
                               int panel, int threads, int grid, double* ws, size_t ws_bytes,
                               double* out, int* status, void* stream) {
    RVGP_CHECK_ARG(F >= 1 && k >= 1, "rvgp_batch_step: bad sizes");
    RVGP_CHECK_ARG(typ == 0 || typ == 1, "rvgp_batch_step: typ must be 0 (matern) or 1 (se)");
    RVGP_CHECK_ARG(ws_bytes >= rvgp_batch_step_ws_bytes(F, k), "rvgp_batch_step: workspace too small");
    RVGP_CHECK_ARG(grid >= 1, "rvgp_batch_step: grid >= 1");
    RVGP_CHECK_ARG(steps >= 1, "rvgp_batch_steps: steps >= 1");
    const int g = grid < F ? grid : F;
    hipStream_t s = as_stream(stream);
#define RVGP_STEP(FN_)                                                                            \
    return FN_(g, F, k, typ, evals, n_rows, G, b, yy, M, lower, u, trainable, m1, m2, t, do_adam, steps, \
               lr, b1, b2, eps, ws, out, status, s)
    if (panel == 16 && threads == 512) RVGP_STEP(launch_step16<512>);
    if (panel == 16 && threads == 1024) RVGP_STEP(launch_step16<1024>);
    if (panel == 32 && threads == 512) RVGP_STEP((launch_step<32, 512>));
    if (panel == 32 && threads == 1024) RVGP_STEP((launch_step<32, 1024>));
#undef RVGP_STEP
    RVGP_CHECK_ARG(false, "rvgp_batch_step: (panel, threads) must be 16 or 32 and 512 or 1024 "
                          "(got %d, %d)", panel, threads);
    return RVGP_EINVAL;
}

extern "C" int rvgp_batch_step(int F, int k, int typ, const double* evals, double n_rows,
                               const double* G, const double* b, const double* yy,
                               const double* M, const double* lower, double* u,
                               const int* trainable, double* m1, double* m2, double* t,
                               int do_adam, double lr, double b1, double b2, double eps,
                               int panel, int threads, int grid, double* ws, size_t ws_bytes,
                               double* out, int* status, void* stream) {
    return rvgp_batch_steps(F, k, typ, evals, n_rows, G, b, yy, M, lower, u, trainable, m1, m2, t,
                            do_adam, 1, lr, b1, b2, eps, panel, threads, grid, ws, ws_bytes, out, status,
                            stream);
}
