// Symmetric eigendecomposition A = V diag(w) V^T (FP64, w ascending) of the
// small projected matrices of the eigensolver's Rayleigh-Ritz step -- the
// dense eigenproblem ARPACK solves inside scipy.sparse.linalg.eigsh, reached
// from RVGP/geometry.py:73.
//
// Three stages, all on the device:
//  1. Householder tridiagonalisation Q^T A Q = T (LAPACK sytd2, lower), one
//     kernel launch per column on up to 64 workgroups that each own a cyclic
//     slab of rows: a launch finishes the previous column's rank-2 update on
//     its rows while forming the next reflector, so the launch boundary is
//     the only synchronisation between workgroups (no device-scope spinning,
//     which on gfx950 means writing back and invalidating L2 that a
//     concurrent stream is using).  Up to kSmallN the matrix fits one
//     workgroup's registers and one launch does all columns.
//  2. Eigenvalues of T by multisection (one wavefront per eigenvalue, its 64
//     lanes evaluating Sturm counts at 64 interior points, ~9 rounds to full
//     precision); eigenvectors of T by inverse iteration, one wavefront per
//     eigenvalue, with modified Gram-Schmidt inside clusters of eigenvalues
//     closer than 1e-7 |T| (elsewhere the vectors are orthogonal to rounding
//     over the gap).
//  3. V = Q Z: the reflectors are applied in blocks of NB in compact WY form
//     (I - Vb Tb Vb^T) by one kernel, each workgroup carrying a few columns
//     of Z in LDS through all the blocks.
#include "common.h"

namespace rvgp {

constexpr int kSyevNB = 32;        // reflectors per compact-WY block
constexpr int kSyevMaxN = 2048;   // inverse iteration holds 6.5 n doubles in LDS

// Column j of the tridiagonalisation (LAPACK sytd2, lower), one launch per
// column on G workgroups; workgroup g owns the rows r = g (mod G) of the
// work matrix W (full symmetric storage).  The launch boundary is the only
// synchronisation between workgroups.  Launch j
//   1. finishes column j-1: w = p - (tau/2)(p^T v) v from the previous
//      launch's p (each owner wrote its rows) and partial sums of p^T v;
//   2. forms row j of the updated matrix W - v w^T - w v^T and from it the
//      reflector v_j, tau_j, d_j, e_j -- redundantly in every workgroup (the
//      same arithmetic in the same order, so every copy is identical);
//   3. applies column j-1's rank-2 update to its own rows r > j (row j is
//      consumed by step 2 and never read again) and, in the same pass,
//      p_r = tau_j W'[r][j+1:] v_j and its share of p^T v.
// Vectors of column j are indexed from row j+1; buffers alternate by parity.
constexpr int kStepThreads = 256;
constexpr int kStepGroups = 64;
constexpr int kStepGroupsMax = 128;
constexpr int kStepChunks = kSyevMaxN / 64;

__global__ __launch_bounds__(kStepThreads) void sytrd_step_kernel(
    int n, double* __restrict__ W, int ldw, int j, double* __restrict__ vbuf,
    double* __restrict__ pbuf, double* __restrict__ sbuf, double* __restrict__ VhT,
    double* __restrict__ d, double* __restrict__ e, double* __restrict__ tau) {
    extern __shared__ double sm[];
    const int G = gridDim.x, g = blockIdx.x;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    constexpr int NW = kStepThreads / 64;
    const int m0 = n - j;        // rows j..n-1: column j-1's vectors, index i <-> row j+i
    const int m = n - j - 1;     // column j's reflector, index i <-> row j+1+i
    double* wprev = sm;          // m0
    double* vprev = wprev + n;   // m0
    double* row = vprev + n;     // m0: row j of the updated matrix, columns j..
    double* v = row + n;         // m
    double* red = v + n;         // 2 * NW
    const int cur = j & 1, prv = cur ^ 1;
    // 1. column j-1's w
    double kk = 0.0, tprev = 0.0;
    if (j > 0) {
        tprev = tau[j - 1];
        double sp = 0.0;
        for (int q = t; q < G; q += kStepThreads) sp += sbuf[(size_t)prv * G + q];
        sp = wave_sum(sp);
        if (lane == 0) red[wv] = sp;
        __syncthreads();
        for (int q = 0; q < NW; ++q) kk += red[q];
        kk *= 0.5 * tprev;
        const double* vp = vbuf + (size_t)prv * n;
        const double* pp = pbuf + (size_t)prv * n;
        for (int i = t; i < m0; i += kStepThreads) {
            const double vi = vp[i];
            vprev[i] = vi;
            wprev[i] = pp[i] - kk * vi;
        }
    }
    __syncthreads();
    // 2. row j (columns j..n-1) after column j-1's update, and its reflector
    for (int c = t; c < m0; c += kStepThreads) {
        double a = W[(size_t)j * ldw + j + c];
        if (j > 0) a -= vprev[0] * wprev[c] + wprev[0] * vprev[c];
        row[c] = a;
    }
    __syncthreads();
    double s2 = 0.0;
    for (int i = 2 + t; i <= m; i += kStepThreads) s2 += row[i] * row[i];
    s2 = wave_sum(s2);
    if (lane == 0) red[NW + wv] = s2;
    __syncthreads();
    s2 = 0.0;
    for (int q = 0; q < NW; ++q) s2 += red[NW + q];
    const double alpha = m >= 1 ? row[1] : 0.0;
    double beta, tj, scal;
    if (s2 == 0.0) {
        tj = 0.0;
        beta = alpha;
        scal = 0.0;
    } else {
        beta = -copysign(sqrt(alpha * alpha + s2), alpha);
        tj = (beta - alpha) / beta;
        scal = 1.0 / (alpha - beta);
    }
    for (int i = t; i < m; i += kStepThreads) v[i] = i == 0 ? 1.0 : row[1 + i] * scal;
    __syncthreads();
    if (g == 0) {
        for (int i = t; i < m; i += kStepThreads) {
            vbuf[(size_t)cur * n + i] = v[i];
            VhT[(size_t)j * n + j + 1 + i] = v[i];
        }
        if (t == 0) {
            d[j] = row[0];
            e[j] = beta;
            tau[j] = tj;
        }
    }
    // 3. own rows r > j: update with column j-1's vectors, then p_r
    double dot = 0.0;
    const int rfirst = j + 1 + ((g - (j + 1) % G) % G + G) % G;  // first r > j with r = g (mod G)
    // a row's columns are loaded in one batch (kStepChunks per lane), so a
    // row costs one memory latency instead of one per 64 columns
    for (int r = rfirst + wv * G; r < n; r += NW * G) {
        const int ir = r - j;        // index of row r in column j-1's vectors
        const double vr = j > 0 ? vprev[ir] : 0.0, wr = j > 0 ? wprev[ir] : 0.0;
        double* Wr = W + (size_t)r * ldw + (j + 1);
        double a[kStepChunks];
#pragma unroll
        for (int q = 0; q < kStepChunks; ++q) {
            const int c = lane + 64 * q;
            a[q] = c < m ? Wr[c] : 0.0;
        }
        double acc = 0.0;
#pragma unroll
        for (int q = 0; q < kStepChunks; ++q) {
            const int c = lane + 64 * q;
            if (c < m) {
                double x = a[q];
                if (j > 0) {
                    x -= vr * wprev[c + 1] + wr * vprev[c + 1];
                    Wr[c] = x;
                }
                acc += x * v[c];
            }
        }
        acc = wave_sum(acc);
        if (lane == 0) {
            const double pr = tj * acc;
            pbuf[(size_t)cur * n + (r - j - 1)] = pr;
            dot += v[r - j - 1] * pr;
        }
        if (j == n - 2 && r == n - 1 && lane == 0) d[n - 1] = Wr[0];
    }
    dot = wave_sum(dot);
    __syncthreads();
    if (lane == 0) red[wv] = dot;
    __syncthreads();
    if (t == 0) {
        double sacc = 0.0;
        for (int q = 0; q < NW; ++q) sacc += red[q];
        sbuf[(size_t)cur * G + g] = sacc;
    }
}

// The same column step with every input of the launch loaded in one batch
// at its start -- the workgroup's own rows (at most RPW per wavefront) into
// registers, row j, column j-1's p and v and the partial sums -- so a launch
// waits on memory once, not once per dependent stage.  For n <= 1024
// (grid of up to 128 workgroups, 16 column chunks per lane).
template <int RPW, int CH>
__global__ __launch_bounds__(kStepThreads) void sytrd_step_prefetch_kernel(
    int n, double* __restrict__ W, int ldw, int j, double* __restrict__ vbuf,
    double* __restrict__ pbuf, double* __restrict__ sbuf, double* __restrict__ VhT,
    double* __restrict__ d, double* __restrict__ e, double* __restrict__ tau) {
    extern __shared__ double sm[];
    const int G = gridDim.x, g = blockIdx.x;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    constexpr int NW = kStepThreads / 64;
    constexpr int PT = (64 * CH + kStepThreads - 1) / kStepThreads;  // row-j entries per thread
    const int m0 = n - j;
    const int m = n - j - 1;
    double* wprev = sm;
    double* vprev = wprev + n;
    double* row = vprev + n;
    double* v = row + n;
    double* red = v + n;
    const int cur = j & 1, prv = cur ^ 1;
    // ---- every load of the launch, issued together
    const int rfirst = j + 1 + ((g - (j + 1) % G) % G + G) % G;
    double a[RPW][CH];
#pragma unroll
    for (int k = 0; k < RPW; ++k) {
        const int r = rfirst + (wv + NW * k) * G;
        const double* Wr = W + (size_t)(r < n ? r : 0) * ldw + (j + 1);
#pragma unroll
        for (int q = 0; q < CH; ++q) {
            const int c = lane + 64 * q;
            a[k][q] = (r < n && c < m) ? Wr[c] : 0.0;
        }
    }
    double rj[PT], pp[PT], vp[PT];
#pragma unroll
    for (int k = 0; k < PT; ++k) {
        const int c = t + kStepThreads * k;
        const bool ok = c < m0;
        rj[k] = ok ? W[(size_t)j * ldw + j + c] : 0.0;
        pp[k] = (ok && j > 0) ? pbuf[(size_t)prv * n + c] : 0.0;
        vp[k] = (ok && j > 0) ? vbuf[(size_t)prv * n + c] : 0.0;
    }
    const double sp = (j > 0 && t < G) ? sbuf[(size_t)prv * G + t] : 0.0;
    const double tprev = j > 0 ? tau[j - 1] : 0.0;
    // ---- column j-1's w
    double kk = wave_sum(sp);
    if (lane == 0) red[wv] = kk;
    __syncthreads();
    kk = 0.0;
    for (int q = 0; q < NW; ++q) kk += red[q];
    kk *= 0.5 * tprev;
#pragma unroll
    for (int k = 0; k < PT; ++k) {
        const int c = t + kStepThreads * k;
        if (c < m0) {
            vprev[c] = vp[k];
            wprev[c] = pp[k] - kk * vp[k];
        }
    }
    __syncthreads();
    // ---- row j after column j-1's update, and its reflector
    double s2 = 0.0;
#pragma unroll
    for (int k = 0; k < PT; ++k) {
        const int c = t + kStepThreads * k;
        if (c < m0) {
            double x = rj[k];
            if (j > 0) x -= vprev[0] * wprev[c] + wprev[0] * vprev[c];
            row[c] = x;
            if (c >= 2) s2 += x * x;
        }
    }
    s2 = wave_sum(s2);
    if (lane == 0) red[NW + wv] = s2;
    __syncthreads();
    s2 = 0.0;
    for (int q = 0; q < NW; ++q) s2 += red[NW + q];
    const double alpha = row[1];
    double beta, tj, scal;
    if (s2 == 0.0) {
        tj = 0.0;
        beta = alpha;
        scal = 0.0;
    } else {
        beta = -copysign(sqrt(alpha * alpha + s2), alpha);
        tj = (beta - alpha) / beta;
        scal = 1.0 / (alpha - beta);
    }
    for (int i = t; i < m; i += kStepThreads) v[i] = i == 0 ? 1.0 : row[1 + i] * scal;
    __syncthreads();
    if (g == 0) {
        for (int i = t; i < m; i += kStepThreads) {
            vbuf[(size_t)cur * n + i] = v[i];
            VhT[(size_t)j * n + j + 1 + i] = v[i];
        }
        if (t == 0) {
            d[j] = row[0];
            e[j] = beta;
            tau[j] = tj;
        }
    }
    // ---- own rows: column j-1's update, then p_r
    double dot = 0.0;
#pragma unroll
    for (int k = 0; k < RPW; ++k) {
        const int r = rfirst + (wv + NW * k) * G;
        if (r < n) {
            const int ir = r - j;
            const double vr = j > 0 ? vprev[ir] : 0.0, wr = j > 0 ? wprev[ir] : 0.0;
            double* Wr = W + (size_t)r * ldw + (j + 1);
            double acc = 0.0;
#pragma unroll
            for (int q = 0; q < CH; ++q) {
                const int c = lane + 64 * q;
                if (c < m) {
                    double x = a[k][q];
                    if (j > 0) {
                        x -= vr * wprev[c + 1] + wr * vprev[c + 1];
                        Wr[c] = x;
                    }
                    acc += x * v[c];
                }
            }
            acc = wave_sum(acc);
            if (lane == 0) {
                const double pr = tj * acc;
                pbuf[(size_t)cur * n + (r - j - 1)] = pr;
                dot += v[r - j - 1] * pr;
                if (j == n - 2 && r == n - 1) d[n - 1] = Wr[0];
            }
        }
    }
    dot = wave_sum(dot);
    __syncthreads();
    if (lane == 0) red[wv] = dot;
    __syncthreads();
    if (t == 0) {
        double sacc = 0.0;
        for (int q = 0; q < NW; ++q) sacc += red[q];
        sbuf[(size_t)cur * G + g] = sacc;
    }
}

// W <- A (full symmetric storage), row stride ldw.
__global__ __launch_bounds__(256) void copy_full_kernel(int n, const double* __restrict__ A, int lda,
                                                        double* __restrict__ W, int ldw) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)n * n) return;
    const int r = (int)(e / n), c = (int)(e - (size_t)r * n);
    W[(size_t)r * ldw + c] = A[(size_t)r * lda + c];
}

__global__ void fill_kernel(size_t cnt, double* __restrict__ p, double val) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cnt) p[i] = val;
}

// 1 / x by the hardware estimate and two Newton steps (a few units in the last
// place): the divisions below sit on chains of n dependent steps, where the
// IEEE sequence costs twice as much (stebz at n = 576: 369 -> 322 us).
__device__ __forceinline__ double rcp_nr(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}

// The whole tridiagonalisation of a matrix of n <= kSmallN in one workgroup,
// the matrix in registers: wave v of NW owns the columns c = v (mod NW), lane
// i of it the rows i + 64 k (k < R) of its C columns.  In step j every wave
// holds the step's v, w and the next reflector u; one pass over its columns
// applies the rank-2 update and accumulates the next product, and the one
// column that the next reflector comes from goes through LDS (one barrier a
// step; its two buffers alternate).  What is left is the chain of a step (the
// barrier, NW partial products from LDS, two wave sums, the reflector's square
// root and reciprocal), which every wave runs: a wave on each SIMD (NW = 4)
// while its columns fit, as more waves only repeat the chain on the same SIMD
// (16 waves: 109 us at n = 64, 4: 67 us).  A launch is 5.2 us a column, a step
// here 1.05 us (n = 64) to 2.6 us (n = 192); the whole solve takes 516 -> 154
// us at n = 64, 994 -> 374 us at 128, 1540 -> 729 us at 192 (200: 1600 ->
// 1260 us, the other stages).  Past 192 the columns no longer fit the
// registers of 8 waves.
constexpr int kSmallN = 192;

// The reflector of the column x (rows from `first` on): v with v[first] = 1
// in place of x, and tau, beta as LAPACK's dlarfg gives them.
template <int R>
__device__ __forceinline__ void small_reflector(double (&x)[R], int lane, int first, double& beta,
                                                double& tau) {
    double alpha = 0.0, s2 = 0.0;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int i = lane + 64 * k;
        if ((first >> 6) == k) alpha = bcast(x[k], first & 63);
        x[k] = i < first ? 0.0 : x[k];
        s2 += i == first ? 0.0 : x[k] * x[k];
    }
    s2 = wave_sum_dpp(s2);
    beta = alpha;
    tau = 0.0;
    double scal = 0.0;
    if (s2 != 0.0) {
        const double nn = fma(alpha, alpha, s2);
        double r = __builtin_amdgcn_rsq(nn);
        r *= fma(-0.5 * nn * r, r, 1.5);
        r *= fma(-0.5 * nn * r, r, 1.5);
        double nrm = nn * r;
        nrm = fma(fma(-nrm, nrm, nn), 0.5 * r, nrm);
        beta = -copysign(nrm, alpha);
        tau = fma(fabs(alpha), r, 1.0);
        scal = copysign(rcp_nr(fabs(alpha) + nrm), alpha);
    }
#pragma unroll
    for (int k = 0; k < R; ++k) x[k] = lane + 64 * k == first ? 1.0 : x[k] * scal;
}

template <int R>
__device__ __forceinline__ double pick(const double (&x)[R], int i) {
    double v = bcast(x[0], i & 63);
#pragma unroll
    for (int k = 1; k < R; ++k) v = (i >> 6) == k ? bcast(x[k], i & 63) : v;
    return v;
}

template <int R, int NW>
__global__ __launch_bounds__(64 * NW) void sytrd_small_kernel(int n, const double* __restrict__ A,
                                                              int lda, double* __restrict__ VhT,
                                                              double* __restrict__ d,
                                                              double* __restrict__ e,
                                                              double* __restrict__ tau) {
    constexpr int C = 64 * R / NW, CG = 4;  // columns of a wave, and of one uniform skip
    __shared__ double part[2][NW][64 * R];
    __shared__ double next[2][64 * R];  // the column of the next reflector
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double W[C][R], u[R], p[R], nx[R];
#pragma unroll
    for (int q = 0; q < C; ++q) {
        const int c = wv + NW * q;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int i = lane + 64 * k;
            W[q][k] = i < n && c < n ? A[(size_t)c * lda + i] : 0.0;
        }
    }
    // the first column's reflector, its product
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int i = lane + 64 * k;
        u[k] = i < n ? A[i] : 0.0;
        p[k] = 0.0;
        if (wv == 1 % NW) next[0][i] = W[0][k];
    }
    double dj = bcast(u[0], 0), beta = 0.0, tj = 0.0;
    if (n > 1) small_reflector<R>(u, lane, 1, beta, tj);
#pragma unroll
    for (int q = 0; q < C; ++q) {
        const double uc = bcast(u[NW * q / 64], (wv + NW * q) & 63);  // column wv + NW q
#pragma unroll
        for (int k = 0; k < R; ++k) p[k] = fma(W[q][k], uc, p[k]);
    }
#pragma unroll
    for (int k = 0; k < R; ++k) part[0][wv][lane + 64 * k] = p[k];
    for (int j = 0; j + 1 < n; ++j) {
        const int buf = j & 1;
        if (wv == (j & (NW - 1))) {  // the outputs of step j, a wave in turn
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const int i = lane + 64 * k;
                if (i > j && i < n) VhT[(size_t)j * n + i] = u[k];
            }
            if (lane == 0) {
                d[j] = dj;
                e[j] = beta;
                tau[j] = tj;
            }
        }
        __syncthreads();
        double w[R], v[R], x[R], dot = 0.0;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            double t = 0.0;
#pragma unroll
            for (int q = 0; q < NW; ++q) t += part[buf][q][lane + 64 * k];
            v[k] = u[k];
            w[k] = lane + 64 * k > j ? tj * t : 0.0;
            x[k] = next[buf][lane + 64 * k];
            dot = fma(w[k], v[k], dot);
        }
        const double kk = 0.5 * tj * wave_sum_dpp(dot);
#pragma unroll
        for (int k = 0; k < R; ++k) w[k] = fma(-kk, v[k], w[k]);
        // column j + 1 with this step's update (v there is 1)
        const double w1 = pick<R>(w, j + 1);
#pragma unroll
        for (int k = 0; k < R; ++k) u[k] = x[k] - fma(w1, v[k], w[k]);
        dj = pick<R>(u, j + 1);
        if (j + 2 >= n) break;
        small_reflector<R>(u, lane, j + 2, beta, tj);
#pragma unroll
        for (int k = 0; k < R; ++k) {
            p[k] = 0.0;
            nx[k] = 0.0;
        }
        // finished columns and those past n carry zeros in v, w or u: no test
#pragma unroll
        for (int g = 0; g < C; g += CG) {
            if (NW * (g + CG) > j + 2 && NW * g < n) {
#pragma unroll
                for (int q = g; q < g + CG; ++q) {
                    constexpr int S = 64 / NW;
                    const int at = (wv + NW * q) & 63;
                    const double vc = bcast(v[q / S], at), wc = bcast(w[q / S], at);
                    const double uc = bcast(u[q / S], at);
                    const bool pub = wv + NW * q == j + 2;
#pragma unroll
                    for (int k = 0; k < R; ++k) {
                        W[q][k] = fma(-wc, v[k], fma(-vc, w[k], W[q][k]));
                        p[k] = fma(W[q][k], uc, p[k]);
                        nx[k] = pub ? W[q][k] : nx[k];
                    }
                }
            }
        }
        const bool own = wv == ((j + 2) & (NW - 1));
#pragma unroll
        for (int k = 0; k < R; ++k) {
            part[buf ^ 1][wv][lane + 64 * k] = p[k];
            if (own) next[buf ^ 1][lane + 64 * k] = nx[k];
        }
    }
    if (threadIdx.x == 0) d[n - 1] = dj;
}

// Number of eigenvalues of T below x (Sturm sequence of the LDL^T pivots,
// with LAPACK's pivmin safeguard against zero pivots).
__device__ __forceinline__ int sturm_count(int n, const double* dd, const double* e2, double x,
                                           double pivmin) {
    double q = dd[0] - x;
    if (fabs(q) <= pivmin) q = -pivmin;
    int c = q < 0.0;
    for (int i = 1; i < n; ++i) {
        q = fma(-e2[i - 1], rcp_nr(q), dd[i] - x);
        if (fabs(q) <= pivmin) q = -pivmin;
        c += q < 0.0;
    }
    return c;
}

// Eigenvalue i of T (ascending) per wavefront: 64-point multisection of the
// Gershgorin interval.  bounds = (lower, upper, pivmin) from tri_bounds_kernel.
__global__ __launch_bounds__(64) void stebz_kernel(int n, const double* __restrict__ d,
                                                   const double* __restrict__ e,
                                                   const double* __restrict__ bounds,
                                                   double* __restrict__ w) {
    extern __shared__ double sm[];
    double* dd = sm;
    double* e2 = sm + n;
    const int lane = threadIdx.x;
    const int i = blockIdx.x;
    for (int q = lane; q < n; q += 64) {
        dd[q] = d[q];
        if (q < n - 1) e2[q] = e[q] * e[q];
    }
    __syncthreads();
    const double pivmin = bounds[2];
    double lo = bounds[0], hi = bounds[1];
    for (int round = 0; round < 24; ++round) {
        const double tol = 2.0 * 2.2204460492503131e-16 * fmax(fabs(lo), fabs(hi)) + 2.0 * pivmin;
        if (hi - lo <= tol) break;
        const double x = lo + (hi - lo) * (double)(lane + 1) / 65.0;
        const int c = sturm_count(n, dd, e2, x, pivmin);
        // lanes with count(x) <= i lie below eigenvalue i; counts grow with
        // the lane, and only the leading run of such lanes is trusted
        const unsigned long long below = __ballot(c <= i);
        const int nb = below == ~0ull ? 64 : __builtin_ctzll(~below);
        const double nlo = nb > 0 ? lo + (hi - lo) * (double)nb / 65.0 : lo;
        const double nhi = nb < 64 ? lo + (hi - lo) * (double)(nb + 1) / 65.0 : hi;
        lo = nlo;
        hi = nhi;
    }
    if (lane == 0) w[i] = 0.5 * (lo + hi);
}

__global__ __launch_bounds__(256) void tri_bounds_kernel(int n, const double* __restrict__ d,
                                                         const double* __restrict__ e,
                                                         double* __restrict__ bounds) {
    __shared__ double slo[256], shi[256], se[256];
    double lo = 1e300, hi = -1e300, em = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) {
        const double a = i > 0 ? fabs(e[i - 1]) : 0.0;
        const double b = i < n - 1 ? fabs(e[i]) : 0.0;
        lo = fmin(lo, d[i] - a - b);
        hi = fmax(hi, d[i] + a + b);
        if (i < n - 1) em = fmax(em, e[i] * e[i]);
    }
    slo[threadIdx.x] = lo;
    shi[threadIdx.x] = hi;
    se[threadIdx.x] = em;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            slo[threadIdx.x] = fmin(slo[threadIdx.x], slo[threadIdx.x + s]);
            shi[threadIdx.x] = fmax(shi[threadIdx.x], shi[threadIdx.x + s]);
            se[threadIdx.x] = fmax(se[threadIdx.x], se[threadIdx.x + s]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double tn = fmax(fabs(slo[0]), fabs(shi[0]));
        const double widen = 2.2204460492503131e-16 * tn * (2.0 * n + 2.0) + 1e-300;
        bounds[0] = slo[0] - widen;
        bounds[1] = shi[0] + widen;
        bounds[2] = 2.2250738585072014e-308 * fmax(1.0, se[0]) / 2.2204460492503131e-16;
        bounds[3] = tn;
    }
}

// Eigenvectors of T by inverse iteration (LAPACK stein): one wavefront per
// cluster leader.  A cluster is a run of eigenvalues with consecutive gaps
// below 1e-7 |T|; its members are computed in order, each iterate
// orthogonalised (modified Gram-Schmidt) against the members before it.
// Eigenvector i is written to row i of Zt (n x n).  The tridiagonal
// factorisation with partial pivoting (dlagtf) and the solves (dlagts) are
// chains of n dependent steps: every lane walks them with the running row in
// registers, the operands of kWalk steps are read from LDS ahead of them, and
// the pivots' reciprocals are kept so that no solve divides.  n = 576: 650 ->
// 247 us, n = 64: 75 -> 25 us (a cluster of four takes four times that).
constexpr int kWalk = 8;

__global__ __launch_bounds__(64) void stein_kernel(int n, const double* __restrict__ d,
                                                   const double* __restrict__ e,
                                                   const double* __restrict__ w,
                                                   const double* __restrict__ bounds,
                                                   double* __restrict__ Zt) {
    extern __shared__ double sm[];
    // arrays of np doubles: entries past n are the identity's, so that the
    // walks run in whole strides
    const int np = (n + kWalk - 1) / kWalk * kWalk + kWalk;
    double* ra = sm;          // 1 / U diagonal
    double* b = ra + np;      // U first super-diagonal
    double* c = b + np;       // multipliers
    double* dd = c + np;      // U second super-diagonal
    double* z = dd + np;      // iterate
    double* y = z + np;       // the iterate between the two solves; the factorisation's T
    int* piv = reinterpret_cast<int*>(y + np);
    const int lane = threadIdx.x;
    const int i0 = blockIdx.x;
    const double tn = bounds[3];
    const double ctol = 1e-7 * tn;
    if (i0 > 0 && w[i0] - w[i0 - 1] <= ctol) return;  // not a cluster leader
    int i1 = i0 + 1;
    while (i1 < n && w[i1] - w[i1 - 1] <= ctol) ++i1;
    const double eps = 2.2204460492503131e-16;
    // pivot floor: eps |T|, and a normal number even for T = 0
    const double delta = eps * fmax(tn, 1e-200);
    double lam_prev = -1e300;
    for (int i = i0; i < i1; ++i) {
        // equal eigenvalues of a cluster are separated so that their shifted
        // systems differ (LAPACK stein)
        double lam = w[i];
        if (i > i0 && lam - lam_prev < 10.0 * eps * fabs(lam) + delta) lam = lam_prev + 10.0 * eps * fabs(lam) + delta;
        lam_prev = lam;
        for (int k = lane; k < np; k += 64) {
            y[k] = k < n ? d[k] - lam : 1.0;      // diagonal
            z[k] = k < n - 1 ? e[k] : 0.0;        // off-diagonal
        }
        __syncthreads();
        double ak = y[0], bk = z[0];  // row k of U in the making
        for (int k0 = 0; k0 < n; k0 += kWalk) {
            double de[kWalk], ee[kWalk + 1];
#pragma unroll
            for (int q = 0; q < kWalk; ++q) {
                de[q] = y[k0 + q + 1];
                ee[q] = z[k0 + q];
            }
            ee[kWalk] = z[k0 + kWalk];
            double r[kWalk], bo[kWalk], mo[kWalk], so[kWalk];
            int po[kWalk];
#pragma unroll
            for (int q = 0; q < kWalk; ++q) {
                const double ck = ee[q], dn = de[q], en = ee[q + 1];
                const bool swap = fmax(fabs(ak), delta) < fabs(ck);
                const double floored = fabs(ak) < delta ? copysign(delta, ak == 0.0 ? 1.0 : ak) : ak;
                r[q] = rcp_nr(swap ? ck : floored);
                const double mult = (swap ? ak : ck) * r[q];
                bo[q] = swap ? dn : bk;
                so[q] = swap ? en : 0.0;
                mo[q] = mult;
                po[q] = swap;
                const double na = fma(-mult, swap ? dn : bk, swap ? bk : dn);
                bk = swap ? -mult * en : en;
                ak = na;
            }
            if (lane == 0) {
#pragma unroll
                for (int q = 0; q < kWalk; ++q) {
                    ra[k0 + q] = r[q];
                    b[k0 + q] = bo[q];
                    c[k0 + q] = mo[q];
                    dd[k0 + q] = so[q];
                    piv[k0 + q] = po[q];
                }
            }
        }
        __syncthreads();
        // deterministic, non-degenerate starting vector
        for (int k = lane; k < np; k += 64) {
            const unsigned h = (unsigned)(k * 2654435761u) ^ (unsigned)(i * 40503u + 17u);
            z[k] = k < n ? 0.5 + (double)(h & 0xffff) / 65536.0 : 0.0;
        }
        __syncthreads();
        for (int it = 0; it < 3; ++it) {
            // forward: the row interchanges and multipliers, z -> y
            double zk = z[0];
            for (int k0 = 0; k0 < n; k0 += kWalk) {
                double zn[kWalk], ck[kWalk];
                int pk[kWalk];
#pragma unroll
                for (int q = 0; q < kWalk; ++q) {
                    zn[q] = z[k0 + q + 1];
                    ck[q] = c[k0 + q];
                    pk[q] = piv[k0 + q];
                }
#pragma unroll
                for (int q = 0; q < kWalk; ++q) {
                    const double keep = pk[q] ? zn[q] : zk, go = pk[q] ? zk : zn[q];
                    zn[q] = keep;
                    zk = fma(-ck[q], keep, go);
                }
                if (lane == 0) {
#pragma unroll
                    for (int q = 0; q < kWalk; ++q) y[k0 + q] = zn[q];
                }
            }
            __syncthreads();
            // back substitution with U, y -> z
            double z1 = 0.0, z2 = 0.0;
            for (int k0 = (n + kWalk - 1) / kWalk * kWalk - kWalk; k0 >= 0; k0 -= kWalk) {
                double yk[kWalk], bq[kWalk], dq[kWalk], rq[kWalk];
#pragma unroll
                for (int q = 0; q < kWalk; ++q) {
                    yk[q] = y[k0 + q];
                    bq[q] = b[k0 + q];
                    dq[q] = dd[k0 + q];
                    rq[q] = ra[k0 + q];
                }
#pragma unroll
                for (int q = kWalk - 1; q >= 0; --q) {
                    const double v = k0 + q < n ? fma(-bq[q], z1, fma(-dq[q], z2, yk[q])) * rq[q] : 0.0;
                    z2 = z1;
                    z1 = v;
                    yk[q] = v;
                }
                if (lane == 0) {
#pragma unroll
                    for (int q = 0; q < kWalk; ++q) z[k0 + q] = yk[q];
                }
            }
            __syncthreads();
            // orthogonalise against the cluster's earlier members, normalise
            for (int q = i0; q < i; ++q) {
                const double* zq = Zt + (size_t)q * n;
                double s = 0.0;
                for (int k = lane; k < n; k += 64) s += zq[k] * z[k];
                s = wave_sum_dpp(s);
                for (int k = lane; k < n; k += 64) z[k] -= s * zq[k];
                __syncthreads();
            }
            // normalise: scale by the largest component first (a solve
            // against a nearly singular system can exceed sqrt(DBL_MAX))
            double amax = 0.0;
            for (int k = lane; k < n; k += 64) amax = fmax(amax, fabs(z[k]));
            amax = wave_max(amax);
            const double sc = amax > 0.0 ? 1.0 / amax : 1.0;
            double nrm = 0.0;
            for (int k = lane; k < n; k += 64) {
                const double zk = z[k] * sc;
                nrm += zk * zk;
            }
            nrm = wave_sum_dpp(nrm);
            const double inv = nrm > 0.0 ? sc / sqrt(nrm) : 1.0;
            __syncthreads();
            for (int k = lane; k < n; k += 64) z[k] *= inv;
            __syncthreads();
        }
        // a sign convention: the largest component positive
        double big = 0.0;
        int arg = 0;
        for (int k = lane; k < n; k += 64)
            if (fabs(z[k]) > big) { big = fabs(z[k]); arg = k; }
        for (int o = 32; o > 0; o >>= 1) {
            const double ob = __shfl_xor(big, o, 64);
            const int oa = __shfl_xor(arg, o, 64);
            if (ob > big || (ob == big && oa < arg)) { big = ob; arg = oa; }
        }
        const double sg = z[arg] < 0.0 ? -1.0 : 1.0;
        for (int k = lane; k < n; k += 64) Zt[(size_t)i * n + k] = sg * z[k];
        __syncthreads();
    }
}

using dbl4 = double __attribute__((ext_vector_type(4)));

// Block reflectors (LAPACK larft, forward, columnwise): Vb (I - Vb Tb Vb^T =
// H_j0 ... H_{j0+NB-1}, Vb = VhT[j0:j0+NB]^T) as VT = Vb Tb, row q of the block
// in VT[j0 + q].  One workgroup per block.  The Gram G = Vb^T Vb and Vb Tb are
// on the matrix cores; row p of Tb depends on itself and G only, so lane p
// holds it in registers and the recursion needs no barrier.  n = 64: 41 ->
// 9 us, n = 576: 87 -> 22 us.
constexpr int kLarftWaves = 8;

__global__ __launch_bounds__(64 * kLarftWaves) void larft_kernel(int n, int nref,
                                                                 const double* __restrict__ VhT,
                                                                 const double* __restrict__ tau,
                                                                 double* __restrict__ VT) {
    constexpr int NB = kSyevNB, LD = NB + 1;
    __shared__ double G[kLarftWaves][NB * LD];  // partial Grams, their sum in G[0]; Tb in G[1]
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane & 15, kq = lane >> 4;
    const int j0 = blockIdx.x * NB;
    const double* V0 = VhT + (size_t)(j0 + m) * n;
    const double* V1 = V0 + (size_t)16 * n;
    const bool ok0 = j0 + m < nref, ok1 = j0 + 16 + m < nref;
    dbl4 g00 = dbl4{0, 0, 0, 0}, g01 = g00, g11 = g00;
    for (int r0 = j0 + 16 * wv; r0 < n; r0 += 16 * kLarftWaves) {
        double a0[4], a1[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int r = r0 + 4 * kq + s;
            a0[s] = ok0 && r < n ? V0[r] : 0.0;
            a1[s] = ok1 && r < n ? V1[r] : 0.0;
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            g00 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0[s], a0[s], g00, 0, 0, 0);
            g01 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0[s], a1[s], g01, 0, 0, 0);
            g11 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1[s], a1[s], g11, 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {  // element r of a lane: row lane/16 + 4 r, column lane%16
        const int row = kq + 4 * r;
        G[wv][row * LD + m] = g00[r];
        G[wv][row * LD + 16 + m] = g01[r];
        G[wv][(16 + row) * LD + 16 + m] = g11[r];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < NB * NB; i += 64 * kLarftWaves) {
        const int at = (i / NB) * LD + i % NB;
        if (i % NB > i / NB) {
            double v = 0.0;
#pragma unroll
            for (int q = 0; q < kLarftWaves; ++q) v += G[q][at];
            G[0][at] = v;
        }
    }
    __syncthreads();
    if (wv == 0) {
        const int p = lane & (NB - 1);
        const double tp = j0 + p < nref ? tau[j0 + p] : 0.0;
        double T[NB];
        int col = 0;
#pragma unroll
        for (int q = 0; q < NB; ++q) {  // T[p][q] = -tau_q sum_{l<q} T[p][l] G[l][q]
            double s0 = 0.0, s1 = 0.0;
#pragma unroll
            for (int l = 0; l + 1 < q; l += 2) {
                s0 = fma(T[l], G[0][l * LD + col], s0);
                s1 = fma(T[l + 1], G[0][(l + 1) * LD + col], s1);
            }
            if (q & 1) s0 = fma(T[q - 1], G[0][(q - 1) * LD + col], s0);
            const double tq = bcast(tp, q);
            T[q] = q == p ? tq : q > p ? -tq * (s0 + s1) : 0.0;
            // the next column's address waits for this one: all 496 reads
            // hoisted would spill
            ++col;
            asm volatile("" : "+v"(col), "+v"(T[q]));
        }
        // one wave, LDS in order: no lane still reads G here
        if (lane < NB) {
#pragma unroll
            for (int q = 0; q < NB; ++q) G[1][p * LD + q] = T[q];
        }
    }
    __syncthreads();
    // VT^T = Tb^T Vb^T
    double at[2][8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        at[0][s] = G[1][(4 * s + kq) * LD + m];
        at[1][s] = G[1][(4 * s + kq) * LD + 16 + m];
    }
    for (int r0 = j0 + 16 * wv; r0 < n; r0 += 16 * kLarftWaves) {
        const int r = r0 + m;
        double b[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const int p = j0 + 4 * s + kq;
            b[s] = p < nref && r < n ? VhT[(size_t)p * n + r] : 0.0;
        }
        dbl4 acc0 = dbl4{0, 0, 0, 0}, acc1 = acc0;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(at[0][s], b[s], acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(at[1][s], b[s], acc1, 0, 0, 0);
        }
        if (r < n) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int q = j0 + kq + 4 * e;
                if (q < nref) VT[(size_t)q * n + r] = acc0[e];
                if (q + 16 < nref) VT[(size_t)(q + 16) * n + r] = acc1[e];
            }
        }
    }
}

// V = H_0 H_1 ... H_{n-2} Z, Z = Zt^T (Zt row i = eigenvector i of T).
// Columns are independent under a left product, so workgroup c0 takes NC
// columns of Z into LDS and applies the reflector blocks last to first:
// Y = Vb^T Z (the rows split over four groups of two waves, a 16-row half of Y
// each), then Z -= (Vb Tb) Y by 16-row tiles, both on the matrix cores with
// the reflectors read from L2.  Two barriers a block.  NC = 16 fills a matrix
// instruction; 8 where 16 columns of Z pass LDS.  n = 64: 26 -> 7 us,
// n = 576: 700 -> 147 us, n = 1000: 2070 -> 360 us.
constexpr int kApplyWaves = 8;

template <int NC>
__global__ __launch_bounds__(64 * kApplyWaves) void apply_q_kernel(int n, int nref,
                                                                   const double* __restrict__ VhT,
                                                                   const double* __restrict__ VT,
                                                                   const double* __restrict__ Zt,
                                                                   double* __restrict__ V, int ldv) {
    constexpr int NB = kSyevNB, KS = kApplyWaves / 2;
    extern __shared__ double sm[];
    const int n16 = (n + 15) & ~15;
    double* Z = sm;                          // n16 x NC, zero past n
    double* Y = Z + (size_t)n16 * NC;        // KS partial Y, NB x NC each
    const int t = threadIdx.x, lane = t & 63;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int m = lane & 15, kq = lane >> 4;
    const bool cok = m < NC;
    const int c0 = blockIdx.x * NC;
    for (int e = t; e < n16 * NC; e += 64 * kApplyWaves) {
        const int c = e / n16, r = e - c * n16;  // coalesced over r
        Z[r * NC + c] = c0 + c < n && r < n ? Zt[(size_t)(c0 + c) * n + r] : 0.0;
    }
    const int nblk = (nref + NB - 1) / NB;
    for (int b = nblk - 1; b >= 0; --b) {
        const int j0 = b * NB;
        __syncthreads();
        {
            const int p = j0 + 16 * (wv & 1) + m, g = wv >> 1;
            const double* Vp = VhT + (size_t)p * n;
            dbl4 acc = dbl4{0, 0, 0, 0};
            for (int r0 = j0 + 16 * g; r0 < n; r0 += 16 * KS) {
                double a[4], z[4];
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const int r = r0 + 4 * kq + s;
                    a[s] = p < nref && r < n ? Vp[r] : 0.0;
                    z[s] = cok ? Z[r * NC + m] : 0.0;
                }
#pragma unroll
                for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], z[s], acc, 0, 0, 0);
            }
            if (cok) {
#pragma unroll
                for (int r = 0; r < 4; ++r) Y[(g * NB + 16 * (wv & 1) + kq + 4 * r) * NC + m] = acc[r];
            }
        }
        __syncthreads();
        double y[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            double v = 0.0;
#pragma unroll
            for (int g = 0; g < KS; ++g) v += cok ? Y[(g * NB + 4 * s + kq) * NC + m] : 0.0;
            y[s] = -v;
        }
        for (int r0 = j0 + 16 * wv; r0 < n; r0 += 16 * kApplyWaves) {
            const int r = r0 + m;
            double a[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int p = j0 + 4 * s + kq;
                a[s] = p < nref && r < n ? VT[(size_t)p * n + r] : 0.0;
            }
            dbl4 acc;
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = cok ? Z[(r0 + kq + 4 * e) * NC + m] : 0.0;
#pragma unroll
            for (int s = 0; s < 8; ++s) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], y[s], acc, 0, 0, 0);
            if (cok) {
#pragma unroll
                for (int e = 0; e < 4; ++e) Z[(r0 + kq + 4 * e) * NC + m] = acc[e];
            }
        }
    }
    __syncthreads();
    for (int e = t; e < n * NC; e += 64 * kApplyWaves) {
        const int r = e / NC, c = e - r * NC;
        if (c0 + c < n) V[(size_t)r * ldv + c0 + c] = Z[e];
    }
}

struct SyevWs {
    size_t d, e, tau, bounds, W, Vh, vb, pb, sb, Zt, total;
    int ldw;
};

static SyevWs syev_layout(int n) {
    SyevWs L{};
    size_t off = 0;
    auto take = [&](size_t doubles) {
        const size_t o = off;
        off += align_up(doubles * sizeof(double), 256);
        return o;
    };
    L.d = take(n);
    L.e = take(n);
    L.tau = take(n);
    L.bounds = take(4);
    L.ldw = n + (n & 1);
    L.W = take((size_t)n * L.ldw + 2);  // + the pair a 16-byte load may touch past the last row
    L.Vh = take((size_t)n * n);
    L.vb = take(2 * (size_t)n);
    L.pb = take(2 * (size_t)n);
    L.sb = take(2 * (size_t)kStepGroupsMax);
    L.Zt = take((size_t)n * n);
    L.total = off;
    return L;
}

}  // namespace rvgp

using namespace rvgp;

extern "C" size_t rvgp_syev_ws_bytes(int n) {
    if (n < 1 || n > kSyevMaxN) return 0;
    return syev_layout(n).total;
}

extern "C" int rvgp_syev(int n, double* A, int lda, double* w, double* V, int ldv, void* ws,
                         size_t ws_bytes, void* stream) {
    RVGP_CHECK_ARG(n >= 1 && n <= kSyevMaxN, "rvgp_syev: need 1 <= n <= %d", kSyevMaxN);
    RVGP_CHECK_ARG(lda >= n && ldv >= n, "rvgp_syev: leading dimension < n");
    const SyevWs L = syev_layout(n);
    RVGP_CHECK_ARG(ws != nullptr && ws_bytes >= L.total, "rvgp_syev: needs %zu bytes of workspace",
                   L.total);
    hipStream_t s = as_stream(stream);
    char* base = static_cast<char*>(ws);
    double* d = reinterpret_cast<double*>(base + L.d);
    double* e = reinterpret_cast<double*>(base + L.e);
    double* tau = reinterpret_cast<double*>(base + L.tau);
    double* bounds = reinterpret_cast<double*>(base + L.bounds);
    double* W = reinterpret_cast<double*>(base + L.W);
    double* VhT = reinterpret_cast<double*>(base + L.Vh);
    double* Vp = reinterpret_cast<double*>(base + L.vb);
    double* Wp = reinterpret_cast<double*>(base + L.pb);
    double* sb = reinterpret_cast<double*>(base + L.sb);
    double* Zt = reinterpret_cast<double*>(base + L.Zt);
    const int ldw = L.ldw;

    // stage 1: tridiagonalisation, one launch per column (reflectors
    // j = 0 .. n-2; the last has length 1 and tau = 0)
    const size_t nn = (size_t)n * n;
    if (n > kSmallN) {
        hipLaunchKernelGGL(copy_full_kernel, dim3(cdiv(nn, 256)), dim3(256), 0, s, n, A, lda, W, ldw);
        RVGP_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(fill_kernel, dim3(cdiv(nn, 256)), dim3(256), 0, s, nn, VhT, 0.0);
    RVGP_LAUNCH_CHECK();
    const size_t stsm = sizeof(double) * (4 * (size_t)n + 2 * (kStepThreads / 64));
    if (n <= kSmallN) {
        const int rows = cdiv(n, 64);
        const auto kern = rows == 1   ? sytrd_small_kernel<1, 4>
                          : rows == 2 ? sytrd_small_kernel<2, 4>
                                      : sytrd_small_kernel<3, 8>;
        hipLaunchKernelGGL(kern, dim3(1), dim3(rows < 3 ? 256 : 512), 0, s, n, A, lda, VhT, d, e, tau);
        RVGP_LAUNCH_CHECK();
    } else if (n <= 1024) {
        // 128 workgroups x 4 wavefronts x 2 rows cover the <= 1023 trailing rows
        const int G = n < kStepGroupsMax ? n : kStepGroupsMax;
        auto kern = sytrd_step_prefetch_kernel<2, 16>;
        RVGP_CHECK_HIP(hipFuncSetAttribute((const void*)kern,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)stsm));
        for (int j = 0; j + 1 < n; ++j) {
            hipLaunchKernelGGL(kern, dim3(G), dim3(kStepThreads), stsm, s, n, W, ldw, j, Vp, Wp,
                               sb, VhT, d, e, tau);
            RVGP_LAUNCH_CHECK();
        }
    } else {
        const int G = kStepGroups;
        RVGP_CHECK_HIP(hipFuncSetAttribute((const void*)sytrd_step_kernel,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)stsm));
        for (int j = 0; j + 1 < n; ++j) {
            hipLaunchKernelGGL(sytrd_step_kernel, dim3(G), dim3(kStepThreads), stsm, s, n, W, ldw,
                               j, Vp, Wp, sb, VhT, d, e, tau);
            RVGP_LAUNCH_CHECK();
        }
    }
    const int nref = n - 1;
    // stage 2: eigenvalues and eigenvectors of T
    hipLaunchKernelGGL(tri_bounds_kernel, dim3(1), dim3(256), 0, s, n, d, e, bounds);
    RVGP_LAUNCH_CHECK();
    hipLaunchKernelGGL(stebz_kernel, dim3(n), dim3(64), sizeof(double) * 2 * n, s, n, d, e, bounds,
                       w);
    RVGP_LAUNCH_CHECK();
    const size_t np = (n + kWalk - 1) / kWalk * kWalk + kWalk;
    const size_t ssm = (sizeof(double) * 6 + sizeof(int)) * np;
    RVGP_CHECK_HIP(hipFuncSetAttribute((const void*)stein_kernel,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)ssm));
    hipLaunchKernelGGL(stein_kernel, dim3(n), dim3(64), ssm, s, n, d, e, w, bounds, Zt);
    RVGP_LAUNCH_CHECK();
    // stage 3: V = H_0 H_1 ... H_{n-2} Z with Z = Zt^T (one fused kernel,
    // a few columns of Z per workgroup)
    const int nblk = (nref + kSyevNB - 1) / kSyevNB;
    if (nblk > 0) {  // W is free by now: it takes Vb Tb
        hipLaunchKernelGGL(larft_kernel, dim3(nblk), dim3(64 * kLarftWaves), 0, s, n, nref, VhT, tau, W);
        RVGP_LAUNCH_CHECK();
    }
    const int nc = n <= 1024 ? 16 : 8;
    const size_t qsm = sizeof(double) * nc * ((size_t)((n + 15) & ~15) + (kApplyWaves / 2) * kSyevNB);
    const auto apply = nc == 16 ? apply_q_kernel<16> : apply_q_kernel<8>;
    RVGP_CHECK_HIP(hipFuncSetAttribute((const void*)apply, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)qsm));
    hipLaunchKernelGGL(apply, dim3(cdiv(n, nc)), dim3(64 * kApplyWaves), qsm, s, n, nref, VhT, W, Zt, V,
                       ldv);
    RVGP_LAUNCH_CHECK();
    return RVGP_OK;
}
