// Per-node frame algebra of the vector-field path:
//   * express_in_local_frame / project_to_manifold (RVGP/geometry.py:165-175,
//     used by dataclass.py:100, 110, 116): c_i = T_i^T v_i, v_i = T_i c_i,
//     v_i <- T_i T_i^T v_i, for F fields at once;
//   * the magnitude renormalisation of vector_diffusion
//     (RVGP/smoothing.py:57-62): out_i <- out_i * a_i / (b_i * |out_i|);
//   * ambient eigenvector rows Phi_i = T_i U_i (dataclass.py:57-59) for a
//     list of nodes, written straight into the GP design matrix.
#include "common.h"

namespace rvgp {

// mode 0: c = T^T v  (in: (F, n, D) -> out: (F, n, d))
// mode 1: v = T c    (in: (F, n, d) -> out: (F, n, D))
// mode 2: v = T T^T v (in/out: (F, n, D))
// G lanes per node, lane p its ambient coordinates p, p + G, ...: vectors and
// frames are read and written in the order they are stored, and for D <= G a
// node's frame stays in registers for all of its workgroup's fields (blockIdx.y,
// blockIdx.y + gridDim.y, ...); the sums over D meet by shuffles.  (A thread per node and field read both 256 bytes apart: n =
// 50,000, F = 16, D = 32, d = 3, 2.1 ms -> 0.17 (mode 0) and 0.10 ms (mode 1), bound by HBM.)
// workgroups that fill the GPU: 2000 fields of 5000 nodes in R^3 take 249, 240 and
// 223 us with 2048, 4096 and 16384, of 512 nodes 23, 23 and 29 us
constexpr int kFrameGroups = 4096;

template <int G>
__global__ __launch_bounds__(256) void frame_kernel(int mode, int F, int n, int D, int d, int ldt,
                                                    const double* __restrict__ T,
                                                    const double* in, double* out) {
    constexpr int DM = 8;  // d <= 8
    const int i = (int)(((size_t)blockIdx.x * 256 + threadIdx.x) / G);
    const int l = threadIdx.x % G;
    const bool live = i < n;
    const double* Ti = T + (size_t)(live ? i : 0) * D * ldt;
    double t[DM];
    const bool once = D <= G;
    auto frame_row = [&](int p) {
#pragma unroll
        for (int q = 0; q < DM; ++q) t[q] = live && q < d && p < D ? Ti[(size_t)p * ldt + q] : 0.0;
    };
    if (once) frame_row(l);
    for (int f = blockIdx.y; f < F; f += gridDim.y) {
        const size_t g = (size_t)f * n + (live ? i : 0);
        double c[DM];
        if (mode == 1) {
#pragma unroll
            for (int q = 0; q < DM; ++q) c[q] = q < d ? in[g * d + q] : 0.0;
        } else {
#pragma unroll
            for (int q = 0; q < DM; ++q) c[q] = 0.0;
            for (int p = l; p < D; p += G) {
                if (!once) frame_row(p);
                const double v = live ? in[g * D + p] : 0.0;
#pragma unroll
                for (int q = 0; q < DM; ++q) c[q] += t[q] * v;
            }
#pragma unroll
            for (int q = 0; q < DM; ++q) {
                if (q >= d) break;
#pragma unroll
                for (int o = G / 2; o > 0; o >>= 1) c[q] += __shfl_xor(c[q], o, 64);
            }
        }
        if (!live) continue;
        if (mode == 0) {
#pragma unroll
            for (int q = 0; q < DM; ++q)
                if (q < d && q % G == l) out[g * d + q] = c[q];
            continue;
        }
        for (int p = l; p < D; p += G) {
            if (!once) frame_row(p);
            double v = 0.0;
#pragma unroll
            for (int q = 0; q < DM; ++q) v += t[q] * c[q];
            out[g * D + p] = v;
        }
    }
}

// out (F*n, d) scaled in place; a, b: (F*n,) magnitudes from the two scalar
// diffusions exp(-tL)|x| and exp(-tL)1.
__global__ void diffusion_normalise_kernel(size_t rows, int d, double* __restrict__ out,
                                           int ldo, const double* __restrict__ a, int lda,
                                           const double* __restrict__ b, int ldb) {
    const size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= rows) return;
    double* o = out + g * ldo;
    double s = 0.0;
    for (int q = 0; q < d; ++q) s += o[q] * o[q];
    const double scale = a[g * lda] / (b[g * ldb] * sqrt(s));
    for (int q = 0; q < d; ++q) o[q] = o[q] * scale;
}

// Phi rows: out[(r*D + p), j] = sum_q T[node_r][p][q] * U[node_r*d + q][j]
template <typename TO>
__global__ void phi_rows_kernel(int m, int n, int D, int d, int ldt, int k,
                                const double* __restrict__ T, const double* __restrict__ U,
                                int ldu, const int* __restrict__ nodes, TO* __restrict__ out,
                                int ldo) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= k) return;
    for (int r = blockIdx.y; r < m; r += gridDim.y) {
        const int i = nodes[r];
        if ((unsigned)i >= (unsigned)n) {
            // a node outside [0, n): the row reads nothing and is NaN
            for (int p = 0; p < D; ++p) out[(size_t)(r * D + p) * ldo + j] = (TO)__builtin_nan("");
            continue;
        }
        const double* Ti = T + (size_t)i * D * ldt;
        double u[8];
        for (int q = 0; q < d; ++q) u[q] = U[(size_t)(i * d + q) * ldu + j];
        for (int p = 0; p < D; ++p) {
            double s = 0.0;
            for (int q = 0; q < d; ++q) s += Ti[p * ldt + q] * u[q];
            out[(size_t)(r * D + p) * ldo + j] = (TO)s;
        }
    }
}

}  // namespace rvgp

using namespace rvgp;

extern "C" int rvgp_frame_apply(int mode, int F, int n, int D, int d, const double* T, int ldt,
                                const double* in, double* out, void* stream) {
    RVGP_CHECK_ARG(mode >= 0 && mode <= 2, "rvgp_frame_apply: mode must be 0, 1 or 2");
    RVGP_CHECK_ARG(d >= 1 && d <= 8 && d <= D && ldt >= d, "rvgp_frame_apply: need 1 <= d <= min(D, 8)");
    const size_t rows = (size_t)F * n;
    if (rows == 0) return RVGP_OK;
    const int G = D <= 4 ? 4 : D <= 8 ? 8 : D <= 16 ? 16 : D <= 32 ? 32 : 64;
    // few nodes: the fields are split until the GPU is full (2000 fields, one
    // workgroup for all of them: 64 nodes in R^3 1690 us, 8 us split)
    const unsigned nodes = cdiv((size_t)n * G, 256), fill = cdiv(kFrameGroups, nodes);
    const dim3 grid(nodes, (unsigned)F < fill ? (unsigned)F : fill), block(256);
    hipStream_t s = as_stream(stream);
#define RVGP_FRAME(GG) \
    hipLaunchKernelGGL((frame_kernel<GG>), grid, block, 0, s, mode, F, n, D, d, ldt, T, in, out)
    if (G == 4) RVGP_FRAME(4);
    else if (G == 8) RVGP_FRAME(8);
    else if (G == 16) RVGP_FRAME(16);
    else if (G == 32) RVGP_FRAME(32);
    else RVGP_FRAME(64);
#undef RVGP_FRAME
    RVGP_LAUNCH_CHECK();
    return RVGP_OK;
}

extern "C" int rvgp_diffusion_normalise(size_t rows, int d, double* out, int ldo, const double* a,
                                        int lda, const double* b, int ldb, void* stream) {
    RVGP_CHECK_ARG(d >= 1 && ldo >= d, "rvgp_diffusion_normalise: bad d/ldo");
    if (rows == 0) return RVGP_OK;
    hipLaunchKernelGGL(diffusion_normalise_kernel, dim3(cdiv(rows, 256)), dim3(256), 0,
                       as_stream(stream), rows, d, out, ldo, a, lda, b, ldb);
    RVGP_LAUNCH_CHECK();
    return RVGP_OK;
}

extern "C" int rvgp_phi_rows(int out_f32, int m, int n, int D, int d, const double* T, int ldt,
                             int k, const double* U, int ldu, const int* nodes, void* out, int ldo,
                             void* stream) {
    RVGP_CHECK_ARG(d >= 1 && d <= 8 && ldt >= d && ldu >= k && ldo >= k && n >= 0,
                   "rvgp_phi_rows: bad sizes");
    if (m == 0 || k == 0) return RVGP_OK;
    dim3 g(cdiv(k, 256), m < 65535 ? m : 65535);
    if (out_f32)
        hipLaunchKernelGGL(phi_rows_kernel<float>, g, dim3(256), 0, as_stream(stream), m, n, D, d, ldt, k,
                           T, U, ldu, nodes, static_cast<float*>(out), ldo);
    else
        hipLaunchKernelGGL(phi_rows_kernel<double>, g, dim3(256), 0, as_stream(stream), m, n, D, d, ldt,
                           k, T, U, ldu, nodes, static_cast<double*>(out), ldo);
    RVGP_LAUNCH_CHECK();
    return RVGP_OK;
}
