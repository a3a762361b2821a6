// a11  The heat kernel's Chebyshev series on a block-CSR operator in FP64
// (replaces the dense scipy expm of RVGP/smoothing.py:13-15):
//     out = sum_j C_j o T_j,   T_1 = (a A + b) T_0 / 2,
//     T_j = (a A + b) T_{j-1} - T_{j-2},
// one coefficient per column and term (C_j, a row of columns).  One launch a
// term: the product, the recurrence and the sum share it, so a term reads the
// operator, gathers T_{j-1}, and reads and writes T_{j-2} and out once.  Terms
// of columns whose series has ended are not formed: columns come ordered by
// the length of their series, and a term runs on the leading ones.
//
// Mapping: V lanes hold a row's columns (16-byte pairs; past 64 columns in groups
// of 64), E lanes split its stored blocks, so that a wave works on 64 / (V E) block rows whatever the
// width -- one wave per row left 56 of 64 lanes idle at 16 columns.  n = 50,000,
// b = 3, 16 columns: 122 + 8 (sum) -> 83 us a term, 57 us where the rows are numbered along a
// space-filling curve; b = 1, 32 columns: 46 + 8 -> 42 and 25 us.
// Bound by the gathers through L1 and L2.
// All groups of columns share a term's launch: 100 fields on 600 nodes of a 3-torus
// 12.8 ms a smoothing (t = 60) in blocks of 64 columns, 9.3 ms by SpMMs, 6.8 ms so.
// Small operators are bound by the launches: the two series of a vector
// diffusion (connection and scalar Laplacian) then share theirs.
#include "common.h"

#pragma clang fp contract(fast)

namespace rvgp {
namespace {

typedef double dbl2 __attribute__((ext_vector_type(2)));

struct Series {
    int nb;
    const int* rowptr;
    const int* cols;
    const double* vals;
    const double* cur;   // T_{j-1}
    double* prev;        // T_{j-2}, overwritten by T_j
    double* out;
    const double* c0;    // term 1: C_0 (out is set); else NULL (out is added to)
    const double* cj;
    int ld, act;         // row stride, columns of this term (both even)
    double a, b;
};

constexpr int kThreads = 256;
constexpr int kColumns = 64;  // of a workgroup; more of them are gridDim.y

template <int B, int V, int E>
__device__ __forceinline__ void term_rows(const Series& s, int wg, int wgs) {
    constexpr int G = V * E, ROWS = kThreads / G;
    // each XCD gets one contiguous range of block rows (wgs is a multiple of 8)
    const int per = wgs >> 3;
    const int lw = (wg & 7) * per + (wg >> 3);
    const int row = lw * ROWS + (int)threadIdx.x / G;
    const int l = threadIdx.x % G;
    const int v = l % V, ed = l / V, c = 2 * v + kColumns * blockIdx.y;
    const bool on = row < s.nb && c < s.act;
    dbl2 y[B];
#pragma unroll
    for (int p = 0; p < B; ++p) y[p] = dbl2(0.0);
    if (on) {
        const int e1 = s.rowptr[row + 1];
        const double* X = s.cur + c;
#pragma unroll 4
        for (int e = s.rowptr[row] + ed; e < e1; e += E) {
            const size_t j = (size_t)s.cols[e] * B;
            const double* blk = s.vals + (size_t)e * (B * B);
            dbl2 x[B];
#pragma unroll
            for (int q = 0; q < B; ++q) x[q] = *reinterpret_cast<const dbl2*>(X + (j + q) * s.ld);
#pragma unroll
            for (int p = 0; p < B; ++p)
#pragma unroll
                for (int q = 0; q < B; ++q) y[p] += blk[p * B + q] * x[q];
        }
    }
#pragma unroll
    for (int o = V; o < G; o <<= 1)
#pragma unroll
        for (int p = 0; p < B; ++p) {
            y[p].x += __shfl_xor(y[p].x, o, 64);
            y[p].y += __shfl_xor(y[p].y, o, 64);
        }
    if (!on) return;
    const dbl2 cj = *reinterpret_cast<const dbl2*>(s.cj + c);
#pragma unroll
    for (int p = 0; p < B; ++p) {
        if (p % E != ed) continue;
        const size_t at = ((size_t)row * B + p) * s.ld + c;
        const dbl2 x = *reinterpret_cast<const dbl2*>(s.cur + at);
        dbl2* po = reinterpret_cast<dbl2*>(s.out + at);
        dbl2 t = s.a * y[p] + s.b * x;
        if (s.c0 != nullptr) {
            t *= 0.5;
            *po = *reinterpret_cast<const dbl2*>(s.c0 + c) * x + cj * t;
        } else {
            t -= *reinterpret_cast<const dbl2*>(s.prev + at);
            *po += cj * t;
        }
        *reinterpret_cast<dbl2*>(s.prev + at) = t;
    }
}

template <int B, int V, int E>
__global__ __launch_bounds__(kThreads) void term_kernel(Series s) {
    term_rows<B, V, E>(s, blockIdx.x, gridDim.x);
}

// both series of a diffusion of one field: workgroups [0, g0) and the rest
template <int B>
__global__ __launch_bounds__(kThreads) void term_pair_kernel(Series s, Series t, int g0) {
    if ((int)blockIdx.x < g0) term_rows<B, 1, 8>(s, blockIdx.x, g0);
    else term_rows<1, 1, 8>(t, blockIdx.x - g0, gridDim.x - g0);
}

template <int V, int E>
constexpr int rows_per_wg() { return kThreads / (V * E); }

template <int V, int E>
int grid_of(int nb) { return 8 * (int)cdiv(cdiv(nb, rows_per_wg<V, E>()), 8); }

template <int V, int E>
void launch_term(const Series& s, int b, hipStream_t st) {
    const dim3 g(grid_of<V, E>(s.nb), cdiv(s.act, kColumns)), t(kThreads);
    if (b == 1) hipLaunchKernelGGL((term_kernel<1, V, E>), g, t, 0, st, s);
    else if (b == 2) hipLaunchKernelGGL((term_kernel<2, V, E>), g, t, 0, st, s);
    else hipLaunchKernelGGL((term_kernel<3, V, E>), g, t, 0, st, s);
}

}  // namespace
}  // namespace rvgp

using namespace rvgp;

extern "C" int rvgp_cheb_series(int nops, const rvgp_series* ops, void* stream) {
    RVGP_CHECK_ARG(nops >= 1 && nops <= 2 && ops != nullptr, "rvgp_cheb_series: one or two series");
    int J = 0;
    for (int o = 0; o < nops; ++o) {
        const rvgp_series& p = ops[o];
        RVGP_CHECK_ARG(p.nb >= 1 && p.b >= 1 && p.b <= 3, "rvgp_cheb_series: block size must be 1, 2 or 3");
        RVGP_CHECK_ARG(p.terms >= 2 && p.active != nullptr, "rvgp_cheb_series: need at least two terms");
        RVGP_CHECK_ARG(p.ld >= 2 && p.ld % 2 == 0 && p.ld <= 65535 * kColumns,
                       "rvgp_cheb_series: the row stride must be even and at most %d", 65535 * kColumns);
        RVGP_CHECK_ARG((((uintptr_t)p.t0 | (uintptr_t)p.t1 | (uintptr_t)p.out | (uintptr_t)p.coef) % 16) == 0 &&
                           p.t0 != p.t1 && p.t0 != p.out && p.t1 != p.out,
                       "rvgp_cheb_series: buffers must be distinct and 16-byte aligned");
        for (int j = 1; j < p.terms; ++j)
            RVGP_CHECK_ARG(p.active[j] >= 1 && p.active[j] <= p.ld && (j == 1 || p.active[j] <= p.active[j - 1]),
                           "rvgp_cheb_series: active columns must not grow from term to term");
        J = p.terms > J ? p.terms : J;
    }
    hipStream_t st = as_stream(stream);
    for (int j = 1; j < J; ++j) {
        Series s[2];
        bool run[2] = {false, false};
        for (int o = 0; o < nops; ++o) {
            const rvgp_series& p = ops[o];
            if (j >= p.terms) continue;
            run[o] = true;
            double* even = static_cast<double*>(p.t0);
            double* odd = static_cast<double*>(p.t1);
            s[o].nb = p.nb;
            s[o].rowptr = p.rowptr;
            s[o].cols = p.cols;
            s[o].vals = p.vals;
            s[o].cur = j % 2 == 1 ? even : odd;
            s[o].prev = j % 2 == 1 ? odd : even;
            s[o].out = p.out;
            s[o].c0 = j == 1 ? p.coef : nullptr;
            s[o].cj = p.coef + (size_t)j * p.ld;
            s[o].ld = p.ld;
            // the first term sets every column of out
            s[o].act = j == 1 ? p.ld : (p.active[j] + 1) / 2 * 2;
            s[o].a = p.a;
            s[o].b = p.shift;
        }
        if (run[0] && run[1] && s[0].act <= 2 && s[1].act <= 2 && ops[1].b == 1) {
            const int g0 = grid_of<1, 8>(s[0].nb), g1 = grid_of<1, 8>(s[1].nb);
            const dim3 g(g0 + g1), t(kThreads);
            if (ops[0].b == 1) hipLaunchKernelGGL((term_pair_kernel<1>), g, t, 0, st, s[0], s[1], g0);
            else if (ops[0].b == 2) hipLaunchKernelGGL((term_pair_kernel<2>), g, t, 0, st, s[0], s[1], g0);
            else hipLaunchKernelGGL((term_pair_kernel<3>), g, t, 0, st, s[0], s[1], g0);
            RVGP_LAUNCH_CHECK();
            continue;
        }
        for (int o = 0; o < nops; ++o) {
            if (!run[o]) continue;
            const int nv = s[o].act / 2, b = ops[o].b;
            if (nv <= 1) launch_term<1, 8>(s[o], b, st);
            else if (nv <= 2) launch_term<2, 4>(s[o], b, st);
            else if (nv <= 4) launch_term<4, 4>(s[o], b, st);
            else if (nv <= 8) launch_term<8, 2>(s[o], b, st);
            else if (nv <= 16) launch_term<16, 1>(s[o], b, st);
            else launch_term<32, 1>(s[o], b, st);
            RVGP_LAUNCH_CHECK();
        }
    }
    return RVGP_OK;
}
