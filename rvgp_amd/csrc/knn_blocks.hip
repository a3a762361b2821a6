// a2  kNN over spatial blocks (RVGP/geometry.py:100-123): rvgp_knn's result
// from the few blocks of candidates that can hold a neighbour (blocks.h).
#include "blocks.h"

namespace rvgp {

// (d, j) before (e, i): the order of the result lists.
__device__ __forceinline__ bool nearer(double d, int j, double e, int i) {
    return d < e || (d == e && j < i);
}

// Insert (d, j) into the right-aligned ascending list (slots [KMAX-k, KMAX)
// live, -inf before them): larger entries shift back by one.
template <int KMAX>
__device__ __forceinline__ void list_insert(double (&bd)[KMAX], int (&bi)[KMAX], double d, int j) {
#pragma unroll
    for (int p = KMAX - 1; p > 0; --p) {
        const bool shift = nearer(d, j, bd[p - 1], bi[p - 1]);
        const bool here = !shift && nearer(d, j, bd[p], bi[p]);
        bi[p] = shift ? bi[p - 1] : (here ? j : bi[p]);
        bd[p] = shift ? bd[p - 1] : (here ? d : bd[p]);
    }
    if (nearer(d, j, bd[0], bi[0])) {
        bd[0] = d;
        bi[0] = j;
    }
}

// The k nearest other points of every point, blocks of 64 queries (one per
// lane) against the blocks whose box can hold a neighbour.  A workgroup of W
// waves shares one query block; wave w takes the candidate blocks
// = w (mod W), the ones next to the query block on the curve first, so that
// the k-th distances are small before the rest is looked at.  Then each lane
// tests one box against the queries' box, survivors are tested query by
// query, and what is left is scanned: candidates by wave-uniform scalar loads
// in groups of four, PROJ (D > 8) by the FP32 box coordinates before the
// FP64 distance.  The waves share their k-th distances (LDS, min) and wave 0
// merges the lists; candidates arrive in any order, so the lists are ordered
// by (distance, index) explicitly.
// Bound by the insertions into the register lists and the scalar loads'
// latency.  n = 100,000 against the scan of all points: D = 32, k = 20 21.7 ->
// 3.8 ms; D = 3, k = 10 10.9 -> 0.62 ms.
template <int DMAX, int KMAX, int W, bool PROJ>
__global__ __launch_bounds__(64 * W) void knn_blocks_kernel(
    const double* __restrict__ xs, const float* __restrict__ ys, const float* __restrict__ box,
    const int* __restrict__ orig, const double* __restrict__ unit, int n, int k, int NB,
    int* __restrict__ nbr) {
    __shared__ unsigned long long thr_sh[64];
    extern __shared__ char lists[];  // waves 1 .. W-1: k x 64 distances, then indices
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // consecutive workgroups go to the XCDs in turn: each XCD gets a run of
    // neighbouring query blocks, whose candidates share its L2
    const int per = (NB + 7) / 8;
    const int qb = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (qb >= NB || (int)(blockIdx.x >> 3) >= per) return;  // whole workgroups
    const int pos = qb * kBlock + lane;
    const int i = orig[pos];
    const double inv2 = unit[1];
    constexpr double INF = __builtin_huge_val();

    double q[DMAX];
#pragma unroll
    for (int c = 0; c < DMAX; ++c) q[c] = pos < n ? xs[(size_t)pos * DMAX + c] : 0.0;
    float yq[kBoxDims];
#pragma unroll
    for (int c = 0; c < kBoxDims; ++c) yq[c] = ys[(size_t)pos * kBoxRow + c];
    double bd[KMAX];
    int bi[KMAX];
#pragma unroll
    for (int p = 0; p < KMAX; ++p) {
        bd[p] = p < KMAX - k ? -INF : INF;
        bi[p] = 0x7fffffff;
    }
    if (threadIdx.x < 64) thr_sh[lane] = 0x7ff0000000000000ULL;
    __syncthreads();

    double thr = i >= 0 ? INF : -INF;  // a lane without a query takes nothing
    float lim = i >= 0 ? __builtin_huge_valf() : -1.0f;
    auto refresh = [&]() {  // the smallest k-th distance any wave has for this query
        if (i >= 0) {
            const double t = __longlong_as_double((long long)thr_sh[lane]);
            thr = bd[KMAX - 1] < t ? bd[KMAX - 1] : t;
            lim = inv2 > 0.0 ? box_limit(thr, inv2) : __builtin_huge_valf();
        }
    };
    auto offer = [&](int o, double acc) {
        // another wave's bound is inclusive: an equal distance can still win
        // by its index
        if (o != i && acc <= thr && nearer(acc, o, bd[KMAX - 1], bi[KMAX - 1]))
            list_insert<KMAX>(bd, bi, acc, o);
    };
    auto scan = [&](int cb) {
        refresh();
        const int c0 = cb * kBlock, c1 = min(n, c0 + kBlock);
        for (int c = c0; c < c1; c += 4) {  // rows past n are zeros, in bounds, never offered
            unsigned live = 0;
            double acc[4] = {0.0, 0.0, 0.0, 0.0};
            if (PROJ) {
                float yc[4][kBoxDims];
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int d = 0; d < kBoxDims; ++d) yc[g][d] = ys[(size_t)(c + g) * kBoxRow + d];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    float s = 0.0f;
#pragma unroll
                    for (int d = 0; d < kBoxDims; ++d) {
                        const float t = yq[d] - yc[g][d];
                        s = fmaf(t, t, s);
                    }
                    if (c + g < c1 && __any(s <= lim)) live |= 1u << g;
                }
            } else {
                double v[4][DMAX];
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int d = 0; d < DMAX; ++d) v[g][d] = xs[(size_t)(c + g) * DMAX + d];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
#pragma unroll
                    for (int d = 0; d < DMAX; ++d) {
                        const double t = __dsub_rn(q[d], v[g][d]);
                        acc[g] = __fma_rn(t, t, acc[g]);
                    }
                    if (c + g < c1 && __any(acc[g] <= thr)) live |= 1u << g;
                }
            }
            if (live == 0) continue;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (!(live & (1u << g))) continue;
                if (PROJ) {
#pragma unroll
                    for (int d = 0; d < DMAX; ++d) {
                        const double t = __dsub_rn(q[d], xs[(size_t)(c + g) * DMAX + d]);
                        acc[g] = __fma_rn(t, t, acc[g]);
                    }
                }
                offer(orig[c + g], acc[g]);
            }
            if (bd[KMAX - 1] < thr) {
                thr = bd[KMAX - 1];
                if (PROJ && inv2 > 0.0) lim = box_limit(thr, inv2);
            }
        }
        if (i >= 0 && bd[KMAX - 1] < INF)
            atomicMin(&thr_sh[lane], (unsigned long long)__double_as_longlong(bd[KMAX - 1]));
    };

    // the blocks around the query block on the curve: 2 W + 1 of them, each
    // wave its own
    const int n0 = max(0, qb - W), n1 = min(NB, qb + W + 1);
    for (int cb = n0 + ((w - n0) % W + W) % W; cb < n1; cb += W) scan(cb);
    __syncthreads();

    const float* qbox = box + (size_t)qb * kBoxStride;
    float ql[kBoxDims], qh[kBoxDims];
#pragma unroll
    for (int d = 0; d < kBoxDims; ++d) {
        ql[d] = qbox[d];
        qh[d] = qbox[kBoxRow + d];
    }
    const int mine = (NB - w + W - 1) / W;           // this wave's blocks: w, w + W, ...
    const int groups = (mine + 63) / 64;
    const int g0 = min(groups - 1, (qb / W) / 64);
    for (int gi = 0; gi < groups; ++gi) {
        const int g = g0 + gi < groups ? g0 + gi : g0 + gi - groups;
        refresh();
        float most = lim;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) most = fmaxf(most, __shfl_xor(most, o, 64));
        const int s = g * 64 + lane, cb = s * W + w;
        bool pass = s < mine && (cb < n0 || cb >= n1);
        if (pass) {
            const float* bx = box + (size_t)cb * kBoxStride;
            float lb = 0.0f;
#pragma unroll
            for (int d = 0; d < kBoxDims; ++d) {
                const float t = fmaxf(0.0f, fmaxf(bx[d] - qh[d], ql[d] - bx[kBoxRow + d]));
                lb = fmaf(t, t, lb);
            }
            pass = lb <= most;
        }
        for (unsigned long long m = __ballot(pass); m != 0; m &= m - 1) {
            const int cbu = (g * 64 + __builtin_ctzll(m)) * W + w;  // wave-uniform
            const float* bx = box + (size_t)cbu * kBoxStride;
            float lb = 0.0f;
#pragma unroll
            for (int d = 0; d < kBoxDims; ++d) {
                const float t = fmaxf(0.0f, fmaxf(bx[d] - yq[d], yq[d] - bx[kBoxRow + d]));
                lb = fmaf(t, t, lb);
            }
            if (__any(lb <= lim)) scan(cbu);
        }
    }

    if (W > 1) {
        double* ld = reinterpret_cast<double*>(lists);
        int* li = reinterpret_cast<int*>(ld + (size_t)(W - 1) * k * 64);
        if (w > 0) {
#pragma unroll
            for (int p = 0; p < KMAX; ++p) {
                if (p < KMAX - k) continue;
                const int e = ((w - 1) * k + p - (KMAX - k)) * 64 + lane;
                ld[e] = bd[p];
                li[e] = bi[p];
            }
        }
        __syncthreads();
        if (w > 0) return;
        for (int s = 0; s < W - 1; ++s)
            for (int p = 0; p < k; ++p) {
                const int e = (s * k + p) * 64 + lane;
                const bool take = i >= 0 && nearer(ld[e], li[e], bd[KMAX - 1], bi[KMAX - 1]);
                if (!__any(take)) break;  // the rest of this list is no nearer
                if (take) list_insert<KMAX>(bd, bi, ld[e], li[e]);
            }
    }
    if (i >= 0) {
#pragma unroll
        for (int p = 0; p < KMAX; ++p)
            if (p >= KMAX - k) nbr[(size_t)i * k + p - (KMAX - k)] = bi[p];
    }
}

template <int DMAX, int KMAX, int W>
static int launch_knn_blocks(hipStream_t st, const double* xs, const float* ys, const float* box,
                              const int* orig, const double* unit, int n, int k, int* nbr) {
    const int NB = (int)cdiv(n, kBlock);
    const size_t lds = (size_t)(W - 1) * k * 64 * (sizeof(double) + sizeof(int));
    auto kern = &knn_blocks_kernel<DMAX, KMAX, W, (DMAX > 8)>;
    if (lds > 48 * 1024)
        RVGP_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3(cdiv(NB, 8) * 8), dim3(64 * W), lds, st, xs, ys, box, orig, unit, n, k,
                       NB, nbr);
    RVGP_LAUNCH_CHECK();
    return RVGP_OK;
}

}  // namespace rvgp

using namespace rvgp;

extern "C" int rvgp_knn_blocks(const void* blocks, size_t bytes, int n, int D, int k, int* nbr,
                               void* stream) {
    RVGP_CHECK_ARG(k > 0 && k < n, "rvgp_knn_blocks: need 0 < k < n (k=%d, n=%d)", k, n);
    RVGP_CHECK_ARG(k <= 64, "rvgp_knn_blocks: k <= 64 supported");
    RVGP_CHECK_ARG(D >= 1 && D <= 64, "rvgp_knn_blocks: 1 <= D <= 64 supported");
    const BlockLayout b = block_layout(n, D, 0);
    RVGP_CHECK_ARG(blocks != nullptr && bytes >= b.total, "rvgp_knn_blocks: buffer too small");
    const char* p = static_cast<const char*>(blocks);
    const double* unit = reinterpret_cast<const double*>(p + b.unit);
    const float* box = reinterpret_cast<const float*>(p + b.box);
    const float* ys = reinterpret_cast<const float*>(p + b.ys);
    const int* orig = reinterpret_cast<const int*>(p + b.orig);
    const double* xs = reinterpret_cast<const double*>(p + b.xs);
    hipStream_t s = as_stream(stream);
#define RVGP_KNN_K(DM, KM, W) return launch_knn_blocks<DM, KM, W>(s, xs, ys, box, orig, unit, n, k, nbr)
#define RVGP_KNN_D(DM)                     \
    do {                                   \
        if (k <= 16) RVGP_KNN_K(DM, 16, 4); \
        else if (k <= 24) RVGP_KNN_K(DM, 24, 4); \
        else if (k <= 32) RVGP_KNN_K(DM, 32, 4); \
        else RVGP_KNN_K(DM, 64, 2);        \
    } while (0)
    switch (padded_dims(D)) {
        case 4: RVGP_KNN_D(4); break;
        case 8: RVGP_KNN_D(8); break;
        case 16: RVGP_KNN_D(16); break;
        case 32: RVGP_KNN_D(32); break;
        default: RVGP_KNN_D(64); break;
    }
#undef RVGP_KNN_D
#undef RVGP_KNN_K
    return RVGP_EINVAL;  // not reached
}
