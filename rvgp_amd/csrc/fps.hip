// a1  Furthest point sampling (RVGP/geometry.py:126-162).
//
// The reference materialises the dense n x n distance matrix and runs a
// numpy argmax/minimum loop.  Here no distance matrix exists: every
// distance is recomputed on the fly with the fixed direct formula of
// common.h, and the whole greedy loop runs in ONE persistent workgroup of
// 1024 threads (16 waves) so that an iteration costs one pass over the
// point set plus one block-wide (value, index) argmax -- no kernel launch
// and no host round trip per selected point.  The diameter (D.max(),
// geometry.py:144) is a separate all-pairs max over upper-triangle tiles.
#include "blocks.h"

#include <type_traits>

namespace rvgp {

// ---- diameter: max over i<j of d2 --------------------------------------
constexpr int kDiamRows = 256;  // points per block (one per thread)

// candidate tile staged in LDS: 32 KB whatever the dimension
template <int DMAX>
struct DiamTile {
    static constexpr int cols = 4096 / DMAX < 128 ? 4096 / DMAX : 128;
};

template <int DMAX>
__global__ __launch_bounds__(kDiamRows) void diam2_kernel(const double* __restrict__ x, int n,
                                                          int D,
                                                          unsigned long long* __restrict__ out) {
    constexpr int kDiamCols = DiamTile<DMAX>::cols;
    __shared__ double tile[kDiamCols * DMAX];
    const int i0 = blockIdx.x * kDiamRows;
    const int j0 = blockIdx.y * kDiamCols;
    if (j0 + kDiamCols - 1 <= i0) return;  // tile entirely at or below the diagonal
    const int i = i0 + threadIdx.x;
    double xi[DMAX];
#pragma unroll
    for (int k = 0; k < DMAX; ++k) xi[k] = (i < n && k < D) ? x[(size_t)i * D + k] : 0.0;
    for (int e = threadIdx.x; e < kDiamCols * D; e += kDiamRows) {
        int jj = e / D, kk = e - jj * D;
        int j = j0 + jj;
        tile[jj * DMAX + kk] = (j < n) ? x[(size_t)j * D + kk] : 0.0;
    }
    __syncthreads();
    double best = 0.0;
    if (i < n) {
        const int jend = min(kDiamCols, n - j0);
        for (int jj = 0; jj < jend; ++jj) {
            if (j0 + jj <= i) continue;
            double acc = 0.0;
#pragma unroll
            for (int k = 0; k < DMAX; ++k)
                if (k < D) {
                    double t = __dsub_rn(xi[k], tile[jj * DMAX + k]);
                    acc = __fma_rn(t, t, acc);
                }
            best = acc > best ? acc : best;
        }
    }
    best = wave_max(best);
    __shared__ double wbest[kDiamRows / kWave];
    if ((threadIdx.x & 63) == 0) wbest[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        double b = wbest[0];
        for (int w = 1; w < kDiamRows / kWave; ++w) b = wbest[w] > b ? wbest[w] : b;
        // Non-negative doubles order like their bit patterns.
        atomicMax(out, (unsigned long long)__double_as_longlong(b));
    }
}

// ---- the greedy loop ---------------------------------------------------
constexpr int kFpsThreads = 1024;
constexpr int kFpsMaxD = 8192;

struct ArgMax {
    double v;
    int i;
};

// (value descending, index ascending): numpy.argmax returns the first max.
__device__ __forceinline__ bool better(double v, int i, double bv, int bi) {
    return v > bv || (v == bv && i < bi);
}

__device__ __forceinline__ ArgMax block_argmax(double v, int i, double* sv, int* si) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        double ov = __shfl_xor(v, o, 64);
        int oi = __shfl_xor(i, o, 64);
        if (better(ov, oi, v, i)) { v = ov; i = oi; }
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { sv[w] = v; si[w] = i; }
    __syncthreads();
    ArgMax r{sv[0], si[0]};
    for (int k = 1; k < kFpsThreads / kWave; ++k)
        if (better(sv[k], si[k], r.v, r.i)) { r.v = sv[k]; r.i = si[k]; }
    __syncthreads();  // sv/si are reused by the next call
    return r;
}

__global__ __launch_bounds__(kFpsThreads) void fps_kernel(
    const double* __restrict__ x, int n, int D, int n_iter, int start, double spacing,
    int use_spacing, const double* __restrict__ diam2, double* __restrict__ ds,
    int* __restrict__ perm, double* __restrict__ lambdas, int* __restrict__ n_sel) {
    extern __shared__ double sx[];  // the selected point's D coordinates
    __shared__ double sv[kFpsThreads / kWave];
    __shared__ int si[kFpsThreads / kWave];
    const double diam = use_spacing ? sqrt(diam2[0]) : 1.0;

    for (int c = threadIdx.x; c < D; c += kFpsThreads) sx[c] = x[(size_t)start * D + c];
    __syncthreads();
    double bv = -1.0;
    int bi = 0x7fffffff;
    for (int j = threadIdx.x; j < n; j += kFpsThreads) {
        double v = sqrt(d2_direct(sx, x + (size_t)j * D, D));
        ds[j] = v;
        if (better(v, j, bv, bi)) { bv = v; bi = j; }
    }
    if (threadIdx.x == 0) {
        perm[0] = start;
        lambdas[0] = 0.0;
    }
    int count = n_iter;
    for (int it = 1; it < n_iter; ++it) {
        ArgMax am = block_argmax(bv, bi, sv, si);
        if (am.v < 0.0) {  // every distance is NaN: no point to select (am.i is none)
            count = it;
            break;
        }
        if (threadIdx.x == 0) {
            perm[it] = am.i;
            lambdas[it] = am.v;
        }
        if (use_spacing && am.v / diam < spacing) {  // geometry.py:156-160
            count = it;
            break;
        }
        for (int c = threadIdx.x; c < D; c += kFpsThreads) sx[c] = x[(size_t)am.i * D + c];
        __syncthreads();
        bv = -1.0;
        bi = 0x7fffffff;
        for (int j = threadIdx.x; j < n; j += kFpsThreads) {
            double v = sqrt(d2_direct(sx, x + (size_t)j * D, D));
            double o = ds[j];
            v = v < o ? v : o;  // np.minimum
            ds[j] = v;
            if (better(v, j, bv, bi)) { bv = v; bi = j; }
        }
        __syncthreads();  // sx is rewritten next iteration
    }
    if (threadIdx.x == 0) n_sel[0] = count;
}

// ---- the greedy loop over spatial blocks ------------------------------------
// The same selections with most of the work left out: a newly selected point
// changes only distances that are larger than its own distance, so a block of
// 64 points whose box (blocks.h) lies at least as far away as the block's
// largest remaining distance keeps every one of its distances.  One workgroup,
// as above, holds each block's box in registers (KB blocks per thread) and its
// largest distance with the point it belongs to in LDS; an iteration is an
// argmax over the blocks, a box test per block and an update of the few blocks
// that pass, one wave each.  The distances and their comparisons are the
// loop's above, so are the results.  Bound by the chain of an iteration
// (argmax, coordinates of the winner, block update, three barriers), whatever
// n is.

// Distances as keys: a non-negative double orders like its bits; -1 (NaN, no
// point) comes before all of them as a signed number.
__device__ __forceinline__ long long dist_key(double v) { return __double_as_longlong(v); }
__device__ __forceinline__ double no_nan(double v, bool valid) { return valid && v >= 0.0 ? v : -1.0; }

// Wave-wide maximum (signed, or unsigned) of a 32-bit value by DPP row moves
// and broadcasts, one instruction a step; in every lane.
template <bool SIGNED>
__device__ __forceinline__ int wave_max32(int v) {
    const int none = SIGNED ? (int)0x80000000 : 0;
#define RVGP_DPP(CTRL, ROWS)                                                            \
    {                                                                                   \
        const int o = __builtin_amdgcn_update_dpp(none, v, CTRL, ROWS, 0xf, false);     \
        v = SIGNED ? (o > v ? o : v) : ((unsigned)o > (unsigned)v ? o : v);             \
    }
    RVGP_DPP(0x111, 0xf)  // row_shr:1
    RVGP_DPP(0x112, 0xf)  // row_shr:2
    RVGP_DPP(0x114, 0xf)  // row_shr:4
    RVGP_DPP(0x118, 0xf)  // row_shr:8
    RVGP_DPP(0x142, 0xa)  // row_bcast:15
    RVGP_DPP(0x143, 0xc)  // row_bcast:31
#undef RVGP_DPP
    return __builtin_amdgcn_readlane(v, 63);
}

// Lane with the wave's largest key, the smallest `id` among equal ones (any
// lane if no lane has a distance); the high words decide first, then the low
// words of the lanes that hold them.
__device__ __forceinline__ int wave_winner(long long key, int id, long long* most) {
    const int h = (int)(key >> 32), hm = wave_max32<true>(h);
    const int lm = wave_max32<false>(h == hm ? (int)key : 0);
    *most = ((long long)hm << 32) | (unsigned)lm;
    unsigned long long m = __ballot(key == *most);
    int l = __builtin_ctzll(m);
    if (hm >= 0 && (m & (m - 1))) {  // several: the smallest id
        const int best = ~wave_max32<false>(key == *most ? ~id : 0);
        l = __builtin_ctzll(__ballot(key == *most && id == best));
    }
    return l;
}

// Smallest distance that does not end the sample: v / diam < spacing
// (geometry.py:156-160) exactly when v < stop_limit -- the division is
// monotone in v -- without a division on every selection's path.
__device__ double stop_limit(double diam, double spacing) {
    if (!(diam > 0.0) || !(spacing > 0.0)) return -1.0;  // 0 / 0 and v / diam < 0 never end it
    double v = spacing * diam;
    if (!(v < __builtin_huge_val())) return v;
    while (v > 0.0 && v / diam >= spacing) v = __longlong_as_double(__double_as_longlong(v) - 1);
    while (v / diam < spacing) v = __longlong_as_double(__double_as_longlong(v) + 1);
    return v;
}

// ---- the greedy loop in registers -------------------------------------------
// Up to R points per thread, coordinates (D <= 3) and squared distances in
// registers, a copy of the coordinates in LDS for the winner's: no global
// memory on an iteration's path, and one LDS hand-over of the waves'
// candidates (two sets, so one barrier an iteration).  The loop keeps squared
// distances -- sqrt is monotone, so the minima and maxima are the same -- and
// takes the root of the winner alone.  Only the lowest-index rule among equal
// distances needs more: different squares can share a root (at most three
// neighbouring doubles do), so whenever another point's square lies within
// kNearTie units in the last place below the largest, the roots are compared
// and the lowest index among equal ones is taken.
// Bound by the instructions of one iteration on four SIMDs.
// n = 2503, 1349 selections: 5.5 -> 1.9 ms (1.4 us a selection).
constexpr int kFpsResidentMax = 256 * 16;
constexpr int kNearTie = 8;

template <int R>
__global__ __launch_bounds__(256) void fps_resident_kernel(
    const double* __restrict__ x, int n, int D, int n_iter, int start, double spacing,
    int use_spacing, const double* __restrict__ diam2, int* __restrict__ perm,
    double* __restrict__ lambdas, int* __restrict__ n_sel) {
    constexpr int NT = 256, NW = NT / kWave;
    extern __shared__ double xl[];  // n x 3
    __shared__ long long wkey[2][NW];
    __shared__ int wid[2][NW], wnear[2][NW], wlow[NW];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const double limit = use_spacing ? stop_limit(sqrt(diam2[0]), spacing) : -1.0;
    double px[R][3], d2[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int j = r * NT + tid;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            px[r][k] = j < n && k < D ? x[(size_t)j * D + k] : 0.0;
            if (j < n) xl[j * 3 + k] = px[r][k];
        }
    }
    __syncthreads();
    double sx[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) sx[k] = xl[start * 3 + k];
    if (tid == 0) {
        perm[0] = start;
        lambdas[0] = 0.0;
    }
    int made = n_iter;
    for (int it = 1; it < n_iter; ++it) {
        // distances to the last selection, and this thread's farthest point
        double far = -2.0;
        int fr = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            double acc = 0.0;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const double t = __dsub_rn(sx[c], px[r][c]);
                acc = __fma_rn(t, t, acc);
            }
            d2[r] = it == 1 ? no_nan(acc, r * NT + tid < n) : (acc < d2[r] ? acc : d2[r]);
            if (d2[r] > far) { far = d2[r]; fr = r; }
        }
        long long most;
        const int id = fr * NT + tid;
        const int l = wave_winner(dist_key(far), id, &most);
        // other points of this wave just below the largest: their high words
        // first, one instruction each, the exact test where those agree
        const int hm = (int)(most >> 32) - 1;
        int near = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) near += __popcll(__ballot((int)(dist_key(d2[r]) >> 32) >= hm));
        if (near > 1) {
            near = 0;
#pragma unroll
            for (int r = 0; r < R; ++r)
                near |= (unsigned long long)(most - dist_key(d2[r]) - 1) < kNearTie;
            near = __any(near);
        } else {
            near = 0;
        }
        const int b = it & 1;
        if (lane == l) {
            wkey[b][w] = most;
            wid[b][w] = id;
            wnear[b][w] = near;
        }
        __syncthreads();
        long long top = wkey[b][0];
        int wino = wid[b][0];
#pragma unroll
        for (int e = 1; e < NW; ++e) {
            const long long o = wkey[b][e];
            const int oi = wid[b][e];
            if (o > top || (o == top && oi < wino)) { top = o; wino = oi; }
        }
        if (top < 0) {  // every distance is NaN: nothing to select
            made = it;
            break;
        }
        near = 0;
#pragma unroll
        for (int e = 0; e < NW; ++e) {
            const unsigned long long below = (unsigned long long)(top - wkey[b][e]);
            near |= below == 0 ? wnear[b][e] : below <= kNearTie;
        }
        const double v = sqrt(__longlong_as_double(top));
        if (near) {
            // the lowest index among the points at distance v
            int lowest = 0x7fffffff;
#pragma unroll
            for (int r = R - 1; r >= 0; --r)
                if (d2[r] >= 0.0 && sqrt(d2[r]) == v) lowest = r * NT + tid;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) lowest = min(lowest, __shfl_xor(lowest, o, 64));
            if (lane == 0) wlow[w] = lowest;
            __syncthreads();
#pragma unroll
            for (int e = 0; e < NW; ++e) wino = min(wino, wlow[e]);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) sx[c] = xl[wino * 3 + c];
        if (tid == 0) {
            perm[it] = wino;
            lambdas[it] = v;
        }
        if (v < limit) {
            made = it;
            break;
        }
    }
    if (tid == 0) n_sel[0] = made;
}

template <int R>
static int launch_fps_resident(hipStream_t s, const double* x, int n, int D, int n_iter, int start,
                               double spacing, int use_spacing, const double* diam2, int* perm,
                               double* lambdas, int* n_sel) {
    const size_t lds = sizeof(double) * 3 * (size_t)n;
    if (lds > 48 * 1024)
        RVGP_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&fps_resident_kernel<R>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((fps_resident_kernel<R>), dim3(1), dim3(256), lds, s, x, n, D, n_iter, start,
                       spacing, use_spacing, diam2, perm, lambdas, n_sel);
    RVGP_LAUNCH_CHECK();
    return RVGP_OK;
}

constexpr int kFpsMaxBlocks = 4096;  // blocks of one launch

// The first four waves hold the boxes and do the argmax and the tests -- more
// would repeat the same instructions on the same SIMDs --, all of them the
// updates, two blocks at a time.  CACHE: each block's candidate (its largest
// distance's point) keeps its box coordinates -- and, DC = 3, its
// coordinates -- in LDS, so that the winner's are at hand without a trip to the
// L2.
template <int KB, int NT, int TT, int DC, bool CACHE>
__global__ __launch_bounds__(NT) void fps_blocks_kernel(
    const double* __restrict__ x, const double* __restrict__ xt, const float* __restrict__ ys,
    const float* __restrict__ box, const int* __restrict__ orig, const double* __restrict__ unit,
    int n, int D, int NB, int start, int n_iter, double spacing, int use_spacing,
    const double* __restrict__ diam2, double* __restrict__ ds, int* __restrict__ perm,
    double* __restrict__ lambdas, int* __restrict__ n_sel) {
    constexpr int NW = NT / kWave, TW = TT / kWave;  // all waves; testing threads, waves
    extern __shared__ long long bkey[];  // NB keys, then limits, ids, positions, the list
    float* blim = reinterpret_cast<float*>(bkey + NB);
    int* bid = reinterpret_cast<int*>(blim + NB);
    int* bpos = bid + NB;
    int* list = bpos + NB;
    float* by = reinterpret_cast<float*>(list + NB);  // CACHE: NB x 6
    double* bx = reinterpret_cast<double*>(by + (NB + (NB & 1)) * kBoxDims);  // and, DC = 3, NB x 3
    __shared__ long long wkey[TW];
    __shared__ int wid[TW], wblk[TW];
    __shared__ int count[2];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const double inv2 = unit[1];
    const double limit = use_spacing ? stop_limit(sqrt(diam2[0]), spacing) : -1.0;
    const int Dn = DC > 0 ? DC : D;

    float lo[KB][kBoxDims], hi[KB][kBoxDims];
#pragma unroll
    for (int q = 0; q < KB; ++q) {
        const int b = tid + q * TT;
        const bool own = w < TW && b < NB;
#pragma unroll
        for (int d = 0; d < kBoxDims; ++d) {
            lo[q][d] = own ? box[(size_t)b * kBoxStride + d] : 0.0f;
            hi[q][d] = own ? box[(size_t)b * kBoxStride + kBoxRow + d] : 0.0f;
        }
    }

    // the distances of blocks b[0], b[1] (b[1] < 0: one block) against the point
    // with coordinates xq, one lane per point; first: there is no distance yet
    auto update = [&](const int (&b)[2], const double* xq, bool first) {
        double v[2], xl[2][3];
        float yl[2][kBoxDims];
        int id[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (b[h] < 0) continue;
            const int p = b[h] * kBlock + lane;
            id[h] = p < n ? orig[p] : 0x7fffffff;
            v[h] = p < n && !first ? ds[p] : 0.0;
            if (CACHE)
#pragma unroll
                for (int d = 0; d < kBoxDims; ++d) yl[h][d] = ys[(size_t)p * kBoxRow + d];
            if (DC == 3)
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    xl[h][k] = xt[((size_t)b[h] * 3 + k) * kBlock + lane];
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (b[h] < 0) continue;
            const int p = b[h] * kBlock + lane;
            double acc = 0.0;
            if (DC == 3) {
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const double t = __dsub_rn(xq[k], xl[h][k]);
                    acc = __fma_rn(t, t, acc);
                }
            } else {
                const double* xb = xt + (size_t)b[h] * Dn * kBlock + lane;
#pragma unroll 8
                for (int k = 0; k < Dn; ++k) {
                    const double t = __dsub_rn(xq[k], xb[(size_t)k * kBlock]);
                    acc = __fma_rn(t, t, acc);
                }
            }
            const double s = sqrt(acc);
            v[h] = first ? no_nan(s, p < n) : (s < v[h] ? s : v[h]);  // np.minimum
            if (p < n) ds[p] = v[h];
            else v[h] = -1.0;
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (b[h] < 0) continue;
            long long most;
            const int l = wave_winner(dist_key(v[h]), id[h], &most);
            if (lane == l) {
                bkey[b[h]] = most;
                bid[b[h]] = id[h];
                bpos[b[h]] = b[h] * kBlock + lane;
                // no distance left that a point beyond this bound could lower
                blim[b[h]] = most < 0 ? -1.0f : inv2 > 0.0 ? box_limit(v[h] * v[h], inv2)
                                                            : __builtin_huge_valf();
                if (CACHE) {
#pragma unroll
                    for (int d = 0; d < kBoxDims; ++d) by[b[h] * kBoxDims + d] = yl[h][d];
                    if (DC == 3)
#pragma unroll
                        for (int d = 0; d < 3; ++d) bx[b[h] * 3 + d] = xl[h][d];
                }
            }
        }
    };

    if (tid == 0) {
        perm[0] = start;
        lambdas[0] = 0.0;
        count[0] = count[1] = 0;
    }
    for (int b = w; b < NB; b += 2 * NW) {
        const int bb[2] = {b, b + NW < NB ? b + NW : -1};
        update(bb, x + (size_t)start * Dn, true);
    }
    __syncthreads();
    int made = n_iter;
    for (int it = 1; it < n_iter; ++it) {
        if (w < TW) {  // argmax over the blocks
            long long k = -1, most;
            int id = 0x7fffffff, bb = 0;
#pragma unroll
            for (int q = 0; q < KB; ++q) {
                const int b = tid + q * TT;
                if (b < NB) {
                    const long long o = bkey[b];
                    const int oi = bid[b];
                    if (o > k || (o == k && oi < id)) { k = o; id = oi; bb = b; }
                }
            }
            const int l = wave_winner(k, id, &most);
            if (lane == l) { wkey[w] = most; wid[w] = id; wblk[w] = bb; }
        }
        if (tid == 0) count[(it + 1) & 1] = 0;  // the next iteration's list
        __syncthreads();
        long long top = wkey[0];
        int wino = wid[0], win = wblk[0];  // the winner and its block
#pragma unroll
        for (int e = 1; e < TW; ++e) {
            const long long o = wkey[e];
            const int oi = wid[e];
            if (o > top || (o == top && oi < wino)) { top = o; wino = oi; win = wblk[e]; }
        }
        wino = __builtin_amdgcn_readfirstlane(wino);
        win = __builtin_amdgcn_readfirstlane(win);
        if (top < 0) {  // every distance is NaN: nothing to select
            made = it;
            break;
        }
        const double v = __longlong_as_double(top);
        if (tid == 0) {
            perm[it] = wino;
            lambdas[it] = v;
        }
        if (v < limit) {
            made = it;
            break;
        }
        const double* xq = x + (size_t)wino * Dn;
        double xw[3];
        if (CACHE && DC == 3) {
#pragma unroll
            for (int d = 0; d < 3; ++d) xw[d] = bx[win * 3 + d];
            xq = xw;
        }
        if (w < TW) {  // blocks that the new point can change
            float y[kBoxDims];
#pragma unroll
            for (int d = 0; d < kBoxDims; ++d)
                y[d] = CACHE ? by[win * kBoxDims + d] : ys[(size_t)bpos[win] * kBoxRow + d];
#pragma unroll
            for (int q = 0; q < KB; ++q) {
                const int b = tid + q * TT;
                bool pass = b < NB;
                if (pass) {
                    float lb = 0.0f;
#pragma unroll
                    for (int d = 0; d < kBoxDims; ++d) {
                        const float t = fmaxf(0.0f, fmaxf(lo[q][d] - y[d], y[d] - hi[q][d]));
                        lb = fmaf(t, t, lb);
                    }
                    pass = lb <= blim[b];
                }
                const unsigned long long mask = __ballot(pass);
                if (mask != 0) {
                    int base = 0;
                    if (lane == 0) base = atomicAdd(&count[it & 1], __popcll(mask));
                    base = __builtin_amdgcn_readfirstlane(base);
                    if (pass) list[base + __popcll(mask & ((1ULL << lane) - 1))] = b;
                }
            }
        }
        __syncthreads();
        const int nl = count[it & 1];
        for (int a = w; a < nl; a += 2 * NW) {
            const int bb[2] = {__builtin_amdgcn_readfirstlane(list[a]),
                               a + NW < nl ? __builtin_amdgcn_readfirstlane(list[a + NW]) : -1};
            update(bb, xq, false);
        }
        __syncthreads();
    }
    if (tid == 0) n_sel[0] = made;
}

template <int KB, int NT, int TT>
static int launch_fps_blocks(hipStream_t s, const double* x, const char* p, const BlockLayout& L, int n,
                             int D, int start, int n_iter, double spacing, int use_spacing,
                             const double* diam2, double* ds, int* perm, double* lambdas, int* n_sel) {
    // keys, limits, ids, positions, list; CACHE: box coordinates and coordinates
    constexpr bool CACHE = KB * TT <= 2048;
    const size_t lds = (size_t)L.NB * 24 + (CACHE ? (size_t)(L.NB + 1) * (24 + 24) : 0);
    auto go = [&](auto* kern) -> int {
        if (lds > 48 * 1024)
            RVGP_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(kern, dim3(1), dim3(NT), lds, s, x,
                           reinterpret_cast<const double*>(p + L.xs),
                           reinterpret_cast<const float*>(p + L.ys),
                           reinterpret_cast<const float*>(p + L.box),
                           reinterpret_cast<const int*>(p + L.orig),
                           reinterpret_cast<const double*>(p + L.unit), n, D, L.NB, start, n_iter,
                           spacing, use_spacing, diam2, ds, perm, lambdas, n_sel);
        RVGP_LAUNCH_CHECK();
        return RVGP_OK;
    };
    return D == 3 ? go(&fps_blocks_kernel<KB, NT, TT, 3, CACHE>) : go(&fps_blocks_kernel<KB, NT, TT, 0, CACHE>);
}

}  // namespace rvgp

using namespace rvgp;

extern "C" int rvgp_fps_diam2(const double* x, int n, int D, double* diam2, void* stream) {
    RVGP_CHECK_ARG(n >= 1 && D >= 1 && D <= 64, "rvgp_fps_diam2: need n >= 1 and 1 <= D <= 64");
    auto* out = reinterpret_cast<unsigned long long*>(diam2);
#define RVGP_DIAM(DM)                                                                    \
    hipLaunchKernelGGL(diam2_kernel<DM>, dim3(cdiv(n, kDiamRows), cdiv(n, DiamTile<DM>::cols)), \
                       dim3(kDiamRows), 0, as_stream(stream), x, n, D, out)
    if (D <= 4) RVGP_DIAM(4);
    else if (D <= 16) RVGP_DIAM(16);
    else if (D <= 32) RVGP_DIAM(32);
    else RVGP_DIAM(64);
#undef RVGP_DIAM
    RVGP_LAUNCH_CHECK();
    return RVGP_OK;
}

extern "C" int rvgp_fps(const double* x, int n, int D, int n_iter, int start_idx, double spacing,
                        int use_spacing, const double* diam2, double* ds, int* perm,
                        double* lambdas, int* n_sel, void* stream) {
    // the selected point is staged in LDS: D <= 8192 (64 KiB); the spacing
    // mode's diameter kernel takes D <= 64
    RVGP_CHECK_ARG(n >= 1 && D >= 1 && D <= kFpsMaxD, "rvgp_fps: need n >= 1 and 1 <= D <= %d",
                   kFpsMaxD);
    RVGP_CHECK_ARG(n_iter >= 1, "rvgp_fps: n_iter must be >= 1");
    RVGP_CHECK_ARG(start_idx >= 0 && start_idx < n, "rvgp_fps: start_idx out of range");
    RVGP_CHECK_ARG(!use_spacing || diam2 != nullptr, "rvgp_fps: spacing mode needs diam2");
    if (D <= 3 && n <= kFpsResidentMax) {
#define RVGP_FPS_RES(R)                                                                          \
    launch_fps_resident<R>(as_stream(stream), x, n, D, n_iter, start_idx, spacing, use_spacing, \
                           diam2, perm, lambdas, n_sel)
        if (n <= 256 * 2) return RVGP_FPS_RES(2);
        if (n <= 256 * 4) return RVGP_FPS_RES(4);
        if (n <= 256 * 6) return RVGP_FPS_RES(6);
        if (n <= 256 * 8) return RVGP_FPS_RES(8);
        if (n <= 256 * 10) return RVGP_FPS_RES(10);
        if (n <= 256 * 13) return RVGP_FPS_RES(13);
        return RVGP_FPS_RES(16);
#undef RVGP_FPS_RES
    }
    hipLaunchKernelGGL(fps_kernel, dim3(1), dim3(kFpsThreads), sizeof(double) * D, as_stream(stream),
                       x, n, D,
                       n_iter, start_idx, spacing, use_spacing, diam2, ds, perm, lambdas, n_sel);
    RVGP_LAUNCH_CHECK();
    return RVGP_OK;
}

extern "C" int rvgp_fps_blocks(const double* x, const void* blocks, size_t bytes, int n, int D,
                               int n_iter, int start_idx, double spacing, int use_spacing,
                               const double* diam2, double* ds, int* perm, double* lambdas,
                               int* n_sel, void* stream) {
    RVGP_CHECK_ARG(n >= 1 && n <= kFpsMaxBlocks * kBlock && D >= 1 && D <= 64,
                   "rvgp_fps_blocks: need 1 <= n <= %d and 1 <= D <= 64", kFpsMaxBlocks * kBlock);
    RVGP_CHECK_ARG(n_iter >= 1, "rvgp_fps_blocks: n_iter must be >= 1");
    RVGP_CHECK_ARG(start_idx >= 0 && start_idx < n, "rvgp_fps_blocks: start_idx out of range");
    RVGP_CHECK_ARG(!use_spacing || diam2 != nullptr, "rvgp_fps_blocks: spacing mode needs diam2");
    const BlockLayout L = block_layout(n, D, 1);
    RVGP_CHECK_ARG(blocks != nullptr && bytes >= L.total, "rvgp_fps_blocks: buffer too small");
    const char* p = static_cast<const char*>(blocks);
    hipStream_t s = as_stream(stream);
#define RVGP_FPS(KB, NT, TT)                                                                          \
    launch_fps_blocks<KB, NT, TT>(s, x, p, L, n, D, start_idx, n_iter, spacing, use_spacing, diam2, ds, \
                              perm, lambdas, n_sel)
    // testing threads and blocks per thread: enough waves for the updates of an
    // iteration, few enough that the tests do not share a SIMD's issue slots
    if (L.NB <= 256) return RVGP_FPS(2, 512, 128);    // n = 8,000: 2.0 us a selection
    if (L.NB <= 512) return RVGP_FPS(2, 1024, 256);   // n = 20,000: 2.3 us (15 us before)
    if (L.NB <= 1024) return RVGP_FPS(2, 1024, 512);  // n = 60,000: 2.7 us
    if (L.NB <= 2048) return RVGP_FPS(4, 1024, 512);  // n = 100,000: 3.5 us (69 us before)
    return RVGP_FPS(16, 512, 256);                    // n = 200,000: 6.2 us
#undef RVGP_FPS
}
