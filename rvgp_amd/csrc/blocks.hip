// Space-filling order and spatial blocks; blocks.h says what a block is and
// why a bound on its box may skip it.
#include "blocks.h"

namespace rvgp {

// Morton key of every point: coordinate d of Y quantised to `bits` bits over
// its range, bits interleaved from the top (coordinate 0 first).  One launch;
// the same keys as ~4 * bits * P elementwise passes over int64 arrays.
__global__ __launch_bounds__(256) void morton_key_kernel(const double* __restrict__ Y, int ldy, int n,
                                                         int P, int bits,
                                                         const double* __restrict__ lo,
                                                         const double* __restrict__ hi,
                                                         long long* __restrict__ key) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const double top = (double)((1LL << bits) - 1);
    auto quant = [&](int d) -> long long {
        const double span = hi[d] - lo[d];
        const double v = rint((Y[(size_t)i * ldy + d] - lo[d]) / (span > 1e-300 ? span : 1e-300) * top);
        return v > 0.0 ? (v < top ? (long long)v : (long long)top) : 0;  // NaN: 0
    };
    long long k = 0;
    if (P <= kBoxDims) {
        long long q[kBoxDims];
#pragma unroll
        for (int d = 0; d < kBoxDims; ++d) q[d] = d < P ? quant(d) : 0;
        for (int b = bits - 1; b >= 0; --b)
#pragma unroll
            for (int d = 0; d < kBoxDims; ++d)
                if (d < P) k = (k << 1) | ((q[d] >> b) & 1);
    } else {
        for (int b = bits - 1; b >= 0; --b)
            for (int d = 0; d < P; ++d) k = (k << 1) | ((quant(d) >> b) & 1);
    }
    key[i] = k;
}

// Box coordinates' unit: half the largest range, as 1 / unit and 1 / unit^2;
// 0 (every bound 0, nothing skipped) for a range that is 0 or not finite.
__global__ void block_unit_kernel(int P, const double* __restrict__ lo, const double* __restrict__ hi,
                                  double* __restrict__ unit) {
    double h = 0.0;
    bool ok = true;
    for (int d = 0; d < P; ++d) {
        const double s = 0.5 * hi[d] - 0.5 * lo[d];
        ok = ok && s >= 0.0 && s < 1e150;
        h = s > h ? s : h;
    }
    ok = ok && h > 1e-150;
    unit[0] = ok ? 1.0 / h : 0.0;
    unit[1] = ok ? (1.0 / h) * (1.0 / h) : 0.0;
}

// One wave per block: gathers its points into curve order (xs: rows padded
// with zeros to DP doubles; or, transposed, D x kBlock per block), their box
// coordinates, the original indices (-1 past n) and the box.
__global__ __launch_bounds__(kBlock) void block_build_kernel(
    const double* __restrict__ x, int n, int D, const double* __restrict__ Y, int ldy, int P,
    const double* __restrict__ lo, const double* __restrict__ hi, const double* __restrict__ unit,
    const long long* __restrict__ order, int transposed, int DP, double* __restrict__ xs,
    float* __restrict__ ys, float* __restrict__ box, int* __restrict__ orig) {
    const int b = blockIdx.x, lane = threadIdx.x;
    const int p = b * kBlock + lane;
    const int i = p < n ? (int)order[p] : -1;
    const bool in = (unsigned)i < (unsigned)n;
    orig[p] = in ? i : -1;
    const double inv = unit[0];
#pragma unroll
    for (int d = 0; d < kBoxRow; ++d) {
        float v = 0.0f;
        if (d < P && in && inv > 0.0) {
            v = (float)((Y[(size_t)i * ldy + d] - (0.5 * lo[d] + 0.5 * hi[d])) * inv);
            if (!(v >= -2.0f && v <= 2.0f)) v = 0.0f;  // NaN: its distances are NaN too
        }
        ys[(size_t)p * kBoxRow + d] = v;
        float a = in ? v : 3.0f, c = in ? v : -3.0f;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            a = fminf(a, __shfl_xor(a, o, 64));
            c = fmaxf(c, __shfl_xor(c, o, 64));
        }
        if (lane == 0) {
            box[(size_t)b * kBoxStride + d] = a;
            box[(size_t)b * kBoxStride + kBoxRow + d] = c;
        }
    }
    if (transposed) {
        for (int k = 0; k < D; ++k)
            xs[((size_t)b * D + k) * kBlock + lane] = in ? x[(size_t)i * D + k] : 0.0;
    } else {
        for (int e = lane; e < kBlock * DP; e += kBlock) {  // coalesced along each row
            const int r = e / DP, k = e - r * DP;
            const int j = __shfl(i, r, 64);
            xs[((size_t)b * kBlock + r) * DP + k] = (j >= 0 && k < D) ? x[(size_t)j * D + k] : 0.0;
        }
    }
}

}  // namespace rvgp

using namespace rvgp;

extern "C" int rvgp_morton_keys(const double* Y, int ldy, int n, int P, const double* lo,
                                const double* hi, long long* keys, void* stream) {
    RVGP_CHECK_ARG(n >= 1 && P >= 1 && P <= 62 && ldy >= P,
                   "rvgp_morton_keys: need n >= 1, 1 <= P <= 62");
    const int bits = 62 / P < 20 ? 62 / P : 20;
    hipLaunchKernelGGL(morton_key_kernel, dim3(cdiv(n, 256)), dim3(256), 0, as_stream(stream), Y, ldy,
                       n, P, bits, lo, hi, keys);
    RVGP_LAUNCH_CHECK();
    return RVGP_OK;
}

extern "C" size_t rvgp_blocks_bytes(int n, int D, int transposed) {
    if (n < 1 || D < 1 || D > 64) return 0;
    return block_layout(n, D, transposed).total;
}

extern "C" int rvgp_blocks(const double* x, int n, int D, const double* Y, int ldy, int P,
                           const double* lo, const double* hi, const long long* order,
                           int transposed, void* blocks, size_t bytes, void* stream) {
    RVGP_CHECK_ARG(n >= 1 && D >= 1 && D <= 64, "rvgp_blocks: need n >= 1 and 1 <= D <= 64");
    RVGP_CHECK_ARG(P >= 1 && P <= kBoxDims && ldy >= P, "rvgp_blocks: need 1 <= P <= %d", kBoxDims);
    const BlockLayout b = block_layout(n, D, transposed);
    RVGP_CHECK_ARG(blocks != nullptr && bytes >= b.total, "rvgp_blocks: buffer too small");
    char* p = static_cast<char*>(blocks);
    hipStream_t s = as_stream(stream);
    double* unit = reinterpret_cast<double*>(p + b.unit);
    hipLaunchKernelGGL(block_unit_kernel, dim3(1), dim3(1), 0, s, P, lo, hi, unit);
    hipLaunchKernelGGL(block_build_kernel, dim3(b.NB), dim3(kBlock), 0, s, x, n, D, Y, ldy, P, lo, hi,
                       unit, order, transposed, padded_dims(D),
                       reinterpret_cast<double*>(p + b.xs), reinterpret_cast<float*>(p + b.ys),
                       reinterpret_cast<float*>(p + b.box), reinterpret_cast<int*>(p + b.orig));
    RVGP_LAUNCH_CHECK();
    return RVGP_OK;
}
