// Shared helpers for the RVGP HIP kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

#include "../../include/rvgp.h"

namespace rvgp {

void set_error(const char* fmt, ...);

// Return-on-error helpers for the C-ABI layer.
#define RVGP_CHECK_ARG(cond, ...)                     \
    do {                                              \
        if (!(cond)) {                                \
            ::rvgp::set_error(__VA_ARGS__);           \
            return RVGP_EINVAL;                       \
        }                                             \
    } while (0)

#define RVGP_CHECK_HIP(expr)                                                     \
    do {                                                                         \
        hipError_t _e = (expr);                                                  \
        if (_e != hipSuccess) {                                                  \
            ::rvgp::set_error("%s:%d %s: %s", __FILE__, __LINE__, #expr,          \
                              hipGetErrorString(_e));                            \
            return RVGP_EHIP;                                                    \
        }                                                                        \
    } while (0)

#define RVGP_LAUNCH_CHECK() RVGP_CHECK_HIP(hipGetLastError())

static inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

static inline unsigned int cdiv(size_t a, size_t b) { return (unsigned int)((a + b - 1) / b); }
static inline size_t align_up(size_t a, size_t b) { return (a + b - 1) / b * b; }

constexpr int kWave = 64;

// Filter values that an optimiser's trial step sends to 0 (a sigma_f of 1e-300, a
// steep filter) are raised to this where 1 / S is taken: it stays finite, S
// itself is as good as 0.
constexpr double kMinFilter = 1e-280;

// Wave-wide reductions via cross-lane shuffles.
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

template <typename T>
__device__ __forceinline__ T wave_max(T v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        T u = __shfl_xor(v, o, 64);
        v = u > v ? u : v;
    }
    return v;
}

// Broadcast lane `l` of v (l wave-uniform) -- v_readlane into an SGPR.
__device__ __forceinline__ float bcast(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double bcast(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Lane l of each row of 16 lanes to all of that row, without a detour over
// scalar registers (whose hazard costs as much as the product).  l is constant
// at every use, so one case is left of the switch.
__device__ __forceinline__ double row_bcast(double v, int l) {
    switch (l) {
#define RVGP_LANE(L)                                                             \
    case L:                                                                      \
        v = __builtin_amdgcn_update_dpp(v, v, 0x150 + L, 0xf, 0xf, true);        \
        break;
        RVGP_LANE(0) RVGP_LANE(1) RVGP_LANE(2) RVGP_LANE(3) RVGP_LANE(4) RVGP_LANE(5)
        RVGP_LANE(6) RVGP_LANE(7) RVGP_LANE(8) RVGP_LANE(9) RVGP_LANE(10) RVGP_LANE(11)
        RVGP_LANE(12) RVGP_LANE(13) RVGP_LANE(14) RVGP_LANE(15)
#undef RVGP_LANE
    }
    return v;
}

// Sum over the wave by DPP row moves and broadcasts, in every lane.
__device__ __forceinline__ double wave_sum_dpp(double v) {
#define RVGP_STEP(CTRL, ROWS)                                                                     \
    {                                                                                             \
        const long long b = __double_as_longlong(v);                                             \
        const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);            \
        const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);    \
        v += __longlong_as_double(((long long)hi << 32) | (unsigned)lo);                          \
    }
    RVGP_STEP(0x111, 0xf)
    RVGP_STEP(0x112, 0xf)
    RVGP_STEP(0x114, 0xf)
    RVGP_STEP(0x118, 0xf)
    RVGP_STEP(0x142, 0xa)
    RVGP_STEP(0x143, 0xc)
#undef RVGP_STEP
    return bcast(v, 63);
}

// Direct squared distance with a fixed operation order:
//   acc = fma(t_k, t_k, acc), t_k = a_k - b_k, k = 0..D-1.
// The CPU oracle uses the same sequence, so results agree bit for bit.
__device__ __forceinline__ double d2_direct(const double* __restrict__ a,
                                            const double* __restrict__ b, int D) {
    double acc = 0.0;
    for (int k = 0; k < D; ++k) {
        double t = __dsub_rn(a[k], b[k]);
        acc = __fma_rn(t, t, acc);
    }
    return acc;
}

}  // namespace rvgp
