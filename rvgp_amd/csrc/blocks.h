// Spatial blocks: the points in the order of a space-filling curve, cut into
// blocks of kBlock consecutive ones with the bounding box of each.
//
// The kNN scan and the farthest-point loop skip a whole block when a lower
// bound of every distance into it says that no point of it can matter; the
// distances themselves are always d2_direct's.  The bounds are FP32 on
// "box coordinates" y (P <= 6 per point): the points' own coordinates for
// D <= 6, else their six leading principal coordinates, shifted and scaled
// into [-1, 1].  An orthonormal projection never lengthens a distance, and
// the scaling keeps FP32 from over- or underflowing whatever the data's units
// are.  kBoxSlack covers the FP32 rounding of the coordinates (6e-8 each) and
// of the bound, kBoxShrink the relative rounding of its sum, so that a block
// is skipped only if every exact distance into it is larger than the limit.
#pragma once
#include "common.h"

namespace rvgp {

constexpr int kBlock = 64;       // points per block: one wave
constexpr int kBoxDims = 6;      // box coordinates per point
constexpr int kBoxRow = 8;       // their row stride (floats)
constexpr int kBoxStride = 16;   // floats per box: lo[8], hi[8]
constexpr float kBoxSlack = 1e-6f;

// FP32 limit such that a bound above it proves d2 > limit2 (limit2: a squared
// distance in the data's units, inv2 = 1 / unit^2): (sqrt(limit2) + slack)^2
// with every rounding upwards.
__device__ __forceinline__ float box_limit(double limit2, double inv2) {
    const float s = sqrtf((float)(limit2 * inv2)) * 1.000001f + kBoxSlack;
    return s * s * 1.00001f + 1e-30f;
}

// coordinates per row of the gathered points
static inline int padded_dims(int D) { return D <= 4 ? 4 : D <= 8 ? 8 : D <= 16 ? 16 : D <= 32 ? 32 : 64; }

// offsets of a blocks buffer (bytes); transposed: coordinates stored D x kBlock
// per block, else in rows of padded_dims(D)
struct BlockLayout {
    size_t unit, box, ys, orig, xs, total;
    int NB;
};

static inline BlockLayout block_layout(int n, int D, int transposed) {
    BlockLayout b;
    b.NB = (int)cdiv(n, kBlock);
    const size_t np = (size_t)b.NB * kBlock;
    b.unit = 0;
    b.box = 256;
    b.ys = b.box + align_up(sizeof(float) * kBoxStride * (size_t)b.NB, 256);
    b.orig = b.ys + align_up(sizeof(float) * kBoxRow * np, 256);
    b.xs = b.orig + align_up(sizeof(int) * np, 256);
    b.total = b.xs + sizeof(double) * (transposed ? D : padded_dims(D)) * np;
    return b;
}

}  // namespace rvgp
