// oriented.h -- the oriented 8-bit node of closest-point queries: its frame's arithmetic,
// shared by the builder (oriented.hip) and the traversal (traverse.h).
#pragma once

#include "gpurt_internal.h"
#include "tri_math.h"

namespace gpurt_impl {

// 1 - nx^2 - ny^2, the square of the normal's z component
__device__ __forceinline__ float frame_z2(float nx, float ny) { return fmaf(-nx, nx, fmaf(-ny, ny, 1.0f)); }

// The smallest rotation that takes the unit vector n (n.z >= 0) to the z axis, as rows:
//   (1 - h nx nx, -h nx ny, -nx), (-h nx ny, 1 - h ny ny, -ny), (nx, ny, nz), h = 1 / (1 + nz).
// It is orthonormal to a few ulps whatever nx and ny are (nz and h follow from them; the
// hardware's square root and reciprocal are good to an ulp).
struct Frame {
    float nx, ny, nz, h;
    __device__ __forceinline__ Frame(float x, float y) : nx(x), ny(y) {
        nz = __builtin_amdgcn_sqrtf(fmaxf(frame_z2(x, y), 0.0f));
        h = __builtin_amdgcn_rcpf(1.0f + nz);
    }
    __device__ __forceinline__ V3 to_local(V3 v) const {
        const float t = fmaf(nx, v.x, ny * v.y);
        const float u = fmaf(h, t, v.z);
        return v3(fmaf(-nx, u, v.x), fmaf(-ny, u, v.y), fmaf(nz, v.z, t));
    }
    __device__ __forceinline__ V3 to_world(V3 v) const {  // the transpose
        const float t = fmaf(nx, v.x, ny * v.y);
        const float u = fmaf(-h, t, v.z);
        return v3(fmaf(nx, u, v.x), fmaf(ny, u, v.y), fmaf(nz, v.z, -t));
    }
};

}  // namespace gpurt_impl
