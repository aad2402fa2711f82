// build_common.h -- device helpers shared by the builder (build.hip) and the treelet
// restructuring (treelet.hip).
#pragma once

#include "gpurt_internal.h"

namespace gpurt_impl {

// per-mesh statistics: [cmin xyz, cmax xyz, max|coord|, unused] as ordered uints.
// k_prep accumulates into kRep replicas (block b uses replica b % kRep) so that the
// atomics of ~N/64 waves do not serialise on 7 addresses; k_reduce_stats folds them.
constexpr int kStat = 8;
constexpr int kRep = 64;

// IEEE floats mapped to uints with the same order (for atomic min/max)
__device__ __forceinline__ uint32_t f2o(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float o2f(uint32_t u) {
    u = (u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u;
    return __uint_as_float(u);
}

// Binary references: internal node i -> i; leaf (sorted primitive p) -> kLeafBit | p.
// An internal node is a 48-byte record of three float4: (lo.xyz, left), (hi.xyz, right),
// (triangles under it, SAH cost, first sorted primitive under it, -), the integers as bits,
// so that a pass that visits a node has all of it from one or two cache lines.
__device__ __forceinline__ void ref_box(uint32_t r, const float4* __restrict__ saabb,
                                        const float4* bnode, float4& lo, float4& hi) {
    const float4* p = (r & kLeafBit) ? saabb + 2 * (size_t)(r & ~kLeafBit) : bnode + 3 * (size_t)r;
    lo = p[0];
    hi = p[1];
}

__device__ __forceinline__ float box_area(float4 lo, float4 hi) {
    float ex = hi.x - lo.x, ey = hi.y - lo.y, ez = hi.z - lo.z;
    return 2.0f * (ex * ez + ex * ey + ey * ez);
}

// SAH costs: an internal node costs kCi per unit of area plus its children; a leaf of
// c triangles costs kCt * c per unit of area.  Subtrees of <= leaf_size triangles are
// always collapsed into one leaf by the wide collapse, so they are priced as leaves.
constexpr float kCi = 1.2f;
constexpr float kCt = 1.0f;

__device__ __forceinline__ float sah_node_cost(float4 lo, float4 hi, uint32_t count, float cl, float cr,
                                               int leaf_size) {
    const float a = box_area(lo, hi);
    if (count <= (uint32_t)leaf_size) return kCt * a * (float)count;
    return kCi * a + cl + cr;
}

}  // namespace gpurt_impl
