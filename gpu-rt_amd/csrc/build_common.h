// build_common.h -- device helpers shared by the builder (build.hip) and the treelet
// restructuring (treelet.hip).
#pragma once

#include "gpurt_internal.h"

namespace gpurt_impl {

// per-mesh statistics: [cmin xyz, cmax xyz, max|coord|, unused] as ordered uints.
// k_prep accumulates into kRep replicas (wave w, of up to 1,024 triangles, uses replica
// w % kRep) so that the waves' atomics do not serialise on 7 addresses; k_reduce_stats folds
// them.
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

// ---- boxes of ranges of primitives ------------------------------------------------------
// rbox holds the boxes (lo, hi) of aligned blocks of 4, 16, 64, ... of N primitives, level
// after level (range_boxes(N) of them); a range of primitives is covered by at most 6
// blocks per level.  Minima and maxima are exact, so a union does not depend on its order.

// minimum and maximum as the hardware's instructions, without the quieting of signalling
// NaNs that fminf and fmaxf put before them (a third of k_orient's instructions; a NaN
// operand is dropped all the same)
__device__ __forceinline__ float vmin(float a, float b) {
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float vmax(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

__device__ __forceinline__ float4 min4(float4 a, float4 b) {
    return make_float4(vmin(a.x, b.x), vmin(a.y, b.y), vmin(a.z, b.z), 0.0f);
}
__device__ __forceinline__ float4 max4(float4 a, float4 b) {
    return make_float4(vmax(a.x, b.x), vmax(a.y, b.y), vmax(a.z, b.z), 0.0f);
}
__device__ __forceinline__ float4 shfl_xor4(float4 v, int o) {
    return make_float4(__shfl_xor(v.x, o), __shfl_xor(v.y, o), __shfl_xor(v.z, o), 0.0f);
}

// The blocks of 4, 16 and 64 primitives and the 256 of this block of threads, whose thread
// t has the box of primitive i = 256 blockIdx.x + t (past N: the empty box).  part: 8
// float4 in LDS.  All threads call it.
__device__ __forceinline__ void write_range_blocks(uint32_t N, uint32_t i, float4 lo, float4 hi, float4* __restrict__ rbox,
                                                   float4* part) {
    const uint32_t tid = threadIdx.x;
    float4* at = rbox;
    uint32_t cnt = N;
    for (int lvl = 1; lvl <= 3; lvl++) {
        const int o = 1 << (2 * (lvl - 1));
        lo = min4(lo, shfl_xor4(lo, o));
        hi = max4(hi, shfl_xor4(hi, o));
        lo = min4(lo, shfl_xor4(lo, 2 * o));
        hi = max4(hi, shfl_xor4(hi, 2 * o));
        cnt = (cnt + 3) / 4;
        const uint32_t e = i >> (2 * lvl);
        if ((tid & (4u * o - 1u)) == 0 && e < cnt) {
            at[2 * (size_t)e] = lo;
            at[2 * (size_t)e + 1] = hi;
        }
        at += 2 * (size_t)cnt;
    }
    if ((tid & 63u) == 0) {
        part[tid >> 6] = lo;
        part[4 + (tid >> 6)] = hi;
    }
    __syncthreads();
    if (tid == 0) {
        at[2 * (size_t)blockIdx.x] = min4(min4(part[0], part[1]), min4(part[2], part[3]));
        at[2 * (size_t)blockIdx.x + 1] = max4(max4(part[4], part[5]), max4(part[6], part[7]));
    }
    __syncthreads();
}

// Union of primitives [l, r) of N; leaf(k, lo, hi) adds primitive k's box.
template <typename Leaf>
__device__ __forceinline__ void range_union(uint32_t l, uint32_t r, uint32_t N, const float4* __restrict__ rbox, Leaf leaf,
                                            float4& lo, float4& hi) {
    lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f);
    hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    // what lies left and right of the whole blocks of 4, then the same a level up
    uint32_t l4 = min((l + 3u) & ~3u, r), r4 = max(r & ~3u, l4);
    for (uint32_t k = l; k < l4; k++) leaf(k, lo, hi);
    for (uint32_t k = r4; k < r; k++) leaf(k, lo, hi);
    const float4* at = rbox;
    uint32_t cnt = (N + 3) / 4;
    l = l4 / 4;
    r = r4 / 4;
    while (l < r) {
        l4 = min((l + 3u) & ~3u, r);
        r4 = max(r & ~3u, l4);
        for (uint32_t k = l; k < l4; k++) {
            lo = min4(lo, at[2 * (size_t)k]);
            hi = max4(hi, at[2 * (size_t)k + 1]);
        }
        for (uint32_t k = r4; k < r; k++) {
            lo = min4(lo, at[2 * (size_t)k]);
            hi = max4(hi, at[2 * (size_t)k + 1]);
        }
        at += 2 * (size_t)cnt;
        cnt = (cnt + 3) / 4;
        l = l4 / 4;
        r = r4 / 4;
    }
}

}  // namespace gpurt_impl
