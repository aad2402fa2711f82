// index_math.h -- index arithmetic of the kernels at sizes that no test on a device reaches, and
// rules of launches, kept apart so that the host can run them over their whole range.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "../../include/gpurt.h"

namespace gpurt_impl {

// A 64-bit value from its halves as __builtin_amdgcn_readfirstlane returns them: ints, so
// each is made unsigned before it is widened (a low half from 2^31 would set every bit of
// the high one).
__host__ __device__ constexpr uint64_t u64_of_halves(int hi, int lo) {
    return (uint64_t)(uint32_t)hi << 32 | (uint32_t)lo;
}

// f(i) for i = first, first + step, ... below n.  The index is 64 bits wide: n may be any
// 32-bit count, and a 32-bit index within a step of 2^32 would wrap and never reach it.
template <typename F>
__host__ __device__ inline void grid_stride(uint32_t n, uint64_t first, uint64_t step, F f) {
    for (uint64_t i = first; i < n; i += step) f((uint32_t)i);
}

// The last m from lo on with off[m] <= key, for off[lo] <= key < off[n] and off[0..n] in
// ascending order (equal entries are empty): steps that double, then halve, so the cost is
// the logarithm of the distance.
template <typename Offsets>
__host__ __device__ inline uint32_t last_from(const Offsets& off, uint32_t n, uint32_t lo, uint64_t key) {
    uint32_t step = 1;
    while (step < n - lo && off[lo + step] <= key) {
        lo += step;
        step *= 2;
    }
    while (step > 1) {
        step /= 2;
        if (step < n - lo && off[lo + step] <= key) lo += step;
    }
    return lo;
}

// Vertex-gradient sums of a backward call: the fixed order (sort by vertex, then segmented sums)
// when the context asks for it, FP32 atomics when it asks for them, and otherwise whichever is
// faster -- the fixed order from about 0.6 M vertex terms, where the atomics' device-wide rate
// (~18 G/s) costs more than the sort's passes (points or rays on a 0.66 M vertex mesh, fixed
// order / atomics, us: 65 K queries 72 / 38, 131 K 82 / 69, 262 K 102 / 132, 524 K 150 / 252).
// Fewer vertices favour it more, though a run of many terms is added 64 at a time by one thread:
// 210 K queries on 6, 42, 642 and 10,242 vertices 590 / 12,100, 155 / 3,400, 100 / 370 and 98 /
// 131 (all on one vertex 1,070 / 13,900).  A call recorded into a HIP graph takes it from 2^21
// terms only: its scratch is a memory node of the graph then.
inline bool fixed_order_rule(int mode, size_t terms, bool recorded) {
    if (mode != GPURT_SUMS_AUTO) return mode == GPURT_SUMS_FIXED_ORDER;
    return terms >= (recorded ? size_t(1) << 21 : size_t(600000));
}

// Waves per CU of a set of n closest points: 16, but 12 for up to 256 points per CU (a
// quarter of 16 waves' lanes) on oriented nodes, where the time is the longest searches' and
// not the lanes'.  12 against 16, us: 65,536 points near 20,000 / 330,000 / 1.3 M triangles 99 /
// 106, 159 / 166, 182 / 194, on a soup of 100,000 triangles 119 / 121, on 20,000 overlapping
// ones 201 / 194; 131,072 on the overlapping ones 319 / 291, 200,000 near 20,000 triangles
// 160 / 125; on FP32 and 8-bit nodes, whose far queries take long, 65,536 uniform on 1.3 M
// 2,200 / 1,890 (FP32, W = 4).
inline int point_waves_per_cu(size_t n, int n_cu, bool oriented) {
    return oriented && n <= (size_t)n_cu * 256 ? 12 : 16;
}

// Wide levels of a W-wide tree over n triangles that get a launch each: what such trees have (5
// K triangles: 8 levels at W = 4, 2.3 M: 16; a level takes about log2(W) binary ones on the way
// down the larger side) and some.  The levels below are one block's, which is no slower for
// the few nodes that a small mesh has there; a large one's binary nodes, whose trees run 22 to
// 48 levels (58 with treelets), need more launches for that: a cluster of 1 M triangles in a
// scene of 64 takes 2,620 us with 22 launches and 570 us with 30; with treelets 7,620 us, with 42 1,370 us.
inline int collapse_launches(uint32_t n, int width, bool treelets) {
    int bits = 1;
    while (bits < 31 && (1u << bits) < n) bits++;
    const int per = width == 8 ? 5 : width == 4 ? 8 : n <= 65536 ? 10 : treelets ? 20 : 14;
    return 2 + bits * per / 10;
}

}  // namespace gpurt_impl
