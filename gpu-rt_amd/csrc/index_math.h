// index_math.h -- index arithmetic of the kernels at sizes that no test on a device reaches,
// kept apart so that the host can run it over their whole range.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

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

}  // namespace gpurt_impl
