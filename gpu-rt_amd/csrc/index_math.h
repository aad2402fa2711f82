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

}  // namespace gpurt_impl
