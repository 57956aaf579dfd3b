// Q6_K weights as matrix operands.
#pragma once

#include "q4_matmul_mfma.h"

namespace mlc_hip {

// (0x6400 | v) is the half 1024 + v: two bytes -> half2 (v0 - 32, v1 - 32), exactly.
__device__ __forceinline__ q4_half2 q6_pair(uint32_t bytes, uint32_t sel) {
    const uint32_t m = __builtin_amdgcn_perm(0x64646464u, bytes, sel);
    const q4_half2 k1056 = {(_Float16)1056.0f, (_Float16)1056.0f};
    return __builtin_bit_cast(q4_half2, m) - k1056;
}

}  // namespace mlc_hip
