// Sums and maxima over the lanes of a wave without LDS: a step is one or two vector instructions, where a shuffle is a
// trip through the LDS pipe of about 50 ns, and a wave that reduces has nothing else to do meanwhile.
#pragma once

#include "paged_decode_kernels.h"

namespace mlc_hip {

static constexpr int kDppRowRor4 = 0x124;   // row_ror:4: within 16 lanes whose values repeat after 8, i -> i^4

// What v = op(v, value of lane i ^ off) for off = 32, 16, ... down to LAST leaves, to the bit: the same lanes meet in
// the same order.
template <int LAST = 1, class Op>
__device__ __forceinline__ float wave_butterfly(float v, Op op) {
    static_assert(LAST == 1 || LAST == 4, "all lanes, or lanes that are equal modulo 4");
    v = across16(across32(v, op), op);
    v = op(v, dpp_f<kDppRowRor8>(v));
    v = op(v, dpp_f<kDppRowRor4>(v));
    if constexpr (LAST == 1) {
        v = op(v, dpp_f<kDppQuadXor2>(v));
        v = op(v, dpp_f<kDppQuadXor1>(v));
    }
    return v;
}
template <int LAST = 1>
__device__ __forceinline__ float wave_max_of(float v) {
    return wave_butterfly<LAST>(v, [](float a, float b) __attribute__((always_inline)) { return fmaxf(a, b); });
}
__device__ __forceinline__ float wave_sum_of(float v) {
    return wave_butterfly(v, [](float a, float b) __attribute__((always_inline)) { return a + b; });
}

}  // namespace mlc_hip
