// Stores that go through the L2 to memory.
//
// A kernel ends with a write-back of the lines its stores left dirty in the L2s: other XCDs have no other way
// to see them.  Nothing else runs meanwhile.  Stores of device scope write through as they are made and leave nothing
// to write back.  That pays where a short kernel stores everything at its end, whole lines at a time: a prefill's
// partial sums (16 MB in a kernel of 16 us) 28.6 -> 26.9 us a call, 4 to 8 % of a call in the ranges of that path.
// The outputs of the Q4_0 matmuls of 32 requests: a step of 22 layers 1 217 -> 1 196 us, of one request 796 -> 794.
// It does not where a kernel stores all along and the L2 does its writing behind other work: the output of a long
// prefill 143 -> 154 us, of an 11264 x 2048 matmul over 512 tokens 80.6 -> 86.6; decode attention and row programs,
// whose outputs are small, did not change.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace mlc_hip {

// 2, 4 or 8 bytes
template <class T>
__device__ __forceinline__ void store_through(T* p, const T& v) {
    typedef std::conditional_t<sizeof(T) == 2, uint16_t, std::conditional_t<sizeof(T) == 4, uint32_t, uint64_t>> word;
    static_assert(sizeof(T) == sizeof(word), "2, 4 or 8 bytes");
    __hip_atomic_store(reinterpret_cast<word*>(p), __builtin_bit_cast(word, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// 16 bytes at base + offset bytes; base is the same for the whole wave
template <class T>
__device__ __forceinline__ void store_through16(void* base, uint32_t offset, const T& v) {
    static_assert(sizeof(T) == 16, "16 bytes");
    typedef uint32_t words __attribute__((ext_vector_type(4)));
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(base, 0, -1, 0x00027000);
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(words, v), rsrc, offset, 0, 16);   // (sc1: device scope)
}

}  // namespace mlc_hip
