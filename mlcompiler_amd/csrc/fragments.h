// Activations as matrix operand fragments: what every kernel that makes them and every kernel that reads them agrees on.
//
// Element (n, k) of a batch, x * s = hi + lo with hi = fp16(x * s), lo = fp16(x * s - hi), sits in
//   frag[(((n / 32 * (K / 16) + k / 16) * 2 + part) * 2 + k / 8 % 2) * width + n % 32][k % 8],  part 0 hi, 1 lo:
// pieces of 8 columns of one request, `width` requests next to each other.  The width is 32, so that a lane's
// operand is one 16-byte load and a wave's are whole 256-byte rows, and 4 or 8 for batches of up to 4 or 8 requests,
// which leaves no places between the requests that exist: a load brings a wave 1 KB of them.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mlc_hip {

__device__ __forceinline__ uint32_t frag_width(uint32_t batch) { return batch <= 4 ? 4u : batch <= 8 ? 8u : 32u; }

// Index in halves of a piece: request n, columns 8 * k8 .. 8 * k8 + 7.
__device__ __forceinline__ size_t frag_piece(uint32_t n, uint32_t k8, uint32_t part, uint32_t K, uint32_t width) {
    return (((((size_t)(n / 32) * (K / 16) + k8 / 2) * 2 + part) * 2 + k8 % 2) * width + n % 32) * 8;
}

}  // namespace mlc_hip
