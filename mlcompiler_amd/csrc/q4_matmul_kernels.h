// The kernels around q4_matmul_kernel (q4_matmul_mfma.h): any-shape Q4_0 matmul, weight repacking, splitting of the
// activations, sum over K slices, and the kernel of option q4_int_operand = 0.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "q4_matmul_mfma.h"

namespace mlc_hip {

// ---- generic path: any rows / cols / stride, raw Q4_0 rows.  One wave per (row, request),
// lanes stride over the columns like the reference kernel; fp32 throughout.
__global__ __launch_bounds__(256) void q4_0_matmul_generic_kernel(
    const uint8_t* __restrict__ weights, const float* __restrict__ x, float* __restrict__ out,
    uint32_t batch, uint32_t rows, uint32_t cols, uint32_t row_stride) {
    const uint32_t wave = blockIdx.x * 4 + threadIdx.x / 64;
    const uint32_t lane = threadIdx.x % 64;
    if (wave >= batch * rows) return;
    const uint32_t b = wave / rows, r = wave - b * rows;
    const uint8_t* row = weights + (size_t)r * row_stride;
    const float* xv = x + (size_t)b * cols;
    float acc = 0.f;
    for (uint32_t c = lane; c < cols; c += 64) {
        const uint32_t blk = c / 32, in_blk = c % 32;
        const uint8_t* p = row + (size_t)blk * 18;
        const uint16_t dbits = (uint16_t)(p[0] | (p[1] << 8));  // rows may start at odd addresses
        const _Float16 d = __builtin_bit_cast(_Float16, dbits);
        const uint8_t byte = p[2 + (in_blk & 15)];
        const int q = (int)(in_blk < 16 ? (byte & 0x0F) : (byte >> 4)) - 8;
        acc += (float)d * (float)q * xv[c];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if (lane == 0) out[(size_t)b * rows + r] = acc;
}

// ---- activations -> operand fragments (fragments.h).  One workgroup per request row:
// s = 2^(14 - exponent(max|x|)).  Rows past `batch` of the last tile are not written here, and nobody reads them.
__global__ __launch_bounds__(256) void q4_split_activations_kernel(
    const float* __restrict__ x, _Float16* __restrict__ frag, float* __restrict__ inv_scale,
    uint32_t batch, uint32_t cols) {
    __shared__ float red[4];
    constexpr int MAXV = 4;  // register-resident groups of 8 columns per thread: cols <= 8192
    const uint32_t n = blockIdx.x;
    const uint32_t width = frag_width(batch);
    const uint32_t groups = cols / 8;
    const bool live = n < batch;
    const float4* xr = reinterpret_cast<const float4*>(x + (size_t)(live ? n : 0) * cols);
    const bool in_regs = groups <= 256 * MAXV;
    float4 v[MAXV][2];
    float amax = 0.f;
    if (live) {
        if (in_regs) {
#pragma unroll
            for (int j = 0; j < MAXV; ++j) {
                const uint32_t k8 = j * 256 + threadIdx.x;
                v[j][0] = v[j][1] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (k8 < groups) { v[j][0] = xr[k8 * 2]; v[j][1] = xr[k8 * 2 + 1]; }
                amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[j][0].x), fabsf(v[j][0].y)), fmaxf(fabsf(v[j][0].z), fabsf(v[j][0].w))));
                amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[j][1].x), fabsf(v[j][1].y)), fmaxf(fabsf(v[j][1].z), fabsf(v[j][1].w))));
            }
        } else {
            for (uint32_t k4 = threadIdx.x; k4 < cols / 4; k4 += 256) {
                const float4 t = xr[k4];
                amax = fmaxf(amax, fmaxf(fmaxf(fabsf(t.x), fabsf(t.y)), fmaxf(fabsf(t.z), fabsf(t.w))));
            }
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    int e = 0;
    if (amax > 0.f && amax < INFINITY) (void)frexpf(amax, &e);  // amax = m * 2^e, m in [0.5, 1)
    int se = 14 - e;
    se = se > 100 ? 100 : (se < -100 ? -100 : se);
    const float s = ldexpf(1.0f, se);
    if (threadIdx.x == 0 && live) inv_scale[n] = ldexpf(1.0f, -se);
    // 8 consecutive columns per thread and step: one 16-byte store to each part
    auto emit = [&](uint32_t k8, const float4& lo4, const float4& hi4) __attribute__((always_inline)) {
        const float in8[8] = {lo4.x, lo4.y, lo4.z, lo4.w, hi4.x, hi4.y, hi4.z, hi4.w};
        q4_half8 hi, lo;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float t = live ? in8[i] * s : 0.f;
            hi[i] = (_Float16)t;
            lo[i] = (_Float16)(t - (float)hi[i]);
        }
        *reinterpret_cast<q4_half8*>(frag + frag_piece(n, k8, 0, cols, width)) = hi;
        *reinterpret_cast<q4_half8*>(frag + frag_piece(n, k8, 1, cols, width)) = lo;
    };
    if (in_regs) {
#pragma unroll
        for (int j = 0; j < MAXV; ++j) {
            const uint32_t k8 = j * 256 + threadIdx.x;
            if (k8 < groups) emit(k8, v[j][0], v[j][1]);
        }
    } else {
        for (uint32_t k8 = threadIdx.x; k8 < groups; k8 += 256) {
            const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
            emit(k8, live ? xr[k8 * 2] : z, live ? xr[k8 * 2 + 1] : z);
        }
    }
}

// Raw Q4_0 rows -> the layout of q4_matmul_mfma.h, one thread per lane of a quad.
__global__ __launch_bounds__(256) void q4_repack_kernel(const uint8_t* __restrict__ raw, uint4* __restrict__ q,
                                                        uint16_t* __restrict__ d, uint32_t tiles, uint32_t nblocks,
                                                        uint32_t nquads, size_t row_stride) {
    const size_t unit = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (unit >= (size_t)tiles * nquads * 64) return;
    const uint32_t lane = (uint32_t)(unit % 64), quad = (uint32_t)(unit / 64 % nquads);
    const size_t tile = unit / 64 / nquads;
    const uint32_t row = lane % 16, kg = lane / 16;
    uint32_t w[4];
    for (uint32_t b = 0; b < 4; ++b) {
        const uint32_t blk = quad * 4 + b;
        const bool real = blk < nblocks;
        const uint8_t* p = raw + (tile * 16 + row) * row_stride + (size_t)(real ? blk : 0) * 18;
        w[b] = 0;
        for (uint32_t e = 0; e < 8; ++e) {
            const uint32_t byte = p[2 + (kg % 2) * 8 + e];
            w[b] |= (kg < 2 ? byte & 15u : byte >> 4) << (4 * (e / 2 + (e % 2) * 4));
        }
        if (kg == 0) d[((tile * nquads + quad) * 16 + row) * 4 + b] = real ? (uint16_t)(p[0] | (p[1] << 8)) : 0;
    }
    q[unit] = make_uint4(w[0], w[1], w[2], w[3]);
}

// Option q4_int_operand = 0: the weights as exact fp16 pairs d * (q - 8) = w_hi + w_lo, three products per block.
// One workgroup of 8 waves: 16 rows x 16 requests (grid y), all of K.
__global__ __launch_bounds__(512) void q4_pairs_kernel(const Q4Args a) {
    constexpr int WAVES = 8;
    __shared__ float red[WAVES * 4 * 64];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t lane = threadIdx.x % 64, l16 = lane % 16, kg = lane / 16;
    const uint32_t tile = blockIdx.x, req0 = blockIdx.y * 16, live = min(16u, a.batch - req0);
    const uint32_t width = frag_width(a.batch), req = req0 + min(l16, live - 1u);
    q4_float4 acc;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = 0.f;
    for (uint32_t blk = wave; blk < a.nblocks; blk += WAVES) {
        const size_t tq = (size_t)tile * a.nquads + blk / 4;
        const uint32_t word = reinterpret_cast<const uint32_t*>(a.q)[(tq * 64 + lane) * 4 + blk % 4];
        const _Float16 d = reinterpret_cast<const _Float16*>(a.d)[(tq * 16 + l16) * 4 + blk % 4];
        const q4_half8 n = q4_unpack(word, 0x64006400u), d8 = {d, d, d, d, d, d, d, d};
        const q4_half8 whi = d8 * n, wlo = __builtin_elementwise_fma(d8, n, -whi);
        const q4_half8 hi = *reinterpret_cast<const q4_half8*>(a.xfrag + frag_piece(req, blk * 4 + kg, 0, a.nblocks * 32, width));
        const q4_half8 lo = *reinterpret_cast<const q4_half8*>(a.xfrag + frag_piece(req, blk * 4 + kg, 1, a.nblocks * 32, width));
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, whi, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, whi, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, wlo, acc, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) red[(wave * 4 + i) * 64 + lane] = acc[i];
    __syncthreads();
    const uint32_t i = threadIdx.x / 64, q = kg * 4 + i;
    if (i >= 4 || q >= live) return;
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) sum += red[(w * 4 + i) * 64 + lane];
    a.out[(size_t)(req0 + q) * a.rows + tile * 16 + l16] = sum * a.inv_scale[req0 + q];
}

// out[i] = slice 0 + slice 1 + ... in that order, eight loads at a time: what this takes is the way to memory and back
// (whole calls, one load at a time -> now: 512 x 4096 at 300 tokens, 25 slices, 37.8 -> 35.6 us; 2048 x 2048 at 512, four,
// 43.9 -> 43.6).
__global__ __launch_bounds__(256) void q4_sum_slices_kernel(const float* __restrict__ slices,
                                                            float* __restrict__ out, uint32_t n,
                                                            uint32_t ksplit) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float s = slices[i];
    for (uint32_t k0 = 1; k0 < ksplit; k0 += 8) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = k0 + j < ksplit ? slices[(size_t)(k0 + j) * n + i] : 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (k0 + j < ksplit) s += v[j];
    }
    out[i] = s;
}

}  // namespace mlc_hip
