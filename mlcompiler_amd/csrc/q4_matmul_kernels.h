// The kernels around q4_matmul_kernel (q4_matmul_mfma.h): any-shape Q4_0 matmul, weight repacking, splitting of the
// activations, sum over K slices, and the kernel of option q4_int_operand = 0.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "q4_matmul_mfma.h"
#include "wave_reduce.h"

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
template <int THREADS>
__global__ __launch_bounds__(THREADS) void q4_split_activations_kernel(
    const float* __restrict__ x, _Float16* __restrict__ frag, float* __restrict__ inv_scale,
    uint32_t batch, uint32_t cols) {
    constexpr int WAVES = THREADS / 64;
    __shared__ float red[WAVES];
    constexpr int MAXV = 2;  // groups of 8 columns that a thread keeps in registers: cols <= 4096 / 16384
    const uint32_t n = blockIdx.x;
    const uint32_t width = frag_width(batch);
    const uint32_t groups = cols / 8;
    const bool live = n < batch;
    const float4* xr = reinterpret_cast<const float4*>(x + (size_t)(live ? n : 0) * cols);
    const bool in_regs = groups <= THREADS * MAXV;
    float4 v[MAXV][2];
    float amax = 0.f;
    if (live) {
        if (in_regs) {
#pragma unroll
            for (int j = 0; j < MAXV; ++j) {
                const uint32_t k8 = j * THREADS + threadIdx.x;
                v[j][0] = v[j][1] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (k8 < groups) { v[j][0] = xr[k8 * 2]; v[j][1] = xr[k8 * 2 + 1]; }
                amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[j][0].x), fabsf(v[j][0].y)), fmaxf(fabsf(v[j][0].z), fabsf(v[j][0].w))));
                amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[j][1].x), fabsf(v[j][1].y)), fmaxf(fabsf(v[j][1].z), fabsf(v[j][1].w))));
            }
        } else {
            for (uint32_t k4 = threadIdx.x; k4 < cols / 4; k4 += THREADS) {
                const float4 t = xr[k4];
                amax = fmaxf(amax, fmaxf(fmaxf(fabsf(t.x), fabsf(t.y)), fmaxf(fabsf(t.z), fabsf(t.w))));
            }
        }
    }
    amax = wave_max_of(amax);
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = amax;
    __syncthreads();
    amax = red[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) amax = fmaxf(amax, red[w]);
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
            const uint32_t k8 = j * THREADS + threadIdx.x;
            if (k8 < groups) emit(k8, v[j][0], v[j][1]);
        }
    } else {
        for (uint32_t k8 = threadIdx.x; k8 < groups; k8 += THREADS) {
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
// One workgroup of 16 waves: RT tiles of 16 rows x ZT groups of 16 requests (grid y) x one K slice (grid z); a wave takes
// every sixteenth quad of blocks.  A workgroup fetches 2 KB of activations per block and group beside a tile's 256 bytes of
// weights, and 17 instructions make a weight word an operand: four tiles where there are workgroups for it, and then two
// groups (8 waves: 132 registers) where those fill five eighths of the CUs.  (Whole calls, us, one tile and group, no quads ->
// now: 28672 x 4096 at 1, 32 and 64 requests 50, 89, 160 -> 35, 46, 76; 4096 x 14336 at 64 96 -> 56; 2048 x 2048 at 32
// 18.8 -> 17.2.)
template <int RT, int ZT, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void q4_pairs_kernel(const Q4Args a) {
    __shared__ float red[WAVES * RT * ZT * 4 * 64];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t lane = threadIdx.x % 64, l16 = lane % 16, kg = lane / 16;
    const uint32_t tile0 = blockIdx.x * RT, req0 = blockIdx.y * (16 * ZT), live = min(16u * ZT, a.batch - req0);
    const uint32_t width = frag_width(a.batch), cols = a.nblocks * 32;
    const uint32_t end = min((blockIdx.z + 1) * a.quads_per_slice, a.nquads);
    q4_float4 acc[RT][ZT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int z = 0; z < ZT; ++z)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[r][z][i] = 0.f;
    for (uint32_t quad = blockIdx.z * a.quads_per_slice + wave; quad < end; quad += WAVES) {
        uint4 word[RT];
        uint2 scale[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const size_t tq = (size_t)(tile0 + r) * a.nquads + quad;
            word[r] = a.q[tq * 64 + lane];
            scale[r] = a.d[tq * 16 + l16];
        }
        q4_half8 hi[4][ZT], lo[4][ZT];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {   // (a block that an incomplete quad lacks has scale 0: the last one again)
            const uint32_t blk = min(quad * 4 + j, a.nblocks - 1u);
#pragma unroll
            for (uint32_t z = 0; z < ZT; ++z) {
                const uint32_t req = req0 + min(z * 16 + l16, live - 1u);
                hi[j][z] = *reinterpret_cast<const q4_half8*>(a.xfrag + frag_piece(req, blk * 4 + kg, 0, cols, width));
                lo[j][z] = *reinterpret_cast<const q4_half8*>(a.xfrag + frag_piece(req, blk * 4 + kg, 1, cols, width));
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const uint32_t w = j == 0 ? word[r].x : j == 1 ? word[r].y : j == 2 ? word[r].z : word[r].w;
                const _Float16 d = __builtin_bit_cast(q4_half2, j < 2 ? scale[r].x : scale[r].y)[j % 2];
                const q4_half8 n = q4_unpack(w, 0x64006400u), d8 = {d, d, d, d, d, d, d, d};
                const q4_half8 whi = d8 * n, wlo = __builtin_elementwise_fma(d8, n, -whi);
#pragma unroll
                for (int z = 0; z < ZT; ++z) {
                    acc[r][z] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[j][z], whi, acc[r][z], 0, 0, 0);
                    acc[r][z] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[j][z], whi, acc[r][z], 0, 0, 0);
                    acc[r][z] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[j][z], wlo, acc[r][z], 0, 0, 0);
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int z = 0; z < ZT; ++z)
#pragma unroll
            for (int i = 0; i < 4; ++i) red[(((wave * RT + r) * ZT + z) * 4 + i) * 64 + lane] = acc[r][z][i];
    __syncthreads();
    for (uint32_t o = threadIdx.x; o < RT * ZT * 256; o += WAVES * 64) {
        const uint32_t r = o / (ZT * 256), z = o / 256 % ZT, i = o / 64 % 4, q = z * 16 + kg * 4 + i;
        if (q >= live) continue;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) sum += red[(((w * RT + r) * ZT + z) * 4 + i) * 64 + lane];
        a.out[((size_t)blockIdx.z * a.batch + req0 + q) * a.rows + (tile0 + r) * 16 + l16] = sum * a.inv_scale[req0 + q];
    }
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
