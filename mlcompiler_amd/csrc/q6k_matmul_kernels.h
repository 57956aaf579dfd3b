// Batched Q6_K matmul for gfx950 (the lm_head of the reference's batched decode step):
// out[b][r] = sum_c W[r][c] * x[b][c], W in Q6_K blocks of 256 weights (210 bytes: 128 bytes of
// low nibbles ql, 64 bytes of high bit pairs qh, 16 int8 scales of 16 weights each, fp16 d;
// value d * scale * (q - 32) with q in 0..63; compiler/runtime/quantization.cpp:142-147,
// 1469-1499), x and out fp32.
//
// Reference: MSL q6_k_matmul_v3_batched (compiler/runtime/metal_runtime.mm:1581-1655), one
// simdgroup per (4 rows, request), fp32 scalar arithmetic.  Here, like the Q4_0 matmul, the
// products run on the matrix cores with fp32-grade accuracy.  d * scale * (q - 32) has up to 24
// significant bits, too many for an fp16 pair, so the scale stays out of the matrix product:
// one MFMA k step covers exactly the 16 columns of one scale group, its operands are the
// exact small integers q - 32 (as fp16) and the activations split x * s = x_hi + x_lo (the
// same fragments as for Q4_0), and the group's sum S = (q-32).x_hi + (q-32).x_lo is added to
// the fp32 accumulator as (d * scale) * S.  The weights are the B operand (a lane holds weight
// row lane % 32), so d * scale is one number per lane, and the activations are the A operand.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "q6k_unpack.h"

namespace mlc_hip {

// ---- generic path: any rows / cols / stride, raw Q6_K rows.  One wave per (row, request),
// lanes stride over the columns like the reference kernel; fp32 throughout.
__global__ __launch_bounds__(256) void q6_k_matmul_generic_kernel(
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
        const uint32_t blk = c / 256, off = c % 256;
        const uint32_t half = off / 128, quarter = (off % 128) / 32, l = off % 32;
        const uint8_t* p = row + (size_t)blk * 210;
        const uint8_t qlb = p[half * 64 + (quarter & 1u) * 32 + l];
        const uint32_t nib = quarter < 2 ? (qlb & 0xFu) : (qlb >> 4);
        const uint32_t hb = (p[128 + half * 32 + l] >> (quarter * 2)) & 3u;
        const int q = (int)(nib | (hb << 4)) - 32;
        const float scale = (float)(int8_t)p[192 + half * 8 + quarter * 2 + l / 16];
        const uint16_t dbits = (uint16_t)(p[208] | (p[209] << 8));
        const float d = (float)__builtin_bit_cast(_Float16, dbits);
        acc += d * scale * (float)q * xv[c];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if (lane == 0) out[(size_t)b * rows + r] = acc;
}

// Repacked weights (made on the host when the matrix enters the weight cache).  A *group* is
// the four k steps (quarters 0-3) of one (block, half, l0) with l0 in {0, 16}: 64 weights of a
// row, packed in 24 bytes that a lane half h reads as three 8-byte pieces:
//   piece 0: ql[half*64 +      l0 + 8h .. +7]   (low nibble: quarter 0, high nibble: quarter 2)
//   piece 1: ql[half*64 + 32 + l0 + 8h .. +7]   (quarters 1 and 3)
//   piece 2: qh[half*32 +      l0 + 8h .. +7]   (bit pair 2*quarter)
//   qa    [rows/32][groups][3][64 lanes] x 8 bytes     groups = cols/256 * 4, lane = h*32 + row%32
//   sc    [rows/32][groups][32 rows] x 4 int8           the group's scale for quarters 0..3
//   d     [rows/32][cols/256][32 rows] fp16
// Group number within a row: block*4 + half*2 + l0/16; its k step for quarter q is
// block*16 + half*8 + q*2 + l0/16 (columns block*256 + half*128 + q*32 + l0 .. +15).
struct Q6KArgs {
    const uint2* qa;
    const uint32_t* sc;
    const _Float16* d;
    const _Float16* xfrag;   // split activations (fragments.h)
    const float* inv_scale;  // [batch]
    float* out;              // [batch][rows]
    uint32_t batch, rows, nblocks;
};

// One workgroup of 8 waves: RT tiles of 32 weight rows x NBT batch tiles of 32 x all of K; the waves deal the groups out
// among themselves (group wave, wave + 8, ...), stream pieces, scales and activation fragments into registers and add
// their sums up in LDS.  NA: accumulator registers per product that are used (4 hold requests 0 .. 7 of the
// batch tile, 8 0 .. 15, 16 all): each costs one instruction per product.
//
// The vector pipe does 15 + NA instructions per tile and k step beside two matrix products (about 6 us of a launch over
// 32000 x 2048 at 32 requests, 4 at one), the weights take 9 us: what counts is that the launch is one round of
// workgroups.  With two tiles per workgroup 32000 rows made 500 of them, and the registers left room for one on
// a CU.  Up to four tiles, whichever leaves the fewest tiles one after the other to a CU (launch_q6k_matmul); a
// group's activations then serve four tiles, and each k step's are fetched into the registers it has just read, one group
// ahead.  Whole calls, us, before -> now: 32000 x 2048 at 1, 16, 32 and 64 requests 34.6, 35.7, 38.1, 65.5 -> 28.7, 30.9, 34.2,
// 48.3 (the kernel at one and 32: 21.2 and 24.5 -> 15.7 and 20.9), 128256 x 2048 at one and 64 91, 207 -> 72, 141; 4096 x 4096 at
// 17 to 32 24 -> 23.
// Up to 16 requests one product does for hi and lo: 32000 x 2048 at 1 and 3 requests 29.1 -> 28.7, 2048 x 2048 at 1 to 16 19.9 -> 19.3, 4096 x
// 4096 22.8 -> 22.1.  2-norm error against float64 at 2048 and 4096 columns 1.10e-7, 1.31e-7 -> 1.07e-7, 1.29e-7.
template <int NBT, int RT, int NA>
__global__ __launch_bounds__(512, 2) void q6_k_matmul_mfma_kernel(const Q6KArgs a) {
    constexpr int WAVES = 8;
    __shared__ float red[WAVES * RT * NBT * NA * 64];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t lane = threadIdx.x % 64;
    const uint32_t l32 = lane % 32, half = lane / 32;
    const uint32_t tile0 = blockIdx.x * RT, tiles = min((uint32_t)RT, a.rows / 32 - tile0);
    const uint32_t groups = a.nblocks * 4;
    const uint32_t ksteps = a.nblocks * 16;
    // (lanes past the last request fetch that one's fragments again; their results are dropped)
    const uint32_t width = frag_width(a.batch);
    // (up to 16 requests: lo of a request sits 2 NA rows behind its hi, in the registers NA further, and one product does for both)
    constexpr bool BOTH = NA < 16;
    static_assert(!BOTH || NBT == 1, "one batch tile");
    constexpr int XP = BOTH ? 1 : 2;
    uint32_t lane_x[NBT];
#pragma unroll
    for (int t = 0; t < NBT; ++t)
        lane_x[t] = BOTH ? (half * width + min(l32 % (2 * NA), a.batch - 1u)) * 16 + min(l32 / (2 * NA), 1u) * 32 * width
                         : (half * width + min(l32, a.batch - 1u - t * 32)) * 16;

    float acc[RT][NBT][NA];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < NBT; ++t)
#pragma unroll
            for (int i = 0; i < NA; ++i) acc[r][t][i] = 0.f;

    // A descriptor per stream in scalar registers and 32 bits per lane.  What lies behind a row's last group reads as zero
    // and moves no data, and so does a tile behind the last one.
    __amdgpu_buffer_rsrc_t qa_desc[RT], sc_desc[RT], d_desc[RT], x_desc[NBT];
#pragma unroll
    for (uint32_t r = 0; r < RT; ++r) {
        const uint32_t real = r < tiles ? 1u : 0u;
        const size_t tile = tile0 + r * real;
        qa_desc[r] = q4_buffer(a.qa + tile * groups * 192, groups * 1536 * real);
        sc_desc[r] = q4_buffer(a.sc + tile * groups * 32, groups * 128 * real);
        d_desc[r] = q4_buffer(a.d + tile * a.nblocks * 32, a.nblocks * 64 * real);
    }
#pragma unroll
    for (int t = 0; t < NBT; ++t) x_desc[t] = q4_buffer(a.xfrag + (size_t)t * ksteps * 32 * width, ksteps * 64 * width);
    struct Weights {
        q4_u32x2 p[RT][3];
        uint32_t sc[RT];
        _Float16 d[RT];
    };
    auto load_w = [&](uint32_t g, Weights& k) __attribute__((always_inline)) {
        constexpr int NT = 2;   // (non-temporal: a weight is read once per launch and need not stay in the L2)
#pragma unroll
        for (int r = 0; r < RT; ++r) {
#pragma unroll
            for (int pc = 0; pc < 3; ++pc)
                k.p[r][pc] = __builtin_bit_cast(q4_u32x2, __builtin_amdgcn_raw_buffer_load_b64(qa_desc[r], g * 1536 + pc * 512 + lane * 8, 0, NT));
            k.sc[r] = __builtin_amdgcn_raw_buffer_load_b32(sc_desc[r], g * 128 + l32 * 4, 0, NT);
            k.d[r] = __builtin_bit_cast(_Float16, __builtin_amdgcn_raw_buffer_load_b16(d_desc[r], g / 4 * 64 + l32 * 2, 0, NT));
        }
        asm volatile("" ::: "memory");
    };
    q4_half8 x[NBT][4][XP];  // [batch tile][quarter][hi, lo]
    auto load_x = [&](uint32_t g, int q) __attribute__((always_inline)) {
        const uint32_t kstep = g / 4 * 16 + (g / 2) % 2 * 8 + q * 2 + g % 2;
#pragma unroll
        for (int t = 0; t < NBT; ++t)
#pragma unroll
            for (int pt = 0; pt < XP; ++pt)
                x[t][q][pt] = __builtin_bit_cast(q4_half8, __builtin_amdgcn_raw_buffer_load_b128(x_desc[t], (kstep * 2 + pt) * 32 * width + lane_x[t], 0, 0));
        asm volatile("" ::: "memory");
    };
    auto multiply = [&](const Weights& k, int q) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const q4_u32x2 ql = k.p[r][q & 1], qh = k.p[r][2];
            // one byte per weight: low nibble | high bit pair << 4
            const uint32_t v0 = ((q >= 2 ? ql.x >> 4 : ql.x) & 0x0F0F0F0Fu) | (((qh.x >> (2 * q)) & 0x03030303u) << 4);
            const uint32_t v1 = ((q >= 2 ? ql.y >> 4 : ql.y) & 0x0F0F0F0Fu) | (((qh.y >> (2 * q)) & 0x03030303u) << 4);
            const q4_half2 n0 = q6_pair(v0, 0x04010400u), n1 = q6_pair(v0, 0x04030402u);
            const q4_half2 n2 = q6_pair(v1, 0x04010400u), n3 = q6_pair(v1, 0x04030402u);
            const q4_half8 w = {n0[0], n0[1], n1[0], n1[1], n2[0], n2[1], n3[0], n3[1]};
            const int s8 = (int)(int8_t)(k.sc[r] >> (8 * q));
            const float gscale = (float)k.d[r] * (float)s8;
#pragma unroll
            for (int t = 0; t < NBT; ++t) {
                q4_float16 s;
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = 0.f;
                s = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[t][q][0], w, s, 0, 0, 0);
                if constexpr (!BOTH) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[t][q][XP - 1], w, s, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < NA; ++i) acc[r][t][i] = fmaf(gscale, BOTH ? s[i] + s[(i + NA) % 16] : s[i], acc[r][t][i]);
                // (here, and not further down, where the compiler would move it with all the products' registers)
#pragma unroll
                for (int i = 0; i < NA; ++i) asm volatile("" : "+v"(acc[r][t][i]));
            }
        }
    };
    // Two groups' weights in flight.  The last turn is a copy of the code without loads (see the Q4_0 kernel; the empty
    // asm statements pin every group of loads where it is written).
    Weights w, next;
    if (wave < groups) {
        load_w(wave, w);
#pragma unroll
        for (int q = 0; q < 4; ++q) load_x(wave, q);
        load_w(wave + WAVES, next);
        uint32_t g = wave;
        for (; g + WAVES < groups; g += WAVES) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                multiply(w, q);
                load_x(g + WAVES, q);
            }
            w = next;
            load_w(g + 2 * WAVES, next);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) multiply(w, q);
    }

    // ---- the waves' sums meet in LDS.  Accumulator layout: lane holds weight row l32 of the
    // tile and, in register i, batch row (i/4)*8 + (lane/32)*4 + i%4 of the batch tile.
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < NBT; ++t)
#pragma unroll
            for (int i = 0; i < NA; ++i) red[(((wave * RT + r) * NBT + t) * NA + i) * 64 + lane] = acc[r][t][i];
    __syncthreads();
    // wave w finishes the (r, t, i) combinations number w, w + 8, ...: 32 consecutive weight rows
    // of one request per half wave
    constexpr int COMBOS = RT * NBT * NA;
#pragma unroll
    for (int c = 0; c < (COMBOS + WAVES - 1) / WAVES; ++c) {
        const uint32_t combo = c * WAVES + wave;
        const uint32_t r = combo / (NBT * NA), t = (combo / NA) % NBT, i = combo % NA;
        const uint32_t b = t * 32 + (i / 4) * 8 + half * 4 + i % 4;
        if (r >= tiles || b >= a.batch) continue;
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) sum += red[(((w * RT + r) * NBT + t) * NA + i) * 64 + lane];
        store_through(&a.out[(size_t)b * a.rows + (tile0 + r) * 32 + l32], sum * a.inv_scale[b]);
    }
}

// As many tiles per workgroup as leave the fewest of them one after the other to a CU, the larger number where that is
// the same.
inline void launch_q6k_matmul(const Q6KArgs& a, size_t n_cu, hipStream_t stream) {
    const size_t tiles = a.rows / 32;
    const int most = a.batch > 32 ? 2 : 4;
    int rt = most;
    for (int r = most / 2; r >= 1; r /= 2) {
        auto cost = [&](size_t n) { return ((tiles + n - 1) / n + n_cu - 1) / n_cu * n; };
        if (cost((size_t)r) < cost((size_t)rt)) rt = r;
    }
    const dim3 grid((unsigned)((tiles + rt - 1) / rt));
#define MLC_Q6(NBT, RT, NA) hipLaunchKernelGGL((q6_k_matmul_mfma_kernel<NBT, RT, NA>), grid, dim3(512), 0, stream, a)
#define MLC_Q6_NA(RT) do { if (a.batch <= 8) MLC_Q6(1, RT, 4); else if (a.batch <= 16) MLC_Q6(1, RT, 8); else MLC_Q6(1, RT, 16); } while (0)
    if (a.batch > 32) {
        if (rt == 2) MLC_Q6(2, 2, 16);
        else MLC_Q6(2, 1, 16);
    } else if (rt == 4) {
        MLC_Q6_NA(4);
    } else if (rt == 2) {
        MLC_Q6_NA(2);
    } else {
        MLC_Q6_NA(1);
    }
#undef MLC_Q6_NA
#undef MLC_Q6
}

}  // namespace mlc_hip
