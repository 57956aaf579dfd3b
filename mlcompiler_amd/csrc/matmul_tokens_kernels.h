// Q4_0 and Q6_K matmul over many tokens (a prompt chunk, a batch of more than 64) for gfx950:
// out[t][r] = sum_c W[r][c] * x[t][c], all tokens in one launch.
//
// The arithmetic is that of the integer-operand kernels in q4_matmul_mfma.h and
// q6k_matmul_kernels.h: exact small integers times activations split into fp16 pairs on the matrix
// cores, every block's (Q4_0) or 16-column group's (Q6_K) sum multiplied with its scale in fp32.
// Those kernels take 64 requests at a time and stream everything through registers, which suits a
// decode batch, where the weights are the traffic.  A prompt chunk is bound by the matrix cores
// instead (two products per weight and token), so here
//   * a workgroup of 4 waves takes 64 tokens x 128 rows; a wave 64 tokens x 32 rows, two token tiles, so
//     that one unpacking of a weight serves two products;
//   * the four waves share the tokens' fragments through LDS, a stage of 64 columns (16 KB) at a time,
//     double buffered (from memory each wave would read 64 bytes a clock, all that a CU's L1 gives);
//   * weights go straight into registers, two stages ahead;
//   * while the matrix pipe works on one block's products, the vector pipe scales and adds the sums of the
//     block before (Q4_0 in the compiler's order: with its order prescribed, as for Q6_K, 70.2 us instead of 66.7 at
//     11264 x 2048 and 512 tokens);
//   * fp32 sums are kept in two levels (4 stages = 256 columns or more, then those sums), so that an
//     element is rounded no more often than in the waves' partial sums of the other kernels;
//   * workgroups of one XCD share row blocks and groups of 8 token blocks;
//   * what is left over by whole rounds of workgroups is split over K where it is a small part of a round
//     (tokens_tail): 4096 x 14336 at 1030 tokens 404 -> 317 us, 28672 x 4096 at 420 255 -> 235.
// Measured (whole synchronous calls, before -> after, us): Q4_0 11264 x 2048 at 128 tokens 51 -> 48, 512
// tokens 161 -> 81, 2047 tokens 609 -> 260; 2048 x 5632 at 512 tokens 171 -> 65; 2048 x 2048 at 2048 tokens
// 443 -> 66; Q6_K 32000 x 2048 at 700 tokens 584 -> 281, at 65 tokens 94 -> 72.  Of the 512-token call the
// kernel took 70 us (64 since) and the split 7 (before: 8 x (15.6 + 4.4)).  At 2047 tokens it did 777 TFLOP/s of fp16
// products, where a large library product reaches 1 180 on the same card at the same clock (2.1 GHz under
// this load): vector and matrix work together fill 80 % of the cycles.  Two row tiles per wave (half the
// LDS reads, 79 us at 512 tokens, 238 against 243 at 2047) and three smaller workgroups per CU without the
// overlap of blocks (64 us at 512, but 10 % behind on K = 14336 and on Q6_K) were measured as well.
// Vector instructions per Q4_0 block and wave 75 -> 59 (addresses through buffer descriptors, nine instead of 13 for an
// unpacked operand): 11264 x 2048 at 512 tokens 78.4 -> 75.8 us, at 2047 236.9 -> 228.6; 4096 x 14336 at 200 99.2 -> 95.2;
// Q6_K 32000 x 2048 at 65 and 700 61.1 -> 59.7 and 255.7 -> 252.  Not kept then: a fresh product in place of clearing the
// first-level sums, with a first level of 256 columns throughout (78 -> 81.6: another schedule); a higher priority for a wave
// in its products (Q6_K at 65 tokens 58.8 -> 57.1, at 700 256 -> 270); the split's stores through the L2 (57 instead of 56).
// Error against 64-bit products, 2-norm: 1.00e-7 to 1.4e-7 relative, before 1.03e-7 to 1.34e-7.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "matmul_tokens_args.h"
#include "q4_matmul_mfma.h"
#include "q6k_unpack.h"
#include "wave_reduce.h"

namespace mlc_hip {

// What q4_split_activations_kernel does (q4_matmul_kernels.h), four tokens per workgroup: neighbouring
// lanes hold neighbouring tokens, so that a store of 16 bytes per lane fills 64-byte pieces of the
// fragments instead of leaving every piece to another workgroup.  256 threads up to 4096 columns (64 per token), else
// 1024: there are few workgroups, and rows that do not fit the registers are read twice (whole calls of 2048 x 5632 at
// 512 tokens 62.5 -> 57.6 us, 4096 x 14336 at 200 tokens 106 -> 101; at 2048 columns both take 7 us).
template <int THREADS>
__global__ __launch_bounds__(THREADS) void tokens_split_kernel(const float* __restrict__ x, _Float16* __restrict__ frag,
                                                           float* __restrict__ inv_scale, uint32_t tokens, uint32_t cols) {
    constexpr int PER = THREADS / 4, WAVES = THREADS / 64;   // threads per token, waves
    constexpr int MAXV = THREADS == 256 ? 8 : 4;   // groups of 8 columns a thread keeps in registers: cols <= 4096 / 8192
    __shared__ float red[WAVES][4];
    const uint32_t n4 = threadIdx.x % 4, n = blockIdx.x * 4 + n4, g0 = threadIdx.x / 4;
    const uint32_t groups = cols / 8, ksteps = cols / 16;
    const bool live = n < tokens, in_regs = groups <= PER * MAXV;
    const float4* xr = reinterpret_cast<const float4*>(x + (size_t)(live ? n : 0) * cols);
    auto max8 = [](float m, const float4& a, const float4& b) __attribute__((always_inline)) {
        m = fmaxf(m, fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))));
        return fmaxf(m, fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fmaxf(fabsf(b.z), fabsf(b.w))));
    };
    float4 v[MAXV][2];
    float amax = 0.f;
    if (in_regs) {
#pragma unroll
        for (int j = 0; j < MAXV; ++j) {
            const uint32_t k8 = j * PER + g0;
            v[j][0] = v[j][1] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (live && k8 < groups) { v[j][0] = xr[k8 * 2]; v[j][1] = xr[k8 * 2 + 1]; }
        }
#pragma unroll
        for (int j = 0; j < MAXV; ++j) amax = max8(amax, v[j][0], v[j][1]);
    } else if (live) {
        for (uint32_t k8 = g0; k8 < groups; k8 += PER) amax = max8(amax, xr[k8 * 2], xr[k8 * 2 + 1]);
    }
    amax = wave_max_of<4>(amax);
    if (threadIdx.x % 64 < 4) red[threadIdx.x / 64][n4] = amax;
    __syncthreads();
    amax = red[0][n4];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) amax = fmaxf(amax, red[w][n4]);
    int e = 0;
    if (amax > 0.f && amax < INFINITY) (void)frexpf(amax, &e);  // amax = m * 2^e, m in [0.5, 1)
    int se = 14 - e;
    se = se > 100 ? 100 : (se < -100 ? -100 : se);
    const float s = ldexpf(1.0f, se);
    if (threadIdx.x < 4 && live) inv_scale[n] = ldexpf(1.0f, -se);
    auto emit = [&](uint32_t k8, const float4& a, const float4& b) __attribute__((always_inline)) {
        const float in8[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        q4_half8 hi, lo;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float t = live ? in8[i] * s : 0.f;
            hi[i] = (_Float16)t;
            lo[i] = (_Float16)(t - (float)hi[i]);
        }
        const size_t base = ((size_t)(n / 32) * ksteps + k8 / 2) * 2;
        const uint32_t lane = (k8 % 2) * 32 + n % 32;
        *reinterpret_cast<q4_half8*>(frag + ((base + 0) * 64 + lane) * 8) = hi;
        *reinterpret_cast<q4_half8*>(frag + ((base + 1) * 64 + lane) * 8) = lo;
    };
    if (in_regs) {
#pragma unroll
        for (int j = 0; j < MAXV; ++j)
            if (const uint32_t k8 = j * PER + g0; k8 < groups) emit(k8, v[j][0], v[j][1]);
    } else {
        for (uint32_t k8 = g0; k8 < groups; k8 += PER) emit(k8, xr[k8 * 2], xr[k8 * 2 + 1]);
    }
}

// One stage's weights of one row tile: 4 k steps of 16 columns.  What a tile holds is read through buffer
// descriptors: a lane's place in a stage is one register for good and the stage a scalar, where a 64-bit address costs
// vector instructions per load.
struct TokensQ4 {
    static constexpr int KSTEPS_PER_SCALE = 2, UNPACK = 0, VALU_PER_PRODUCT = 0;   // (the compiler's order)
    // (the layout is that of 16-row tiles and quads of blocks: a stage is half a quad, and k step s of its blocks
    // takes the column groups 2 s and 2 s + 1)
    struct Place {
        __amdgpu_buffer_rsrc_t q, d;
        uint32_t q_lane, d_lane;
        uint32_t ones;   // 0x64006400, in a vector register: with a literal, and + or are two instructions
        __device__ __forceinline__ Place(const TokensArgs& a, uint32_t tile, uint32_t lane) {
            const uint32_t nquads = (a.nblocks + 3) / 4, half = lane % 32 / 16;
            q = q4_buffer(a.q + (size_t)tile * 2 * nquads * 128, 2 * nquads * 1024);
            d = q4_buffer(a.d + (size_t)tile * 2 * nquads * 64, 2 * nquads * 128);
            q_lane = half * nquads * 1024 + (lane / 32 * 16 + lane % 16) * 16;
            d_lane = half * nquads * 128 + lane % 16 * 8;
            ones = 0x64006400u;
            asm volatile("" : "+v"(ones));
        }
    };
    uint2 q[2];     // [k step of a block]: a word per block
    q4_half2 d;     // a scale per block
    bool real;
    __device__ __forceinline__ void load(const TokensArgs& a, const Place& at, uint32_t stage, uint32_t end) {
        const uint32_t st = min(stage, a.stages - 1u);   // past the end: the last stage again, with scale 0
        real = stage < end;
#pragma unroll
        for (uint32_t s = 0; s < 2; ++s)
            q[s] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(at.q, at.q_lane + s * 512, st / 2 * 1024 + st % 2 * 8, 0));
        d = __builtin_bit_cast(q4_half2, __builtin_amdgcn_raw_buffer_load_b32(at.d, at.d_lane, st / 2 * 128 + st % 2 * 4, 0));
    }
    static __device__ __forceinline__ uint32_t kstep(const TokensArgs& a, uint32_t stage, uint32_t k) {
        return min(stage * 2 + k / 2, a.nblocks - 1u) * 2 + (k & 1u);
    }
    __device__ __forceinline__ q4_half8 operand(int k, const Place& at) const {
        return q4_unpack(k < 2 ? q[k & 1].x : q[k & 1].y, at.ones);
    }
    __device__ __forceinline__ float scale(int k) const { return real ? (float)d[k / 2] : 0.0f; }
};

struct TokensQ6 {   // a stage is one group (see Q6KArgs): k step = quarter
    static constexpr int KSTEPS_PER_SCALE = 1, UNPACK = 12, VALU_PER_PRODUCT = 10;
    struct Place {
        __amdgpu_buffer_rsrc_t q, sc, d;
        uint32_t lane;
        __device__ __forceinline__ Place(const TokensArgs& a, uint32_t tile, uint32_t l) : lane(l) {
            q = q4_buffer(a.q + (size_t)tile * a.stages * 192, a.stages * 1536);
            sc = q4_buffer(a.sc + (size_t)tile * a.stages * 32, a.stages * 128);
            d = q4_buffer(a.d + (size_t)tile * a.nblocks * 32, a.nblocks * 64);
        }
    };
    uint2 p[3];
    uint32_t s;
    _Float16 d;
    bool real;
    __device__ __forceinline__ void load(const TokensArgs& a, const Place& at, uint32_t stage, uint32_t end) {
        const uint32_t gi = min(stage, a.stages - 1u);
        real = stage < end;
#pragma unroll
        for (uint32_t i = 0; i < 3; ++i)
            p[i] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(at.q, at.lane * 8 + i * 512, gi * 1536, 0));
        s = __builtin_amdgcn_raw_buffer_load_b32(at.sc, at.lane % 32 * 4, gi * 128, 0);
        d = __builtin_bit_cast(_Float16, __builtin_amdgcn_raw_buffer_load_b16(at.d, at.lane % 32 * 2, gi / 4 * 64, 0));
    }
    static __device__ __forceinline__ uint32_t kstep(const TokensArgs& a, uint32_t stage, uint32_t k) {
        const uint32_t gi = min(stage, a.stages - 1u);
        return gi / 4 * 16 + (gi / 2) % 2 * 8 + k * 2 + gi % 2;
    }
    __device__ __forceinline__ q4_half8 operand(int k, const Place&) const {
        const uint2 ql = p[k & 1], qh = p[2];
        const uint32_t v0 = ((k >= 2 ? ql.x >> 4 : ql.x) & 0x0F0F0F0Fu) | (((qh.x >> (2 * k)) & 0x03030303u) << 4);
        const uint32_t v1 = ((k >= 2 ? ql.y >> 4 : ql.y) & 0x0F0F0F0Fu) | (((qh.y >> (2 * k)) & 0x03030303u) << 4);
        const q4_half2 n0 = q6_pair(v0, 0x04010400u), n1 = q6_pair(v0, 0x04030402u);
        const q4_half2 n2 = q6_pair(v1, 0x04010400u), n3 = q6_pair(v1, 0x04030402u);
        return q4_half8{n0[0], n0[1], n1[0], n1[1], n2[0], n2[1], n3[0], n3[1]};
    }
    __device__ __forceinline__ float scale(int k) const {
        return (real ? (float)d : 0.0f) * (float)(int)(int8_t)(s >> (8 * k));
    }
};

template <class W>
__global__ __launch_bounds__(256, 2) void matmul_tokens_kernel(const TokensArgs a) {
    constexpr int GROUP = 4;   // stages per turn of the main loop
    __shared__ q4_half8 xs[2][2][4][2][64];   // [buffer][token tile][k step][hi, lo][lane]
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t lane = threadIdx.x % 64;

    // workgroup -> (slice, group of 8 token blocks, row block, token block); XCD x (workgroups x,
    // x + 8, ...) takes a contiguous run of that order
    const bool tail = blockIdx.x >= a.whole;
    const uint32_t n = tail ? a.rest : a.whole, tail_slice = tail ? (blockIdx.x - a.whole) / a.rest : 0u;
    const uint32_t id = tail ? (blockIdx.x - a.whole) - tail_slice * a.rest : blockIdx.x;
    const uint32_t xcd = id % 8, per = n / 8, rem = n % 8;
    uint32_t t = xcd * per + min(xcd, rem) + id / 8;
    const uint32_t in_tail = t;
    const uint32_t per_k = a.token_blocks * a.row_blocks;
    const uint32_t slice = tail ? 0u : t / per_k;
    t = tail ? a.whole + t : t - slice * per_k;
    const uint32_t group = t / (8 * a.row_blocks);
    t -= group * 8 * a.row_blocks;
    const uint32_t in_group = min(8u, a.token_blocks - group * 8);
    const uint32_t token_block = group * 8 + t % in_group, row_block = t / in_group;

    const uint32_t tile = row_block * 4 + wave, tiles = a.rows / 32;
    const uint32_t tile_in = min(tile, tiles - 1u);   // (a tile past the end: the last one again, not stored)
    const uint32_t s0 = tail ? tail_slice * a.tail_stages : slice * a.stages_per_slice;
    const uint32_t s1 = min(s0 + (tail ? a.tail_stages : a.stages_per_slice), a.stages);

    q4_float16 acc[2], total[2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[x][e] = total[x][e] = 0.f;

    const typename W::Place at(a, tile_in, lane);
    const __amdgpu_buffer_rsrc_t x_desc = q4_buffer(a.xfrag + (size_t)token_block * 2 * a.ksteps * 1024, 2 * a.ksteps * 2048);
    // (the stage in the lane's offset: as a scalar offset Q6_K 32000 x 2048 at 700 tokens took 271 us instead of 256)
    q4_half8 st[2][2];   // this thread's part of the next stage: k step `wave`
    auto fetch_x = [&](uint32_t stage) __attribute__((always_inline)) {
        const uint32_t ks = W::kstep(a, stage, wave);
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int p = 0; p < 2; ++p)
                st[x][p] = __builtin_bit_cast(q4_half8, __builtin_amdgcn_raw_buffer_load_b128(
                    x_desc, lane * 16 + p * 1024 + (x * a.ksteps + ks) * 2048, 0, 0));
    };
    auto store_x = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int p = 0; p < 2; ++p) xs[buf][x][wave][p][lane] = st[x][p];
    };
    // LDS traffic of this wave done, then everybody's; loads from memory stay in flight
    auto barrier = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    W w[2];
    fetch_x(s0);
    w[0].load(a, at, s0, s1);
    w[1].load(a, at, s0 + 1, s1);
    asm volatile("" ::: "memory");   // (this and the ones below keep the loads where they are written)
    store_x(0);
    barrier();
    // A step is one scale's columns: its products go to s[step % 2], and while the matrix pipe works on
    // them the vector pipe scales and adds the step before.
    constexpr int KS = W::KSTEPS_PER_SCALE, STEPS = 4 / KS;
    uint32_t stage_group = 0;
    for (uint32_t base = s0; base < s1; base += GROUP, ++stage_group) {
        q4_float16 s[2][2];
        float sc[2];
        auto add = [&](int n) __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[x][e] = fmaf(sc[n], s[n][x][e], acc[x][e]);
        };
#pragma unroll
        for (int i = 0; i < GROUP; ++i) {
            // buffer i % 2 holds stage base + i; st the one after it, on its way
            fetch_x(base + i + 1);
            asm volatile("" ::: "memory");
#pragma unroll
            for (int step = 0; step < STEPS; ++step) {
                const int n = (i * STEPS + step) % 2;
                q4_half8 xa[KS][2][2], wk[KS];
#pragma unroll
                for (int k = 0; k < KS; ++k)
#pragma unroll
                    for (int p = 0; p < 2; ++p)
#pragma unroll
                        for (int x = 0; x < 2; ++x) xa[k][p][x] = xs[i % 2][x][step * KS + k][p][lane];
                sc[n] = w[i % 2].scale(step * KS);
#pragma unroll
                for (int k = 0; k < KS; ++k) wk[k] = w[i % 2].operand(step * KS + k, at);
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int e = 0; e < 16; ++e) s[n][x][e] = 0.f;
#pragma unroll
                for (int k = 0; k < KS; ++k)
#pragma unroll
                    for (int p = 0; p < 2; ++p)
#pragma unroll
                        for (int x = 0; x < 2; ++x)
                            s[n][x] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xa[k][p][x], wk[k], s[n][x], 0, 0, 0);
                if (i + step > 0) add(1 - n);
                // the scheduler's order: fragments, then the products with the vector work between them
                if constexpr (W::VALU_PER_PRODUCT > 0) {
                    __builtin_amdgcn_sched_group_barrier(0x100, 4 * KS, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, W::UNPACK, 0);
#pragma unroll
                    for (int m = 0; m < 4 * KS; ++m) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, W::VALU_PER_PRODUCT, 0);
                    }
                }
            }
            w[i % 2].load(a, at, base + i + 2, s1);
            asm volatile("" ::: "memory");
            store_x((i + 1) % 2);   // (last read before the barrier in front of this stage)
            barrier();
        }
        add((GROUP * STEPS - 1) % 2);
        if ((stage_group & a.flush_mask) == a.flush_mask || base + GROUP >= s1) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    total[x][e] += acc[x][e];
                    acc[x][e] = 0.f;
                }
        }
    }

    if (tile >= tiles) return;
    if (tail) {
        // (who waits for whom: tagged_words.h)
        const uint32_t tag = launch_tag(a.tags.tag, a.tags.tag_dev ? *a.tags.tag_dev : 0u);
        uint64_t* const mine = a.meet + (size_t)in_tail * 8192 + wave * 2048 + lane;
        if (tail_slice + 1 < a.tail_slices) {
            if (a.tags.test_flags & 1u) return;
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    st_tagged(mine + (size_t)tail_slice * a.rest * 8192 + (x * 16 + e) * 64, (uint64_t)tag << 32 | __float_as_uint(total[x][e]));
            return;
        }
        uint32_t spins = 0;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            float others[16] = {};
            for (uint32_t sl = 0; sl + 1 < a.tail_slices; ++sl) {
                const uint64_t* src = mine + (size_t)sl * a.rest * 8192 + x * 1024;
                uint64_t word[16];
                for (;;) {
                    bool ok = true;
#pragma unroll
                    for (int e = 0; e < 16; ++e) word[e] = ld_tagged(src + e * 64);
#pragma unroll
                    for (int e = 0; e < 16; ++e) ok = ok && (uint32_t)(word[e] >> 32) == tag;
                    if (__all(ok)) break;
                    if (++spins >= a.tags.spin_limit) {
                        if (!ok) report_fault(a.tags.fault);
                        break;
                    }
                }
#pragma unroll
                for (int e = 0; e < 16; ++e) others[e] += __uint_as_float((uint32_t)word[e]);
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) total[x][e] = others[e] + total[x][e];
        }
    }
    // lane: weight row lane % 32 of the tile; register e: token (e/4)*8 + (lane/32)*4 + e%4
    float* out = a.out + (size_t)slice * a.tokens * a.rows + tile * 32 + lane % 32;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const uint32_t token = token_block * 64 + x * 32 + (e / 4) * 8 + lane / 32 * 4 + e % 4;
            if (token < a.tokens) out[(size_t)token * a.rows] = total[x][e] * a.inv_scale[token];
        }
}

}  // namespace mlc_hip
