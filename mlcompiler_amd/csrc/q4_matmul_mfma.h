// Batched Q4_0 matmul for gfx950: out[b][r] = sum_c W[r][c] * x[b][c], W in Q4_0 blocks
// (32 weights: fp16 scale d, 16 bytes of nibbles; weight j in the low nibble of byte j,
// weight j+16 in the high nibble, value d * (nibble - 8)), x and out fp32.
//
// Reference: MSL q4_0_matmul_v3_batched (compiler/runtime/metal_runtime.mm:710-785), one
// simdgroup per (4 rows, request), fp32 scalar arithmetic.  With a decode batch of up to 64
// requests this is a GEMM (M = rows, N = batch, K = cols) that should be bound by reading the
// weights once, so here it runs on the matrix cores (fp32 accumulate) with fp32-grade accuracy:
//   * an activation is split x*s = x_hi + x_lo (fp16 each, relative error 2^-22), s a power of
//     two per request that places the row's largest magnitude at 2^13..2^14;
//   * q4_matmul_kernel takes the integers q - 8 as operand, exact in fp16, and adds every block's sum
//     (q-8).x_hi + (q-8).x_lo to the result as d * sum: nothing is dropped.  There the activations may
//     also come with one power-of-two scale per (request, block of 32 columns) (BS), which a kernel
//     that produces 32 neighbouring columns of a request can compute on its own: the epilogues
//     (gate/up split + SiLU * up; residual add + RMSNorm) and the decode attention write the next
//     matmul's fragments that way;
//   * option q4_int_operand = 0 (q4_pairs_kernel): a weight d*(q-8) has at most 15 significant bits, so
//     it is EXACTLY w_hi + w_lo with w_hi = fp16(d*(q-8)) and w_lo = fma(d, q-8, -w_hi), and
//     out = (W_hi.X_hi + W_hi.X_lo + W_lo.X_hi) / s; the dropped W_lo.X_lo is below 2^-22 of the products.
// The weights are repacked once, on the device, when they enter the library's weight cache
// (q4_repack_kernel); the activations are split by a small kernel, or by whoever produces them, into
// matrix operand fragments, so that a fragment is one 16-byte load per lane.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "fragments.h"
#include "store_through.h"
#include "tagged_words.h"
#include "paged_decode_kernels.h"
#include "paged_rope_kernels.h"

namespace mlc_hip {

typedef _Float16 q4_half2 __attribute__((ext_vector_type(2)));
typedef _Float16 q4_half8 __attribute__((ext_vector_type(8)));
typedef float q4_float4 __attribute__((ext_vector_type(4)));
typedef float q4_float16 __attribute__((ext_vector_type(16)));

// ---- repacked weights: tiles of 16 rows, quads of 4 blocks (128 columns), for
// v_mfma_f32_16x16x32_f16, whose K is one block.
//   q  [rows/16][nquads][64 lanes] x 4 words: lane kg * 16 + row % 16, word b: the 8 weights kg*8 .. +7 of
//      block quad * 4 + b, weight e in nibble e / 2 + (e % 2) * 4 (q4_unpack)
//   d  [rows/16][nquads][16 rows] x 4 halves
// One 16-byte load brings a lane the weights of four blocks, 1 KB per wave in a row.  Blocks past the last one
// have scale 0.
struct Q4Args {
    const uint4* q;             // repacked weights (q4_repack_kernel)
    const uint2* d;
    const _Float16* xfrag;      // split activations (fragments.h)
    const float* inv_scale;     // [batch]
    const float* xrows;         // kQ4Rows: [batch][nblocks * 32], in place of the fragments
    float* out;                 // [batch][rows]; q4_pairs_kernel with K slices: the slice buffer [slices][batch][rows]
    uint32_t batch, rows, nblocks, nquads, quads_per_slice, slices;
    // slices > 1: where the workgroups of all slices but the last leave their sums for those of the last
    uint64_t* meet;             // [slices - 1][batch][rows] tagged words
    TagArgs tags;
    // The grid's x dimension: row groups (of RT tiles) times z groups of 16 requests, see q4_matmul_kernel.
    uint32_t row_groups, z_groups;
    // Kernels built with BS: the activations were split with one power-of-two scale per (request,
    // block of 32 columns) instead of one per request: x = (hi + lo) * scale.  The scales are
    // [batch tile of 32][nblocks][32 requests]; inv_scale is not read.
    const float* blk_scale;
    // SILU (slices == 1, rows = 2 * ffn_inner): the output is a fused gate/up row; row group j takes columns
    // 32 j .. 32 j + 31 of the gate half and of the up half and its epilogue also does the gate/up split and
    // SiLU(gate) * up -> gate, up, silu_out ([batch][ffn_inner] each).  With split_frag set it goes on
    // to split the 32 products of every request into the fragments of the matmul that consumes
    // them (K = ffn_inner), scaled per (request, block): block j of that matmul is exactly this
    // row group's 32 columns.
    uint32_t ffn_inner;
    float* gate;
    float* up;
    float* silu_out;
    _Float16* split_frag;
    float* split_blk_scale;
    // ADD (32 or 64 rows per workgroup): the epilogue also does the residual add that follows
    // the matmul (add_out = out + add_resid, [batch][rows]) and, with split_frag set, leaves every request's sum of squares over
    // every 32 columns in ssq_out[request][rows / 32] (the RMSNorm that follows is
    // finished by the matmul that reads it, see ssq_in) and writes add_out * add_gamma as the
    // split-fp16 fragments of that matmul (split_frag / split_blk_scale, K = rows).  add_gamma[c] for
    // c < add_n_gamma, 1 beyond.
    const float* add_resid;
    float* add_out;
    const float* add_gamma;
    uint32_t add_n_gamma;
    float* ssq_out;
    // ssq_in set (BS kernels): the activations are h * rms_gamma of an RMSNorm whose per-request factor
    // 1 / sqrt(mean(h^2) + eps) is still missing: it is computed here from the ssq_tiles partial
    // sums of squares per request (ssq_in[request][ssq_tiles], summed in a fixed order) and multiplied into
    // the result, and the workgroups also write the RMSNorm's own output rms_out = h * factor * rms_gamma
    // ([batch][rms_len], h = rms_src), every thread of the grid one element of its z group's requests.
    const float* ssq_in;
    uint32_t ssq_tiles, rms_len;
    float rms_eps;
    const float* rms_src;
    float* rms_out;
    const float* rms_gamma;     // as add_gamma
    uint32_t rms_n_gamma;
};
// ... and for the kernels built for ROPE (out is a fused qkv row of rope.qkv_rows = rows
// floats per request), whose epilogue also does what qkv_split_rope_cast_kernel would do with that row.
// (A type of its own: the launches without it need not carry its page rows.)
struct Q4RopeArgs : Q4Args {
    RopeArgs rope;
};
static constexpr uint32_t kQ4RopeOffset = (sizeof(Q4Args) + alignof(RopeArgs) - 1) / alignof(RopeArgs) * alignof(RopeArgs);
static_assert(sizeof(Q4RopeArgs) == kQ4RopeOffset + sizeof(RopeArgs), "where the kernel finds rope in its arguments");
static constexpr uint32_t kQ4LeadBytes = 5 * 8 + 4 * 4;   // arguments in front of them
static_assert(kQ4LeadBytes % alignof(Q4RopeArgs) == 0, "no padding behind them");

// Maximum / sum over the 32 lanes of a half wave, every lane gets the result.
__device__ __forceinline__ float q4_half_wave_max(float v) {
    v = fmaxf(v, dpp_f<kDppQuadXor1>(v));
    v = fmaxf(v, dpp_f<kDppQuadXor2>(v));
    v = fmaxf(v, dpp_f<kDppHalfMirror>(v));
    v = fmaxf(v, dpp_f<kDppRowRor8>(v));
    const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
}
__device__ __forceinline__ float q4_half_wave_sum(float v) {
    v += dpp_f<kDppQuadXor1>(v);
    v += dpp_f<kDppQuadXor2>(v);
    v += dpp_f<kDppHalfMirror>(v);
    v += dpp_f<kDppRowRor8>(v);
    const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
}

// One value per lane, the 32 lanes of a half wave holding columns col0 .. col0+31 (one Q4_0 block)
// of request b: writes them as hi + lo fp16 fragments of a matmul with K = k_cols, scaled by the
// block's own power of two, and the scale that undoes it (q4_split_activations_kernel's scale, per block).
__device__ __forceinline__ void q4_emit_block(float v, uint32_t b, uint32_t col, uint32_t k_cols, _Float16* frag,
                                              float* blk_scale, uint32_t width) {
    const float amax = q4_half_wave_max(fabsf(v));
    int e = 0;
    if (amax > 0.f && amax < INFINITY) (void)frexpf(amax, &e);
    int se = 14 - e;
    se = se > 100 ? 100 : (se < -100 ? -100 : se);
    const float tv = __builtin_ldexpf(v, se);
    const _Float16 hi = (_Float16)tv;
    const _Float16 lo = (_Float16)(tv - (float)hi);
    store_through(&frag[frag_piece(b, col / 8, 0, k_cols, width) + col % 8], hi);
    store_through(&frag[frag_piece(b, col / 8, 1, k_cols, width) + col % 8], lo);
    if (col % 32 == 0) store_through(&blk_scale[((size_t)(b / 32) * (k_cols / 32) + col / 32) * 32 + b % 32], __builtin_ldexpf(1.0f, -se));
}

// Two matmuls in one launch (q4_chain_kernel): what the first one's workgroups leave for the second one's, K columns of R
// requests, as tagged words (tagged_words.h).  First, for every quad of K (128 columns), in lines of its own (every workgroup's
// waves poll them: with all quads' scales side by side, in the memory of one or two channels, a word took 2 us to arrive):
//   [4][R]    a block's scale
//   [4][R]    ... and its sum of squares (of the RMSNorm in between)
//   [R][128]  {hi, lo} of an activation, the fragments of the second matmul
// and behind the quads [R][K], the values that the RMSNorm reads.
// All of it kQ4LinkCopies times, for the workgroups x % copies of the second matmul: a word that all of them poll in one place
// is late by as much as their loads take turns there.
struct Q4Link {
    uint64_t* words;
    TagArgs tags;
};
static constexpr uint32_t kQ4LinkCopies = 8;
__host__ __device__ __forceinline__ uint32_t q4_link_quad(uint32_t R) { return (R * 136 + 31) / 32 * 32; }
__host__ __device__ __forceinline__ size_t q4_link_sum(uint32_t K, uint32_t R) { return (size_t)((K + 127) / 128) * q4_link_quad(R); }
__host__ __device__ __forceinline__ size_t q4_link_words(uint32_t K, uint32_t R) { return q4_link_sum(K, R) + (size_t)K * R; }

// What q4_emit_block does, as those words.
__device__ __forceinline__ void q4_emit_words(float v, float sum, float ssq, uint32_t b, uint32_t col, uint32_t K, uint32_t R,
                                              uint64_t* words, uint32_t tag) {
    const float amax = q4_half_wave_max(fabsf(v));
    int e = 0;
    if (amax > 0.f && amax < INFINITY) (void)frexpf(amax, &e);
    int se = 14 - e;
    se = se > 100 ? 100 : (se < -100 ? -100 : se);
    const float tv = __builtin_ldexpf(v, se);
    const _Float16 hi = (_Float16)tv;
    const _Float16 lo = (_Float16)(tv - (float)hi);
    const uint64_t t = (uint64_t)tag << 32;
    uint64_t* const quad = words + (size_t)(col / 128) * q4_link_quad(R);
    st_tagged(quad + 8 * R + b * 128 + col % 128, t | __builtin_bit_cast(uint16_t, hi) | (uint32_t)__builtin_bit_cast(uint16_t, lo) << 16);
    if (col % 32 == 0) {
        const uint32_t blk = col / 32 % 4 * R + b;
        st_tagged(quad + blk, t | __float_as_uint(__builtin_ldexpf(1.0f, -se)));
        st_tagged(quad + 4 * R + blk, t | __float_as_uint(ssq));
    }
    st_tagged(words + q4_link_sum(K, R) + (size_t)b * K + col, t | __float_as_uint(sum));
}

// The split + RoPE + cast (+ paged write) of one element of a request's fused qkv row, by the
// thread that just produced it; the partner of its (even, odd) pair sits in the neighbouring
// lane.  Same arithmetic, element for element, as qkv_split_rope_cast_kernel.  What the thread
// needs from memory for it (its cos / sin pair, its request's page row) is fetched before the
// matmul's main loop, so that the epilogue adds no memory round trip to the kernel's tail.
struct Q4RopeFetch {
    float c, s;        // rotation of this element's pair (1, 0 where none applies)
    uint64_t page_row; // page_id * page_size + slot
};

__device__ __forceinline__ Q4RopeFetch q4_rope_prefetch(const RopeArgs& p, const uint64_t* page_rows, uint32_t req,
                                                         uint32_t feat) {
    Q4RopeFetch f = {1.0f, 0.0f, 0ull};
    if (req >= p.batch || feat >= p.q_rows + p.k_rows + p.v_rows) return f;
    const bool is_q = feat < p.q_rows;
    const bool is_k = !is_q && feat < p.q_rows + p.k_rows;
    const uint32_t local = is_q ? feat : (is_k ? feat - p.q_rows : feat - p.q_rows - p.k_rows);
    if (is_q || is_k) {
        const uint32_t d = (local & ~1u) % p.head_dim;
        if (d < p.rotary_dim) {
            const uint32_t ci = req * (p.rotary_dim / 2) + d / 2;
            f.c = p.cos_table[ci];
            f.s = p.sin_table[ci];
        }
    }
    if (!is_q && (is_k ? p.k_pages : p.v_pages)) f.page_row = page_rows[req];
    return f;
}

__device__ __forceinline__ void q4_rope_epilogue(const RopeArgs& p, const Q4RopeFetch& f, uint32_t req,
                                                 uint32_t feat, float val) {
    const float other = __shfl_xor(val, 1);
    const bool odd = (feat & 1u) != 0;
    const float2 x = odd ? make_float2(other, val) : make_float2(val, other);
    if (feat >= p.q_rows + p.k_rows + p.v_rows) return;
    const bool is_q = feat < p.q_rows;
    const bool is_k = !is_q && feat < p.q_rows + p.k_rows;
    const uint32_t local = is_q ? feat : (is_k ? feat - p.q_rows : feat - p.q_rows - p.k_rows);
    float2 y = x;
    if ((is_q || is_k) && (local & ~1u) % p.head_dim < p.rotary_dim) y = rope_rotate(x, f.c, f.s);
    const float mine = odd ? y.y : y.x;
    if (is_q) {
        store_through(&p.q[(size_t)req * p.q_rows + local], mine);
        return;
    }
    float* f32 = is_k ? p.k : p.v;
    const uint32_t rows = is_k ? p.k_rows : p.v_rows;
    if (f32) store_through(&f32[(size_t)req * rows + local], mine);
    const _Float16 h = (_Float16)mine;
    _Float16* f16 = is_k ? p.k_f16 : p.v_f16;
    if (f16) store_through(&f16[(size_t)req * rows + local], h);
    _Float16* pool = is_k ? p.k_pages : p.v_pages;
    if (pool) store_through(&pool[(size_t)f.page_row * rows + local], h);
}

typedef uint32_t q4_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t q4_u32x4 __attribute__((ext_vector_type(4)));

// A buffer descriptor of `bytes` bytes: loads behind its end return zero and move no data.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t q4_buffer(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00027000);
}

// 0x64006400 in a register the compiler does not see into: (w & mask) | ones is then one instruction (with two
// constants it takes two, an instruction of three operands having room for one).
__device__ __forceinline__ uint32_t q4_ones() {
    uint32_t ones = 0x64006400u;
    asm("" : "+v"(ones));
    return ones;
}
// The 8 weights of a word of the repacked layout as halves q - 8, exactly: (0x6400 | n) is the half
// 1024 + n, (0x6400 | n << 4) is 1024 + 16 n.  Nine instructions.
__device__ __forceinline__ q4_half8 q4_unpack(uint32_t w, uint32_t ones) {
    const q4_half2 k1032 = {(_Float16)1032.0f, (_Float16)1032.0f}, k72 = {(_Float16)72.0f, (_Float16)72.0f};
    const q4_half2 k16th = {(_Float16)0.0625f, (_Float16)0.0625f};
    const uint32_t v = w >> 8;
    const q4_half2 n0 = __builtin_bit_cast(q4_half2, (w & 0x000F000Fu) | ones) - k1032;
    const q4_half2 n1 = __builtin_elementwise_fma(__builtin_bit_cast(q4_half2, (w & 0x00F000F0u) | ones), k16th, -k72);
    const q4_half2 n2 = __builtin_bit_cast(q4_half2, (v & 0x000F000Fu) | ones) - k1032;
    const q4_half2 n3 = __builtin_elementwise_fma(__builtin_bit_cast(q4_half2, (v & 0x00F000F0u) | ones), k16th, -k72);
    return q4_half8{n0[0], n0[1], n1[0], n1[1], n2[0], n2[1], n3[0], n3[1]};
}

__device__ __forceinline__ float q4_silu_times(float g, float u) {  // walker_kernels.h: silu_times
    const float silu = g / (1.0f + expf(-g));
    return silu * u;
}

// What the epilogue of q4_matmul_kernel does besides storing the result.
// kQ4Rows: nothing; its activations come as rows of floats (xrows), which it splits itself.
enum Q4Form { kQ4Plain = 0, kQ4Silu = 1, kQ4Rope = 2, kQ4Add = 3, kQ4Rows = 4 };

// One workgroup of 16 (or 8) waves: RT tiles of 16 weight rows x up to 16 requests x one K slice.  The slice's
// quads of blocks are dealt out to the waves; a wave streams its quads' nibbles and scales (one quad ahead) and
// activation fragments (XD blocks ahead) straight from memory into registers, unpacks and multiplies; there is
// no staging memory and no barrier until the waves' sums meet in LDS at the end.
//
// The matrix product runs over the exact integers q - 8 and the block scale d is applied to each block's sum
// in fp32, acc += d * ((q-8).x_hi + (q-8).x_lo): per 16 rows and block two MFMAs, 9 instructions to unpack and
// one (with block scales two) per accumulator register.  The weights are the B operand (a lane holds weight
// row lane % 16, so d is one number per lane), the activations the A operand.  No product is rounded and no
// term is dropped: what remains is the fp32 rounding of the additions and of one multiply per block.
//
// These kernels are bound by the vector pipe of the CUs they run on as soon as the weights are there: one
// of them takes 1.7 us until its first loads are back, whatever it loads.  Hence 16 x 16 products:
// of a 32 x 32 product's 16 accumulator registers a batch of up to 16 requests uses half, and each costs
// one to three instructions per block.  NI: accumulator registers per product that are used: request r sits
// in row (r / NI) * 4 + r % NI of the A operand, so that 4 NI requests leave the registers NI .. 3 empty.
//
// More than 16 requests: z groups of 16, workgroups of their own that read the same weights at the same
// time on the same XCD (workgroup x: row group x / (8 Z) * 8 + x % 8, z group x / 8 % Z).  Each fetches its
// own activations only, 4 bytes per request and column through one CU's memory path, which would be the
// longest stream of a workgroup that had them all.  (NI = 1: the A operand has room for hi and lo of a request
// in different rows, and one product does for both; with NI = 2 that is no faster and spills.  2-norm error against float64, two
// products -> one: 0.95e-7 .. 1.07e-7 -> 0.85e-7 .. 0.98e-7.)  ZT = 2 or 4: so many groups in one
// workgroup, which unpacks a weight once for all of them.  That takes 158 or 245 registers, one workgroup of 8 waves to a
// CU, and so pays where such workgroups fill their rounds (launch_q4).
//
// Measured, kernel times in us, before (32 x 32 products, one workgroup per 32 rows, branches or clamps around the loads of
// a wave's last blocks) -> now.  One request of the 1 B shape: qkv (2560 x 2048) 7.0 -> 4.5, out-projection with the
// residual add 8.4 -> 4.6, gate/up with SiLU (11264 x 2048) 11.2 -> 7.0, down (2048 x 5632) 8.1 and 5.0 for the sum of
// its K slices -> 5.5 with the residual add, three slices that meet in here; a step of 22 layers 1 145 -> 801 (845 with the
// fragments of 32 requests as they are for larger batches; 670 with everything since but q4_chain_kernel, 609 with that).  32 requests: qkv 7.5 -> 6.9,
// gate/up 13.3 -> 13.3, a step 1 330 -> 1 199 (1 108).  16 requests of the 8 B shape: gate/up (28672 x 4096) 28.9 -> 23,
// a layer 140 -> 112 (106).  2-norm error against float64 of rows of 2048 to 14336: 0.95e-7 .. 1.17e-7, before 1.03e-7 .. 1.62e-7.
//
// The arguments that the first loads need come in front and as scalars: they are in registers when a wave starts (kernel
// argument preload, build.py), so that weights and activations are requested at once and what the epilogue reads, whose
// addresses take a fetch of the other arguments, behind them.  (From the argument segment, epilogue first -> now: steps of
// 22 layers of the 1 B shape 757 -> 740 us at one request, 1 160 -> 1 121 at 32, a layer of the 8 B shape at 16 109.2 -> 107.)
//
// LINK: the kernel is one of two matmuls in a launch (q4_chain_kernel): kQ4LinkOut, the first (residual add), leaves the
// second one's activations as tagged words, kQ4LinkIn, the second, takes them from there: at most QUADS quads per wave, whose
// weights are unpacked while the wave has to wait.
enum Q4LinkKind { kQ4LinkNone = 0, kQ4LinkOut = 1, kQ4LinkIn = 2 };

template <int NI, int RT, int WAVES, bool BS, int ZT>
struct Q4Lds {
    static constexpr bool PACKED = NI < 4;
    static constexpr int XQ = PACKED ? 2 * NI : 1, QR = 4 * NI * ZT;
    static constexpr int TILE_PITCH = NI * 64 + 16;         // floats per tile (16: bank spread)
    float red[WAVES * RT * ZT * TILE_PITCH];
    // BS: a quad's scales, [block][request]: fetched by a load of 4 bytes per lane, handed out from here.  (A load of
    // every lane's own scales per block would take as long as one of the block's two fragments: what bounds these
    // kernels next to the vector pipe is the 64 bytes a clock that a CU's loads return.)
    __attribute__((aligned(16))) float scales[BS ? WAVES : 1][ZT][64];
    q4_u32x4 packed[PACKED ? WAVES : 1][PACKED ? XQ * 64 : 1];
    float rms_scale[BS ? QR : 1];         // BS with ssq_in: every request's RMSNorm factor
};

template <int NI, int RT, int WAVES, bool BS, int FORM, int ZT = 1>
__global__ __launch_bounds__(WAVES * 64, ZT > 1 ? 2 : 4) void q4_matmul_kernel(
    const uint4* const w_q, const uint2* const w_d, const _Float16* const xfrag, const float* const blk_scale, const float* const ssq_in,
    const uint32_t nblocks, const uint32_t quads_per_slice, const uint32_t row_groups, const uint32_t batch_z,
    const std::conditional_t<FORM == kQ4Rope, Q4RopeArgs, Q4Args> a) {
    // (The body itself and LDS arrays of their own, not a call of q4_matmul_workgroup: behind one, given the arrays in a struct or as
    // pointers, the compiler takes 174 registers instead of 156 for gate/up at 32 requests, and the launch 12.74 us instead of 12.60.)
    constexpr int LINK = kQ4LinkNone, QUADS = 1;
    typedef Q4Lds<NI, RT, WAVES, BS, ZT> Lds;
    __shared__ decltype(Lds::red) red;
    __shared__ __attribute__((aligned(16))) decltype(Lds::scales) scales;
    __shared__ decltype(Lds::packed) packed;
    __shared__ decltype(Lds::rms_scale) rms_scale;
    const uint32_t block_x = blockIdx.x, slice = blockIdx.y, rope_args_offset = kQ4LeadBytes + kQ4RopeOffset;
    const Q4Link link{};
#include "q4_matmul_workgroup.h"
}

// ... and as one of two matmuls in a launch.
template <int NI, int RT, int WAVES, bool BS, int FORM, int ZT, int LINK, int QUADS, class Args>
__device__ __forceinline__ void q4_matmul_workgroup(
    Q4Lds<NI, RT, WAVES, BS, ZT>& lds, const uint32_t block_x, const uint32_t slice, const uint32_t rope_args_offset,
    const uint4* const w_q, const uint2* const w_d, const _Float16* const xfrag, const float* const blk_scale, const float* const ssq_in,
    const uint32_t nblocks, const uint32_t quads_per_slice, const uint32_t row_groups, const uint32_t batch_z, const Args& a,
    const Q4Link& link) {
    auto& red = lds.red;
    auto& scales = lds.scales;
    auto& packed = lds.packed;
    auto& rms_scale = lds.rms_scale;
#include "q4_matmul_workgroup.h"
}

// Two matmuls of up to 4 requests in one launch: one with the residual add that starts an RMSNorm, and the one that reads
// the norm.  The first matmul's workgroups come first, in all their K slices; the second one's request their weights, and then wait
// for the first one's sums as tagged words (tagged_words.h: why the waits end).  That takes a launch's start and end and the second
// one's way to its first weights off the chain of launches that a step is, and its unpacking, 0.7 us of the vector pipe per four
// row tiles: while it waits a wave holds its weights as halves in up to 64 registers.
//
// Measured: out-projection and gate/up of the 1 B shape at one request, in a kernel trace, 4.6 and 6.9 us and a launch's 2.3 in
// between, 9.1 in one launch; down-projection and qkv 6.2 and 4.0, 9.2.  From the start, by the time stamps of a probe build (out-projection
// and gate/up): the first one's weights back 1.5, its sums published 3.5 (vector pipe, 16 waves), seen 4.3, all words in LDS 4.9,
// products 5.9, waves' sums met 6.3, stored 7.4.  With one copy of the words, a quad's scales in the lines of all the others', they were
// seen at 5.5.  Steps of 22 layers and the lm_head, us, option q4_chain 0 -> 1, 600 cached tokens: 1, 2, 3, 4 requests 670, 678, 686, 695 ->
// 609, 638, 649, 668; a build for 5 and 8 requests 771, 778 -> 763, 784 (every workgroup fetches 8 bytes per request and column): two
// launches there.
template <int FORM>
struct Q4ChainArgs {
    Q4Args first;
    std::conditional_t<FORM == kQ4Rope, Q4RopeArgs, Q4Args> second;
    Q4Link link;
};
static_assert(sizeof(Q4Args) % alignof(Q4RopeArgs) == 0, "where q4_chain_kernel finds the second one's rope in its arguments");
template <int RT, int QUADS, int FORM>
__global__ __launch_bounds__(1024, 4) void q4_chain_kernel(
    const uint4* const w_q, const uint2* const w_d, const _Float16* const xfrag, const float* const blk_scale, const float* const ssq_in,
    const uint32_t nblocks, const uint32_t quads_per_slice, const uint32_t row_groups, const uint32_t batch_blocks, const Q4ChainArgs<FORM> c) {
    __shared__ union {
        Q4Lds<1, 2, 16, true, 1> first;
        Q4Lds<1, RT, 16, true, 1> second;
    } lds;
    const uint32_t batch_z = (batch_blocks & 0xFFFFu) | 1u << 16, blocks = batch_blocks >> 16;   // (of the first matmul)
    if (blockIdx.x < blocks) {
        const uint32_t per_slice = (row_groups + 7) / 8 * 8;
        uint32_t slice = 0, x = blockIdx.x;
        for (; x >= per_slice; x -= per_slice) ++slice;
        q4_matmul_workgroup<1, 2, 16, true, kQ4Add, 1, kQ4LinkOut, 0>(lds.first, x, slice, 0, w_q, w_d, xfrag, blk_scale, ssq_in, nblocks,
                                                                    quads_per_slice, row_groups, batch_z, c.first, c.link);
    } else {
        q4_matmul_workgroup<1, RT, 16, true, FORM, 1, kQ4LinkIn, QUADS>(
            lds.second, blockIdx.x - blocks, 0, kQ4LeadBytes + (uint32_t)sizeof(Q4Args) + kQ4RopeOffset, c.second.q, c.second.d,
            nullptr, nullptr, nullptr, c.second.nblocks, c.second.quads_per_slice, c.second.row_groups, batch_z, c.second, c.link);
    }
}

}  // namespace mlc_hip
