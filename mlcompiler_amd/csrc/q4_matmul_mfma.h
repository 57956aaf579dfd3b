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
// fragments of 32 requests as they are for larger batches; 703 with everything since).  32 requests: qkv 7.5 -> 6.9,
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

template <int NI, int RT, int WAVES, bool BS, int FORM, int ZT, int LINK, int QUADS, class Args>
__device__ __forceinline__ void q4_matmul_workgroup(
    Q4Lds<NI, RT, WAVES, BS, ZT>& lds, const uint32_t block_x, const uint32_t slice, const uint32_t rope_args_offset,
    const uint4* const w_q, const uint2* const w_d, const _Float16* const xfrag, const float* const blk_scale, const float* const ssq_in,
    const uint32_t nblocks, const uint32_t quads_per_slice, const uint32_t row_groups, const uint32_t batch_z, const Args& a,
    const Q4Link& link) {
    constexpr bool LINKED = LINK == kQ4LinkIn;
    static_assert(LINK == kQ4LinkNone || (NI == 1 && WAVES == 16 && BS && ZT == 1), "two matmuls in a launch: up to 4 requests");
    static_assert(LINK != kQ4LinkOut || FORM == kQ4Add, "the first of two: with the residual add");
    constexpr bool ROWS_IN = FORM == kQ4Rows;
    static_assert(!ROWS_IN || (NI < 4 && BS), "rows of floats: up to 8 requests, split by block");
    static_assert(FORM != kQ4Silu || RT == 4, "SiLU epilogue: 32 rows of gate and 32 of up");
    static_assert(FORM != kQ4Add || RT % 2 == 0, "residual add: whole blocks of the next matmul's K");
    // Up to 8 requests: a quad's activations come 1 KB per load, without the places of requests that do not
    // exist, and each lane's operand from LDS.  (16-byte loads of 64 lanes cost 16 clocks of the return path, however
    // many of them ask for the same bytes or for none.)
    constexpr bool PACKED = NI < 4, BOTH = NI == 1;
    constexpr uint32_t WIDTH = PACKED ? 4 * NI : 32;
    constexpr int XQ = PACKED ? 2 * NI : 1;          // loads per quad
    // blocks of activations in registers: as far as 128 registers per wave go
    constexpr int XD = PACKED ? (RT == 4 ? 1 : 2) : RT == 4 ? 2 : 4;
    static_assert(ZT == 1 || (RT == 4 && WAVES == 8 && !PACKED), "more than one group of 16 requests: one workgroup of 8 waves to a CU");
    constexpr int X_TILES = (ZT + 1) / 2;            // batch tiles of 32 that the workgroup has a part of
    constexpr int QR = 4 * NI * ZT;                       // requests of the workgroup
    constexpr int TILE_PITCH = Q4Lds<NI, RT, WAVES, BS, ZT>::TILE_PITCH;
    auto& red = lds.red;
    auto& scales = lds.scales;
    auto& packed = lds.packed;
    auto& rms_scale = lds.rms_scale;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t lane = threadIdx.x % 64, l16 = lane % 16, kg = lane / 16;
    const uint32_t batch = batch_z & 0xFFFFu, z_groups = batch_z >> 16, nquads = (nblocks + 3) / 4;
    const uint32_t z8 = 8 * z_groups;
    const uint32_t row_group = block_x / z8 * 8 + block_x % 8, zg = block_x / 8 % z_groups;
    if (row_group >= row_groups) return;           // (the grid is a multiple of 8 row groups)
    const uint32_t req0 = zg * (16 * ZT), live = min((uint32_t)QR, batch - req0);   // (the last group may be smaller)
    // tile r of the workgroup
    const uint32_t tile0 = FORM == kQ4Silu ? row_group * 2 : row_group * RT;
    auto tile_of = [&](int r) __attribute__((always_inline)) {
        return FORM == kQ4Silu && r >= 2 ? row_groups * 2 + tile0 + (uint32_t)r - 2u : tile0 + (uint32_t)r;
    };

    // ---- thread -> output: row `row` of the workgroup's (SiLU: column of its 32), request req0 + q
    constexpr uint32_t ROWS = FORM == kQ4Silu ? 32 : 16 * RT, PER_PASS = WAVES * 64 / ROWS;
    constexpr int PASSES = (QR + PER_PASS - 1) / PER_PASS;   // outputs per thread
    const uint32_t row = threadIdx.x % ROWS, qi = threadIdx.x / ROWS;
    // (which request: so that the 64 lanes of a wave read 64 different banks)
    constexpr uint32_t SB = 2 * NI;
    const uint32_t q_any = ROWS == 16   ? (qi % 4) * NI + qi / 4
                           : ROWS == 32 ? (qi & ~(1u | SB)) | ((qi & 1u) ? SB : 0u) | ((qi & SB) ? 1u : 0u)
                                        : qi;
    // (kQ4LinkOut: the threads that would have nothing to do leave the other matmul copies of its words)
    static_assert(LINK != kQ4LinkOut || (ROWS == 32 && PASSES == 1 && PER_PASS / QR == kQ4LinkCopies), "a thread per word and copy");
    const uint32_t q = LINK == kQ4LinkOut ? q_any % QR : q_any, copy = LINK == kQ4LinkOut ? q_any / QR : 0u;
    const bool has_out = (LINK == kQ4LinkOut || qi < QR) && q < live;
    const uint32_t b = req0 + q, col = tile0 * 16 + row;

    // ---- main loop
    struct QuadW {
        q4_u32x4 q[RT];
        q4_u32x2 d[RT];
        float sc[ZT];   // BS: the scale of request l16 in block kg of the quad
        q4_u32x4 x[XQ];   // PACKED: the quad's activations
    };
    struct BlockX {
        q4_half8 hi[ZT], lo[ZT];   // (BOTH: hi[0] has both)
    };
    // Everything is fetched with buffer loads: a descriptor per stream in scalar registers and 32 bits per lane.  Their
    // descriptors end where the data does; what lies behind (the last blocks of an incomplete quad, the weights
    // behind a wave's last quad) reads as zero.
    const uint32_t first = slice * quads_per_slice + wave, end = min((slice + 1) * quads_per_slice, nquads);
    __amdgpu_buffer_rsrc_t q_desc[RT], d_desc[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const size_t tile = (size_t)tile_of(r) * nquads;
        q_desc[r] = q4_buffer(w_q + tile * 64, end * 1024);
        d_desc[r] = q4_buffer(w_d + tile * 16, end * 128);
    }
    __amdgpu_buffer_rsrc_t x_desc[X_TILES];
#pragma unroll
    for (int t = 0; t < X_TILES; ++t)
        x_desc[t] = ROWS_IN ? q4_buffer(xfrag, batch * nblocks * 128) : q4_buffer(xfrag + (size_t)(req0 / 32 + t) * nblocks * 2048, nblocks * WIDTH * 128);
    const __amdgpu_buffer_rsrc_t s_desc = q4_buffer(BS ? blk_scale + (size_t)(req0 / 32) * nblocks * 32 : nullptr, nblocks * 128);
    // (request of this lane's row of the A operand; rows without one repeat another's.  Four groups: more than 48 requests,
    // so that the third and the fourth group's are in the second batch tile)
    uint32_t x_lane[ZT];   // (two 16-column steps, hi and lo of each)
    if constexpr (PACKED) {
        // BOTH: hi of request r in row r * 4 and lo in the next one, so that one product has both
        const uint32_t m = l16 % 4, xreq = min(l16 / 4 * NI + (BOTH ? 0u : min(m, (uint32_t)NI - 1u)), live - 1u);
        x_lane[0] = (kg / 2 * 4 * WIDTH + kg % 2 * WIDTH + (BOTH ? min(m, 1u) * 2 * WIDTH : 0u) + xreq) * 16;
    }
#pragma unroll
    for (int z = 0; z < (PACKED ? 0 : ZT); ++z) {
        const uint32_t xreq = min(l16 / 4 * NI + min(l16 % 4, (uint32_t)NI - 1u) + z * 16, live - 1u) + req0 % 32 - z / 2 * 32;
        x_lane[z] = (kg / 2 * 4 * WIDTH + kg % 2 * WIDTH + xreq) * 16;
    }
    const uint32_t s_lane = kg * 128 + (req0 % 32 + l16) * 4;
    auto load_w = [&](uint32_t quad, QuadW& k) __attribute__((always_inline)) {
        constexpr int NT = 2;   // (non-temporal: a weight is read once per launch and need not stay in the L2)
        if constexpr (BS && !LINKED && !ROWS_IN) {
#pragma unroll
            for (int z = 0; z < ZT; ++z)
                k.sc[z] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(s_desc, quad * 512 + s_lane + z * 64, 0, 0));
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            k.q[r] = __builtin_bit_cast(q4_u32x4, __builtin_amdgcn_raw_buffer_load_b128(q_desc[r], quad * 1024 + lane * 16, 0, NT));
            k.d[r] = __builtin_bit_cast(q4_u32x2, __builtin_amdgcn_raw_buffer_load_b64(d_desc[r], quad * 128 + l16 * 8, 0, NT));
        }
        if constexpr (ROWS_IN) {
            // (two requests per register quad, two columns of each; a lane behind the last column fetches the first ones, and drops them)
            const uint32_t at = quad * 512 + lane * 8;
#pragma unroll
            for (int n = 0; n < QR; ++n) {
                const q4_u32x2 v = __builtin_bit_cast(q4_u32x2, __builtin_amdgcn_raw_buffer_load_b64(
                    x_desc[0], min((uint32_t)n, live - 1u) * (nblocks * 128) + (at < nblocks * 128 ? at : 0u), 0, 0));
                k.x[n / 2][n % 2 * 2] = v[0];
                k.x[n / 2][n % 2 * 2 + 1] = v[1];
            }
        } else if constexpr (PACKED && !LINKED) {
#pragma unroll
            for (int i = 0; i < XQ; ++i)
                k.x[i] = __builtin_bit_cast(q4_u32x4, __builtin_amdgcn_raw_buffer_load_b128(x_desc[0], quad * (XQ * 1024) + i * 1024 + lane * 16, 0, 0));
        }
        asm volatile("" ::: "memory");
    };
    auto load_x = [&](uint32_t blk, BlockX& k) __attribute__((always_inline)) {
        if constexpr (PACKED) return;
#pragma unroll
        for (int z = 0; z < ZT; ++z) {
            k.hi[z] = __builtin_bit_cast(q4_half8, __builtin_amdgcn_raw_buffer_load_b128(x_desc[z / 2], blk * 4096 + x_lane[z], 0, 0));
            k.lo[z] = __builtin_bit_cast(q4_half8, __builtin_amdgcn_raw_buffer_load_b128(x_desc[z / 2], blk * 4096 + x_lane[z] + 1024, 0, 0));
        }
        asm volatile("" ::: "memory");
    };
    // The other matmul's words of a quad (LINKED), into the places of LDS that loaded ones would go to.  A word of
    // every block first: few loads while there is nothing to be had.
    [[maybe_unused]] uint32_t link_tag = 0, link_spins = 0;
    [[maybe_unused]] const uint64_t* const link_words =
        LINKED ? link.words + block_x % kQ4LinkCopies * q4_link_words(nblocks * 32, batch) : nullptr;
    [[maybe_unused]] auto link_wait = [&](auto get) __attribute__((always_inline)) {
        while (!__all(get())) {
            if (++link_spins >= link.tags.spin_limit) {
                if (lane == 0) report_fault(link.tags.fault);
                break;
            }
        }
    };
    [[maybe_unused]] auto receive = [&](uint32_t quad) __attribute__((always_inline)) {
        const bool has_cols = quad * 128 + lane * 2 < nblocks * 32, has_scale = l16 < live && quad * 4 + kg < nblocks;
        const uint64_t* const words = link_words + (size_t)quad * q4_link_quad(batch);
        const uint64_t none = (uint64_t)link_tag << 32;
        uint64_t sc = none;
        link_wait([&]() __attribute__((always_inline)) {
            if (has_scale) sc = ld_tagged(words + kg * batch + l16);
            return (uint32_t)(sc >> 32) == link_tag;
        });
        scales[wave][0][lane] = __uint_as_float((uint32_t)sc);
        uint32_t* const to = reinterpret_cast<uint32_t*>(packed[wave]);
        const uint32_t piece = lane / 8 * 4 * WIDTH + lane / 4 % 2 * WIDTH;   // (columns 2 * lane and the next one: k step lane / 8)
        const uint64_t* const frag = words + 8 * batch + lane * 2;
        uint64_t wd[4][2];
#pragma unroll
        for (uint32_t n = 0; n < 4; ++n) wd[n][0] = wd[n][1] = none;
        link_wait([&]() __attribute__((always_inline)) {
            bool ok = true;
#pragma unroll
            for (uint32_t n = 0; n < 4; ++n)
                if (n < live && has_cols) {
                    wd[n][0] = ld_tagged(frag + n * 128);
                    wd[n][1] = ld_tagged(frag + n * 128 + 1);
                }
#pragma unroll
            for (uint32_t n = 0; n < 4; ++n) ok = ok && (uint32_t)(wd[n][0] >> 32) == link_tag && (uint32_t)(wd[n][1] >> 32) == link_tag;
            return ok;
        });
#pragma unroll
        for (uint32_t n = 0; n < 4; ++n) {
            if (n >= live) break;
            const uint32_t w0 = (uint32_t)wd[n][0], w1 = (uint32_t)wd[n][1];
            to[(piece + n) * 4 + lane % 4] = (w0 & 0xFFFFu) | w1 << 16;
            to[(piece + 2 * WIDTH + n) * 4 + lane % 4] = w0 >> 16 | (w1 & 0xFFFF0000u);
        }
        asm volatile("" ::: "memory");
    };
    // A quad's rows of floats (ROWS_IN) into the places of LDS that its fragments would go to: a block is 16 lanes, one power of two
    // for it as in q4_emit_block.
    [[maybe_unused]] auto split_rows = [&](uint32_t quad, const QuadW& k) __attribute__((always_inline)) {
        const bool has_cols = quad * 128 + lane * 2 < nblocks * 32;
        uint32_t* const to = reinterpret_cast<uint32_t*>(packed[wave]);
        const uint32_t piece = lane / 8 * 4 * WIDTH + lane / 4 % 2 * WIDTH;   // (columns 2 * lane and the next one: k step lane / 8)
#pragma unroll
        for (int n = 0; n < QR; ++n) {
            if ((uint32_t)n >= live) break;
            const float x0 = has_cols ? __uint_as_float(k.x[n / 2][n % 2 * 2]) : 0.f, x1 = has_cols ? __uint_as_float(k.x[n / 2][n % 2 * 2 + 1]) : 0.f;
            float amax = fmaxf(fabsf(x0), fabsf(x1));
            amax = fmaxf(amax, dpp_f<kDppQuadXor1>(amax));
            amax = fmaxf(amax, dpp_f<kDppQuadXor2>(amax));
            amax = fmaxf(amax, dpp_f<kDppHalfMirror>(amax));
            amax = fmaxf(amax, dpp_f<kDppRowRor8>(amax));
            const int e = amax < INFINITY ? __builtin_amdgcn_frexp_expf(amax) : 0;   // (0 where amax is)
            int se = 14 - e;
            se = se > 100 ? 100 : (se < -100 ? -100 : se);
            const float t0 = __builtin_ldexpf(x0, se), t1 = __builtin_ldexpf(x1, se);
            const q4_half2 hi = {(_Float16)t0, (_Float16)t1}, lo = {(_Float16)(t0 - (float)hi[0]), (_Float16)(t1 - (float)hi[1])};
            to[(piece + n) * 4 + lane % 4] = __builtin_bit_cast(uint32_t, hi);
            to[(piece + 2 * WIDTH + n) * 4 + lane % 4] = __builtin_bit_cast(uint32_t, lo);
            if (l16 == 0) scales[wave][0][kg * 16 + n] = __builtin_ldexpf(1.0f, -se);
        }
        asm volatile("" ::: "memory");
    };
    auto read_x = [&](int j, BlockX& k) __attribute__((always_inline)) {
        const uint32_t piece = j * 8 * WIDTH + x_lane[0] / 16;
        k.hi[0] = __builtin_bit_cast(q4_half8, packed[wave][piece]);
        if constexpr (!BOTH) k.lo[0] = __builtin_bit_cast(q4_half8, packed[wave][piece + 2 * WIDTH]);
        asm volatile("" ::: "memory");
    };
    const uint32_t ones = q4_ones();
    q4_float4 zero;
#pragma unroll
    for (int i = 0; i < 4; ++i) zero[i] = 0.f;
    float acc[RT][ZT][NI] = {};
    // (wk_of: weights that have been unpacked already)
    auto multiply = [&](const QuadW& w, int j, const BlockX& x, auto wk_of) __attribute__((always_inline)) {
        // (the scales of this lane's requests in block j, see `turn`)
        [[maybe_unused]] float sc[ZT][NI];
        if constexpr (BS) {
#pragma unroll
            for (int z = 0; z < ZT; ++z)
#pragma unroll
                for (int i = 0; i < NI; ++i) sc[z][i] = scales[wave][z][j * 16 + kg * NI + i];
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const q4_half2 dd = __builtin_bit_cast(q4_half2, (uint32_t)w.d[r][j / 2]);
            const float d = (float)dd[j % 2];
            const q4_half8 wk = wk_of(r);
#pragma unroll
            for (int z = 0; z < ZT; ++z) {
                q4_float4 s = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.hi[z], wk, zero, 0, 0, 0);
                if constexpr (!BOTH) s = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.lo[z], wk, s, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < NI; ++i)
                    acc[r][z][i] = fmaf(BS ? d * sc[z][i] : d, BOTH ? s[i] + s[(i + NI) % 4] : s[i], acc[r][z][i]);
                // (here, and not further down, where the compiler would move it: a quad's products do not fit
                // the 128 registers a wave has)
#pragma unroll
                for (int i = 0; i < NI; ++i) asm volatile("" : "+v"(acc[r][z][i]));
            }
        }
        if constexpr (PACKED && RT == 4 && (WAVES == 16 || !BS)) __builtin_amdgcn_sched_barrier(0);   // (for the same reason)
    };
    // Rounding errors grow with the number of blocks added up in a row: a quad's sums go to a second set of registers
    // where there is room for one, else those of four quads (of two where 8 waves share K: as many blocks of 4096 columns
    // as 16 waves add up) to LDS, where the waves' sums meet anyway.  (2-norm error against float64, with one level -> now:
    // 9216 x 14336 at 17 requests 1.58e-7 -> 1.11e-7, 512 x 11008 at 33 1.22e-7 -> 1.07e-7, 28672 x 4096 at 17 1.10e-7 ->
    // 1.02e-7.  It takes 0.5 to 0.8 % of a layer of 4096 columns at up to 16 requests; adding to LDS after every quad with
    // ds_add costs 1.3 to 5 times the kernel.)
    constexpr bool TWO_LEVELS = RT * NI * ZT <= 8;
    [[maybe_unused]] float total[RT][ZT][NI] = {};
    [[maybe_unused]] uint32_t in_a_row = 0;
    [[maybe_unused]] bool flushed = false;
    auto each = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int z = 0; z < ZT; ++z)
#pragma unroll
                for (int i = 0; i < NI; ++i) f(red[((wave * RT + r) * ZT + z) * TILE_PITCH + i * 64 + lane], total[r][z][i], acc[r][z][i]);
    };
    auto flush = [&]() __attribute__((always_inline)) {
        if constexpr (TWO_LEVELS) each([](float&, float& sum, float& v) __attribute__((always_inline)) { sum += v; });
        else if (flushed) each([](float& sum, float&, float& v) __attribute__((always_inline)) { sum += v; });
        else each([](float& sum, float&, float& v) __attribute__((always_inline)) { sum = v; });
        each([](float&, float&, float& v) __attribute__((always_inline)) { v = 0.f; });
        flushed = true;
    };
    // A wave's quads are first, first + WAVES, ...  While one is multiplied the next one's weights are on the way, and
    // activations XD blocks ahead.  The last one is a copy of the code that fetches nothing: a load costs its share
    // of the return path even where it reads nothing, and behind a branch around loads the compiler waits as if
    // they had not been issued, and so for all of them.  (The empty asm statements pin every group of
    // loads where it is written: without them they move down to just before their use.)
    QuadW w, next;
    BlockX x[XD];
    auto turn = [&](uint32_t quad, auto more) __attribute__((always_inline)) {
        if constexpr (ROWS_IN) {
            split_rows(quad, w);
        } else if constexpr (BS) {   // (a wave's own: LDS operations of a wave are in order)
#pragma unroll
            for (int z = 0; z < ZT; ++z) scales[wave][z][lane] = w.sc[z];
        }
        if constexpr (PACKED) {
            if constexpr (!ROWS_IN) {
#pragma unroll
                for (int i = 0; i < XQ; ++i) packed[wave][i * 64 + lane] = w.x[i];
            }
            if constexpr (XD > 1) read_x(0, x[0]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if constexpr (PACKED)
                if (j + XD - 1 < 4) read_x(j + XD - 1, x[(j + XD - 1) % XD]);
            multiply(w, j, x[j % XD], [&](int r) __attribute__((always_inline)) { return q4_unpack(w.q[r][j], ones); });
            if (j + XD < 4) load_x(quad * 4 + j + XD, x[j % XD]);
            else if constexpr (decltype(more)::value) load_x((quad + WAVES) * 4 + j + XD - 4, x[j % XD]);
        }
    };
    QuadW link_w[LINKED ? QUADS : 1];
    if constexpr (LINKED) {
#pragma unroll
        for (int n = 0; n < QUADS; ++n) load_w(first + n * WAVES, link_w[n]);
    } else if (first < end) {
        load_w(first, w);
#pragma unroll
        for (int i = 0; i < XD; ++i) load_x(first * 4 + i, x[i]);
        if (first + WAVES < end) load_w(first + WAVES, next);
    }
    // ---- what the epilogue reads besides the sums is fetched before the main loop, so that it adds no memory
    // round trip to the kernel's tail
    [[maybe_unused]] Q4RopeFetch rope_pre[PASSES];
    [[maybe_unused]] float resid_pre[PASSES] = {}, gamma_pre = 1.0f, inv_pre[PASSES] = {};
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        const uint32_t bp = b + p * PER_PASS;
        const bool has = has_out && q + p * PER_PASS < live;
        if constexpr (FORM == kQ4Rope) {
            rope_pre[p] = {1.0f, 0.0f, 0ull};
            if (has) rope_pre[p] = q4_rope_prefetch(a.rope, rope_page_rows(a.rope, rope_args_offset), bp, col);
        }
        if constexpr (FORM == kQ4Add)
            if (has) resid_pre[p] = a.add_resid[(size_t)bp * a.rows + col];
        if constexpr (!BS)
            if (has) inv_pre[p] = a.inv_scale[bp];
    }
    if constexpr (FORM == kQ4Add)
        if (col < a.add_n_gamma) gamma_pre = a.add_gamma[col];
    // The RMSNorm that the producer of the activations left unfinished (ssq_in): a wave sums up the partials of
    // one or two requests, and the row group writes 1024 elements of the norm's own output at the end.
    constexpr int RMS_N = 16 * ZT / WAVES;   // requests per wave, and elements per thread
    constexpr int SSQ_NL = 2;           // partials per lane: up to 128 tiles, rows of 4096 (the host checks)
    [[maybe_unused]] float ssq_part[RMS_N][SSQ_NL] = {}, rms_h[RMS_N] = {}, rms_gamma[RMS_N];
    const uint32_t rms_el = row_group * (1024 * ZT) + threadIdx.x;
    if constexpr (BS) {
        if (LINKED || ssq_in) {
#pragma unroll
            for (int n = 0; n < RMS_N; ++n) {
                const uint32_t sq = wave + n * WAVES, el = rms_el + n * WAVES * 64;
#pragma unroll
                for (int j = 0; j < SSQ_NL; ++j) {
                    const uint32_t tl = lane + j * 64;
                    if (!LINKED && sq < live && tl < a.ssq_tiles) ssq_part[n][j] = ssq_in[(size_t)(req0 + sq) * a.ssq_tiles + tl];
                }
                rms_gamma[n] = 1.0f;
                if (el < live * a.rms_len) {
                    const uint32_t rc = el % a.rms_len;
                    if constexpr (!LINKED) rms_h[n] = a.rms_src[(size_t)req0 * a.rms_len + el];
                    if (rc < a.rms_n_gamma) rms_gamma[n] = a.rms_gamma[rc];
                }
            }
        }
    }
    uint32_t tag_add = 0;   // (K slices of a captured pass)
    if constexpr (LINK == kQ4LinkNone) {
        if (a.slices > 1 && a.tags.tag_dev) tag_add = *a.tags.tag_dev;
    } else {
        if (link.tags.tag_dev) tag_add = *link.tags.tag_dev;   // (of the same pass: a.tags has none or the same)
        link_tag = launch_tag(link.tags.tag, tag_add);
    }
    asm volatile("" ::: "memory");

    auto finish_rms = [&]() __attribute__((always_inline)) {
        if (LINKED || ssq_in) {
#pragma unroll
            for (int m = 0; m < RMS_N; ++m) {
                float part = q4_half_wave_sum(ssq_part[m][0] + ssq_part[m][1]);
                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(part), __float_as_uint(part), false, false);
                part = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
                const uint32_t sq = wave + m * WAVES;
                if (lane == 0 && sq < live) rms_scale[sq] = 1.0f / sqrtf(part / (float)a.rms_len + a.rms_eps);
            }
        }
    };
    [[maybe_unused]] uint64_t ssq_word[SSQ_NL];
    [[maybe_unused]] auto get_ssq = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < SSQ_NL; ++j) {
            const uint32_t tl = lane + j * 64;
            ssq_word[j] = (uint64_t)link_tag << 32;
            if (tl < nblocks) ssq_word[j] = ld_tagged(link_words + (size_t)(tl / 4) * q4_link_quad(batch) + (4 + tl % 4) * batch + wave);
        }
    };
    if constexpr (BS && !LINKED) finish_rms();
    if constexpr (LINKED) {
        static_assert(TWO_LEVELS && RT * QUADS <= 4, "a wave's weights unpacked: at most 64 registers");
        q4_half8 wk[QUADS][RT][4];
#pragma unroll
        for (int n = 0; n < QUADS; ++n)
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    wk[n][r][j] = q4_unpack(link_w[n].q[r][j], ones);
                    asm volatile("" : "+v"(wk[n][r][j]));   // (now, and not where they are used)
                }
#pragma unroll
        for (int n = 0; n < QUADS; ++n) {
            const uint32_t quad = first + n * WAVES;
            if (quad >= end) break;
            receive(quad);
            if (n == 0 && wave < live) get_ssq();   // (on their way during the products)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                read_x(j, x[0]);
                multiply(link_w[n], j, x[0], [&](int r) __attribute__((always_inline)) { return wk[n][r][j]; });
            }
            if (n + 1 < QUADS) flush();
        }
    } else if (first < end) {
        uint32_t quad = first;
        for (; quad + WAVES < end; quad += WAVES) {
            turn(quad, std::true_type());
            // (not before this point: the copy waits for the loads)
#pragma unroll
            for (int r = 0; r < RT; ++r) asm volatile("" : "+v"(next.q[r]), "+v"(next.d[r]));
            w = next;
            load_w(quad + 2 * WAVES, next);
            // (behind the loads: a branch in front of them makes the compiler wait for more of them)
            if constexpr (TWO_LEVELS) {
                flush();
            } else if (++in_a_row == WAVES / 4) {
                flush();
                in_a_row = 0;
            }
        }
        turn(quad, std::false_type());
    }

    [[maybe_unused]] uint64_t rms_word = 0;
    [[maybe_unused]] const uint64_t* rms_at = nullptr;   // this thread's element of the norm, if it has one
    if constexpr (LINKED) {
        // the other matmul's sums of squares: wave n adds up request n's
        static_assert(RMS_N == 1, "one element of the norm per thread");
        if (wave < live) {
            if (first >= end) get_ssq();
            bool again = false;
            link_wait([&]() __attribute__((always_inline)) {
                if (again) get_ssq();
                again = true;
                bool ok = true;
#pragma unroll
                for (int j = 0; j < SSQ_NL; ++j) ok = ok && (uint32_t)(ssq_word[j] >> 32) == link_tag;
                return ok;
            });
#pragma unroll
            for (int j = 0; j < SSQ_NL; ++j) ssq_part[0][j] = __uint_as_float((uint32_t)ssq_word[j]);
        }
        if (rms_el < live * a.rms_len) {
            rms_at = link_words + q4_link_sum(a.rms_len, batch) + rms_el;
            rms_word = ld_tagged(rms_at);
        }
        finish_rms();
    }

    // ---- the waves' sums meet in LDS.  A lane holds weight row l16 of the tile and, in register i, request
    // kg * NI + i.
    flush();
    if constexpr (TWO_LEVELS) each([](float& sum, float& v, float&) __attribute__((always_inline)) { sum = v; });
    __syncthreads();
    if constexpr (BS) {
        // the norm's own output: h * factor * gamma, the arithmetic of rms_norm_batched_kernel
        if constexpr (LINKED) {
            link_wait([&]() __attribute__((always_inline)) {
                if (rms_at && (uint32_t)(rms_word >> 32) != link_tag) rms_word = ld_tagged(rms_at);
                return !rms_at || (uint32_t)(rms_word >> 32) == link_tag;
            });
            rms_h[0] = __uint_as_float((uint32_t)rms_word);
        }
        if (LINKED || ssq_in) {
#pragma unroll
            for (int m = 0; m < RMS_N; ++m) {
                const uint32_t el = rms_el + m * WAVES * 64;
                if (el < live * a.rms_len)
                    store_through(&a.rms_out[(size_t)req0 * a.rms_len + el], rms_h[m] * rms_scale[el / a.rms_len] * rms_gamma[m]);
            }
        }
    }
    if (!has_out) return;   // (whole half waves where the epilogue works across lanes: 32 rows share q)
    auto sum_of = [&](uint32_t tile_row, uint32_t sq, float inv) __attribute__((always_inline)) {
        const uint32_t s16 = sq % (4 * NI);
        const float* p = red + (tile_row / 16 * ZT + sq / (4 * NI)) * TILE_PITCH + (s16 % NI) * 64 + s16 / NI * 16 + tile_row % 16;
        float sum[WAVES];   // (added up in pairs: fewer roundings on the way of each)
#pragma unroll
        for (int k = 0; k < WAVES; ++k) sum[k] = p[k * RT * ZT * TILE_PITCH];
#pragma unroll
        for (int step = 1; step < WAVES; step *= 2)
#pragma unroll
            for (int k = 0; k < WAVES; k += 2 * step) sum[k] += sum[k + step];
        if constexpr (BS) return LINKED || ssq_in ? sum[0] * rms_scale[sq] : sum[0];
        else return sum[0] * inv;
    };
    if constexpr (FORM == kQ4Silu) {
        // the 32 lanes of a half wave hold one request's 32 columns, one block of the consuming matmul's K
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const uint32_t qp = q + p * PER_PASS, bp = b + p * PER_PASS;
            if (qp >= live) break;
            const float gv = sum_of(row, qp, inv_pre[p]), uv = sum_of(32 + row, qp, inv_pre[p]);
            const float prod = q4_silu_times(gv, uv);
            store_through(&a.out[(size_t)bp * a.rows + col], gv);
            store_through(&a.out[(size_t)bp * a.rows + a.ffn_inner + col], uv);
            store_through(&a.gate[(size_t)bp * a.ffn_inner + col], gv);
            store_through(&a.up[(size_t)bp * a.ffn_inner + col], uv);
            store_through(&a.silu_out[(size_t)bp * a.ffn_inner + col], prod);
            if (a.split_frag) q4_emit_block(prod, bp, col, a.ffn_inner, a.split_frag, a.split_blk_scale, WIDTH);
        }
        return;
    }
    // K slices: all but the last leave their sums as tagged words and are done; the last one's workgroups, which are the
    // last of the launch, add them to their own in slice order (tagged_words.h: why the wait ends).
    const uint32_t tag = launch_tag(a.tags.tag, tag_add);
    if (slice + 1 < a.slices) {
        if ((a.tags.test_flags & 1u) || copy != 0) return;
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const uint32_t qp = q + p * PER_PASS, bp = b + p * PER_PASS;
            if (qp >= live) break;
            st_tagged(a.meet + ((size_t)slice * batch + bp) * a.rows + col,
                      (uint64_t)tag << 32 | __float_as_uint(sum_of(row, qp, inv_pre[p])));
        }
        return;
    }
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        const uint32_t qp = q + p * PER_PASS, bp = b + p * PER_PASS;
        if (qp >= live) break;
        float val = sum_of(row, qp, inv_pre[p]);
        if (a.slices > 1) {
            constexpr uint32_t AT_ONCE = 4;
            float others = 0.f;
            uint32_t spins = 0;
            for (uint32_t s0 = 0; s0 + 1 < a.slices; s0 += AT_ONCE) {
                const uint64_t* src = a.meet + ((size_t)s0 * batch + bp) * a.rows + col;
                uint64_t word[AT_ONCE];
                for (;;) {
                    bool ok = true;
#pragma unroll
                    for (uint32_t s = 0; s < AT_ONCE; ++s)
                        if (s0 + s + 1 < a.slices) word[s] = ld_tagged(src + (size_t)s * batch * a.rows);
#pragma unroll
                    for (uint32_t s = 0; s < AT_ONCE; ++s)
                        if (s0 + s + 1 < a.slices) ok = ok && (uint32_t)(word[s] >> 32) == tag;
                    if (__all(ok)) break;
                    if (++spins >= a.tags.spin_limit) {
                        if (!ok) report_fault(a.tags.fault);
                        break;
                    }
                }
#pragma unroll
                for (uint32_t s = 0; s < AT_ONCE; ++s)
                    if (s0 + s + 1 < a.slices) others += __uint_as_float((uint32_t)word[s]);
            }
            val = others + val;
        }
        if constexpr (LINK == kQ4LinkOut) {
            // (what the other matmul waits for first)
            const float hv = val + resid_pre[p], ssq = q4_half_wave_sum(hv * hv);
            if (!(link.tags.test_flags & 1u))
                q4_emit_words(hv * gamma_pre, hv, ssq, bp, col, a.rows, batch, link.words + copy * q4_link_words(a.rows, batch), link_tag);
            if (copy != 0) return;   // (whole half waves)
        }
        store_through(&a.out[(size_t)bp * a.rows + col], val);
        if constexpr (FORM == kQ4Rope) q4_rope_epilogue(a.rope, rope_pre[p], bp, col, val);   // (the lanes of a pair share b)
        if constexpr (FORM == kQ4Add) {
            // residual add, this request's sum of squares over a half wave's 32 columns, and h * gamma as the next
            // matmul's fragments
            const float hv = val + resid_pre[p];
            store_through(&a.add_out[(size_t)bp * a.rows + col], hv);
            if (LINK == kQ4LinkNone && a.split_frag) {   // (else the add is all)
                const float ssq = q4_half_wave_sum(hv * hv);
                if (row % 32 == 0) store_through(&a.ssq_out[(size_t)bp * (a.rows / 32) + col / 32], ssq);
                q4_emit_block(hv * gamma_pre, bp, col, a.rows, a.split_frag, a.split_blk_scale, WIDTH);
            }
        }
    }
}

template <int NI, int RT, int WAVES, bool BS, int FORM, int ZT = 1>
__global__ __launch_bounds__(WAVES * 64, ZT > 1 ? 2 : 4) void q4_matmul_kernel(
    const uint4* const w_q, const uint2* const w_d, const _Float16* const xfrag, const float* const blk_scale, const float* const ssq_in,
    const uint32_t nblocks, const uint32_t quads_per_slice, const uint32_t row_groups, const uint32_t batch_z,
    const std::conditional_t<FORM == kQ4Rope, Q4RopeArgs, Q4Args> a) {
    __shared__ Q4Lds<NI, RT, WAVES, BS, ZT> lds;
    q4_matmul_workgroup<NI, RT, WAVES, BS, FORM, ZT, kQ4LinkNone, 0>(lds, blockIdx.x, blockIdx.y, kQ4LeadBytes + kQ4RopeOffset, w_q, w_d, xfrag,
                                                                  blk_scale, ssq_in, nblocks, quads_per_slice, row_groups, batch_z, a, Q4Link{});
}

// Two matmuls of up to 4 requests in one launch: one with the residual add that starts an RMSNorm, and the one that reads
// the norm.  The first matmul's workgroups come first, in all their K slices; the second one's request their weights, and then wait
// for the first one's sums as tagged words (tagged_words.h: why the waits end).  That takes a launch's start and end and the second
// one's way to its first weights off the chain of launches that a step is, and its unpacking, 0.7 us of the vector pipe per four
// row tiles: while it waits a wave holds its weights as halves in up to 64 registers.
//
// Measured: out-projection and gate/up of the 1 B shape at one request 12.0 us in two launches, 8.0 in one, of which, from the
// start: the first one's weights back 1.5, its sums published 3.5 (vector pipe, 16 waves), seen 4.3, all words in LDS 4.9, products
// 5.9, waves' sums met 6.3, stored 7.4.  With one copy of the words, a quad's scales in the lines of all the others' they were seen at
// 5.5.  Steps of 22 layers, us, two launches -> one: 1, 2, 3, 4 requests 683, 696, 702, 705 -> 618, 643, 654, 673; a
// build for 5 and 8 requests 771, 778 -> 763, 784 (every workgroup fetches 8 bytes per request and column): two launches there.
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
