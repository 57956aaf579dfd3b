// Arguments, rules and launches of the chunked prefill attention (paged_prefill_inst.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace mlc_hip {

static constexpr size_t kPrefillEmbWords = 960;   // words of tables that travel inside the kernel arguments

struct PrefillArgs {
    float4* part_o;      // keys split over workgroups: the parts' sums [part][wave of the grid][head_dim / 8][lane], as the
    float2* part_ml;     // lanes hold them, and their (reference, sum of weights) [part][wave of the grid][32 rows]
    const _Float16* q;
    const _Float16* k_pages;
    const _Float16* v_pages;
    float* o;
    // page_table_offsets [batch] | seq_lens [batch] | q_start [batch] | flat page table: in pinned host
    // memory, or null and inside the arguments (emb)
    const uint32_t* tables;
    uint32_t batch, chunk, num_heads, kv_heads, page_size;
    uint32_t row_blocks;  // workgroups along the chunk
    float scale_log2e;
    uint32_t emb[kPrefillEmbWords];
};
static constexpr int kPfKeys = 32;   // keys per tile
static constexpr int kPfRows = 32;   // chunk rows per wave
static constexpr int kPfWaves = 8;   // waves per workgroup

// GQA ratio 8: 64 rows of four heads per workgroup where there are enough key tiles, else 32 rows of all eight.  Both have 256
// (row, head) pairs; the kernel with 64 rows reads an operand from LDS for two products, and takes longer until its first tile.
// (Whole calls, us, 32 -> 64 rows, by tiles of the longest
// row block.  head_dim 64: 2 tiles 20.3 -> 21.3, 4 23.3 -> 23.9, 8 25.9 -> 26.2, 34.1 -> 32.8 and 24.5 -> 24.5, 9 30.8 -> 31.5, 10 34.0 -> 31.5
// and 41.9 -> 41.4, 12 37.5 -> 34.1, 25 47.1 -> 40.4, 128 124 -> 110.  128: 4 28.6 -> 30.1, 8 48.5 -> 51.4 and 30.3 -> 30.6, 10 60.8 -> 63.2,
// 12 50.8 -> 51.7 and 52.5 -> 51.8, 16 62.5 -> 60.7 and 40.2 -> 38.5, 25 58.1 -> 53.8, 128 162 -> 146.)
// And it takes workgroups of its own for a last row block of at most 32 rows: only where they are no more rounds over the CUs, or
// hardly more.  (By rounds of 32 and of 64 rows, 19 or 47 tiles, 32 -> 64 rows: equal 0.99 to 1.15 times as fast; 1 and 2 0.63
// to 0.83, 2 and 4 0.65 to 0.75, 2 and 3 0.78 to 0.86, 3 and 4, 4 and 5 0.86 to 0.97, 5 and 6 0.93 to 1.01, 11 and 12 0.95 to 0.98.  32
// requests of 32 rows behind 3 000 keys with 8 KV heads of 128 153 -> 201 us, 40 of 96 behind 1 000 208 -> 224: both 32 rows.)
// pairs: requests x KV heads.
inline bool prefill_rows64_ratio8(size_t head_dim, size_t max_tiles, size_t chunk, size_t pairs, size_t n_cu) {
    const auto rounds = [&](size_t blocks) { return (blocks * pairs + n_cu - 1) / n_cu; };
    return max_tiles >= (head_dim == 64 ? 10u : 16u) && rounds((chunk + 63) / 64 * 2) * 20 <= rounds((chunk + 31) / 32) * 21;
}

inline bool prefill_shape_supported(size_t head_dim, size_t page_size, size_t num_heads,
                                    size_t kv_heads) {
    const size_t g = kv_heads ? num_heads / kv_heads : 0;
    return (head_dim == 64 || head_dim == 128) && page_size % kPfKeys == 0 &&
           (g == 1 || g == 2 || g == 4 || g == 8);
}

// A prefill of few rows leaves most of the chip idle while each workgroup walks all of the keys, 0.77 us (head_dim
// 64) or 0.97 us (128) per 32-key tile; its keys are then cut into parts, at most as many as there are CUs for,
// of at least two tiles.  Writing the parts and adding them up takes 2 us and 0.36 us per MB of them (measured:
// 1.4 to 2.9 us where they are 1 to 4 MB, 3.2 to 4.5 for 5 to 8 MB, 7.7 for 15 and 16): the number of parts is the one
// with the least sum, and one where that saves less than 1 us.
// max_tiles: key tiles of the longest row block.  Whole calls in us, one part (or, in brackets, the parts of a
// rule that asked for 16 tiles and four per part, laid out by rows) -> now: 32 rows at 32 / 4 heads of 64 behind 224,
// 320, 416 keys 23.0, 25.2, 27.5 -> 20.8, 21.1, 21.0; of 128 behind 416 33.3 -> 23.3, four requests of that
// 33.9 -> 27.6; 3 x 77 rows behind up to 900 keys (36 workgroups) 39.9 (32.1) -> 26.4, 256 rows behind 3 840 at 32 / 8
// heads of 128 (32) 117 (50.6) -> 46.4, 64 rows behind 8 000 (53) -> 40, 700 rows from scratch at 16 / 4 heads
// of 64 (31.4) -> 25.6; two parts (4 x 256 rows behind up to 2 000, 128 workgroups) 77 -> 67.  Where both are equal:
// 2 x 256 rows behind 400 at 32 / 8 heads of 128, 39.8 with one part, 39.3 with three (37.8).
inline size_t prefill_wgs(size_t batch, size_t chunk, size_t num_heads, size_t kv_heads) {
    const size_t rows_per_wg = kPfRows * kPfWaves / (num_heads / kv_heads);
    return (chunk + rows_per_wg - 1) / rows_per_wg * kv_heads * batch;
}
inline uint32_t prefill_splits(size_t wgs, size_t head_dim, size_t max_tiles, size_t n_cu, size_t part_bytes) {
    const size_t one = wgs * kPfWaves * kPfRows * (head_dim + 2) * 4, tile_ns = head_dim == 64 ? 770 : 970;
    const size_t most = std::min({n_cu / wgs, max_tiles / 2, part_bytes / one, (size_t)64});
    size_t best = 1, best_ns = max_tiles * tile_ns - std::min<size_t>(max_tiles * tile_ns, 1000);
    for (size_t p = 2; p <= most; ++p) {
        const size_t ns = (max_tiles + p - 1) / p * tile_ns + 2000 + p * one / 2800;
        if (ns < best_ns) best = p, best_ns = ns;
    }
    return (uint32_t)best;
}

// stages: LDS pipeline depth (2, 4, 6 or 8; anything else selects 6).  rows64: 64 chunk rows per
// wave, else 32.  splits: parts into which every workgroup's keys are cut (more than
// one: 32 rows per wave, partial sums in a.part_o / part_ml, prefill_splits() says how many).
void launch_prefill_64(const PrefillArgs& a, int stages, bool rows64, uint32_t splits, hipStream_t stream);
void launch_prefill_128(const PrefillArgs& a, int stages, bool rows64, uint32_t splits, hipStream_t stream);
inline void launch_prefill(const PrefillArgs& a, size_t head_dim, int stages, bool rows64, uint32_t splits, hipStream_t stream) {
    (head_dim == 64 ? launch_prefill_64 : launch_prefill_128)(a, stages, rows64, splits, stream);
}

}  // namespace mlc_hip
