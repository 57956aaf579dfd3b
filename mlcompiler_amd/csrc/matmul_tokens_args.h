// Arguments and launches of the matmuls over many tokens (matmul_tokens_inst.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tagged_words.h"

namespace mlc_hip {

struct TokensArgs {
    const uint2* q;          // repacked weights: Q4Args::q / Q6KArgs::qa
    const uint32_t* sc;      // Q6KArgs::sc (Q4_0: not read)
    const _Float16* d;       // Q4Args::d / Q6KArgs::d
    const _Float16* xfrag;   // split activations of token_blocks * 64 rows, 32 requests wide (fragments.h, tokens_split_kernel)
    const float* inv_scale;  // [tokens]
    float* out;              // [tokens][rows], or the slice buffer [ksplit][tokens][rows]
    uint32_t tokens, rows;
    uint32_t ksteps;         // cols / 16
    uint32_t nblocks;        // cols / 32 (Q4_0) or cols / 256 (Q6_K)
    uint32_t stages, stages_per_slice;   // stages of 64 columns
    uint32_t token_blocks, row_blocks;   // blocks of 64 tokens / 128 rows
    uint32_t flush_mask;                 // a first-level sum ends where (stage group number & mask) == mask, groups of 4
    // The first `whole` workgroups take a tile (64 tokens x 128 rows) and a slice of K each, as above.  Those behind them
    // take the last `rest` tiles, in tail_slices slices of K: all slices but the last leave their sums for the last one.
    uint32_t whole, rest, tail_slices, tail_stages;
    uint64_t* meet;                      // [tail_slices - 1][rest][64 * 128] tagged words
    TagArgs tags;
};

void launch_tokens_split(const float* x, _Float16* frag, float* inv_scale, uint32_t tokens, uint32_t cols, unsigned grid, hipStream_t stream);
void launch_matmul_tokens(bool q6, const TokensArgs& a, unsigned grid, hipStream_t stream);

}  // namespace mlc_hip
