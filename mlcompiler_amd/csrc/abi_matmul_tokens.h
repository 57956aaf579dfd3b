// Host side of the Q4_0 and Q6_K matmuls over more than 64 tokens.
//
// A section of the one translation unit mlc_hip.hip, which includes it once, in order, after the
// sections before it; not a header for anybody else.

namespace {

// The largest piece of an input that is split at a time, and the K slices' buffer: workspaces of one
// size for good (a buffer that grows would put an end to the captured passes).
constexpr size_t kTokensFragBytes = 64u << 20, kTokensSliceBytes = 32u << 20;

// How one piece is divided: K is split where the workgroups would leave CUs idle (two fit one), in whole groups of
// 4 stages, and never into more slices than the buffer holds.
struct TokensPlan {
    uint32_t stages_per_slice;
    size_t ksplit;
};
TokensPlan tokens_plan(size_t wgs, size_t slots, size_t stages, size_t out_bytes) {
    size_t ksplit = std::max<size_t>(1, std::min({slots / wgs, stages / 4, kTokensSliceBytes / out_bytes}));
    const size_t per = ((stages + ksplit - 1) / ksplit + 3) / 4 * 4;
    return {(uint32_t)per, (stages + per - 1) / per};   // (rounding up leaves no more slices than before)
}

// All tokens of a call with more than 64 in one launch per piece (matmul_tokens_kernels.h).
// Returns 0 where the call has to go 64 requests at a time instead: workspaces not at hand.
int matmul_tokens(bool q6, TokensArgs a, const float* in, float* out, size_t batch, size_t rows, size_t cols) {
    const size_t piece = kTokensFragBytes / (4 * cols) / 64 * 64;
    if (piece == 0) return 0;
    for (const char* name : {"tokens_x_fragments", "tokens_x_inv_scale", "tokens_k_slices"})
        if (g_capturing && !g.cached.count(name)) return 0;
    _Float16* frag = static_cast<_Float16*>(cached_buffer("tokens_x_fragments", kTokensFragBytes));
    float* inv = static_cast<float*>(cached_buffer("tokens_x_inv_scale", kTokensFragBytes / 64));   // (cols >= 64)
    float* slices = static_cast<float*>(cached_buffer("tokens_k_slices", kTokensSliceBytes));
    if (!frag || !inv || !slices) return 0;
    a.xfrag = frag;
    a.inv_scale = inv;
    a.rows = (uint32_t)rows;
    a.ksteps = (uint32_t)(cols / 16);
    a.stages = (uint32_t)((cols + 63) / 64);
    a.row_blocks = (uint32_t)((rows + 127) / 128);
    for (size_t bo = 0; bo < batch; bo += piece) {
        const size_t bn = std::min(piece, batch - bo);
        float* o = out + bo * rows;
        a.tokens = (uint32_t)bn;
        a.token_blocks = (uint32_t)((bn + 63) / 64);
        launch_tokens_split(in + bo * cols, frag, inv, (uint32_t)bn, (uint32_t)cols, a.token_blocks * 16, g.stream);
        const size_t wgs = (size_t)a.token_blocks * a.row_blocks;
        const TokensPlan plan = tokens_plan(wgs, 2 * (size_t)g.n_cu, a.stages, bn * rows * 4);
        a.stages_per_slice = plan.stages_per_slice;
        // (first-level sums of 4, 8 or 16 stages: about as many as there are of them)
        a.flush_mask = a.stages_per_slice <= 48 ? 0 : a.stages_per_slice <= 512 ? 1 : 3;
        a.out = plan.ksplit > 1 ? slices : o;
        launch_matmul_tokens(q6, a, (unsigned)(wgs * plan.ksplit), g.stream);
        if (plan.ksplit > 1) {
            const uint32_t n = (uint32_t)(bn * rows);
            hipLaunchKernelGGL(q4_sum_slices_kernel, dim3((n + 255) / 256), dim3(256), 0, g.stream, slices, o, n,
                               (uint32_t)plan.ksplit);
        }
    }
    return 1;
}

}  // namespace
