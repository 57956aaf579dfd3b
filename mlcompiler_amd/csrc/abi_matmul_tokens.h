// Host side of the Q4_0 and Q6_K matmuls over more than 64 tokens.
//
// A section of the one translation unit mlc_hip.hip, which includes it once, in order, after the
// sections before it; not a header for anybody else.

namespace {

// The largest piece of an input that is split at a time, and the K slices' buffer: workspaces of one
// size for good (a buffer that grows would put an end to the captured passes).
constexpr size_t kTokensFragBytes = 64u << 20, kTokensSliceBytes = 32u << 20;

// The last round's K slices: at least so many stages each, at most so many of them, and what they leave each other (64 x 128
// words of 8 bytes for each of fewer than `slots` workgroups).
constexpr size_t kTokensTailStages = 8, kTokensTailSlices = 4, kTokensMeetBytes = 32u << 20;

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

// The tiles left over by whole rounds of the slots: a quarter of a round or less leaves every CU one workgroup or none, and
// two to a CU do more than one.  They go to several workgroups each, a slice of K for every one, whose sums meet inside the
// launch.  That costs about 5 us, hence the longer K the more such tiles (whole calls, us, whole K / slices; Q4_0):
//   tiles left | 16 stages   | 32 stages    | 64 stages     | 88, 224
//   32         | 52.5 / 51.2 | 80.1 / 68.6  | 254.8 / 235.2 | 404 / 317 (8 slices at most: 312)
//   64         | 51.4 / 51.3 | 77.9 / 69.7  |               | 177 / 152 (157)
//   96         | 51.3 / 52.4 | 78.1 / 73.2  | 125.5 / 116.2 |
//   128        | 50.7 / 53.0 | 76.5 / 77.8  | 124.8 / 119.0 | 388 / 357
// 192 tiles in two slices (11264 x 2048, 512 tokens): 75.8 / 78.5.  Q6_K, 32 tiles, 32 stages: 82.4 / 72.2.
struct TokensTail {
    uint32_t whole, rest, slices, stages;
};
TokensTail tokens_tail(size_t wgs, size_t slots, size_t stages) {
    const size_t rest = wgs % slots;
    if (wgs < slots || rest == 0 || rest > std::min(slots / 4, 3 * stages)) return {(uint32_t)wgs, 0, 1, 0};
    const size_t n = std::min({slots / rest, stages / kTokensTailStages, kTokensTailSlices});
    if (n < 2) return {(uint32_t)wgs, 0, 1, 0};
    const size_t per = ((stages + n - 1) / n + 3) / 4 * 4;
    return {(uint32_t)(wgs - rest), (uint32_t)rest, (uint32_t)((stages + per - 1) / per), (uint32_t)per};
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
        const size_t slots = 2 * (size_t)g.n_cu;
        const TokensPlan plan = tokens_plan(wgs, slots, a.stages, bn * rows * 4);
        a.stages_per_slice = plan.stages_per_slice;
        // (first-level sums of 4, 8 or 16 stages: about as many as there are of them)
        a.flush_mask = a.stages_per_slice <= 48 ? 0 : a.stages_per_slice <= 512 ? 1 : 3;
        // All tiles in slices: they meet inside the launch too where they are few or short (rows x columns at tokens, summed by
        // a kernel behind / in the launch, us: two slices 6144 x 4096 at 300 64.2 / 60.9, 11264 x 2048 at 128 45.1 / 41.7; four
        // of 8 stages 2048 x 2048 at 512 42.3 / 39.2, of 16 4096 x 4096 at 256 47.8 / 47.4, of 24 2048 x 5632 at 512 56.6 /
        // 58.4, of 56 4096 x 14336 at 200 98.5 / 100.3).
        const TokensTail none{(uint32_t)(wgs * plan.ksplit), 0, 1, 0};
        TokensTail tail = none;
        const bool meet = sliced_tags_left() && (slots - 1) * 65536 <= kTokensMeetBytes;
        if (meet && plan.ksplit == 1) tail = tokens_tail(wgs, slots, a.stages);
        else if (meet && plan.ksplit <= (plan.stages_per_slice <= 16 ? kTokensTailSlices : 3)) tail = {0, (uint32_t)wgs, (uint32_t)plan.ksplit, plan.stages_per_slice};
        // (room to meet in is taken by the first call that has use for it, and a call that finds none does without)
        a.meet = tail.rest ? meeting_words("tokens_k_meet", kTokensMeetBytes) : nullptr;
        if (!a.meet) tail = none;
        const bool sum = plan.ksplit > 1 && !tail.rest;
        a.out = sum ? slices : o;
        a.whole = tail.whole;
        a.rest = tail.rest;
        a.tail_slices = tail.slices;
        a.tail_stages = tail.stages;
        a.tags = tail.rest ? next_sliced_tags() : TagArgs{};
        if (tail.rest && !scratch_follow(g.stream)) return 0;
        launch_matmul_tokens(q6, a, tail.whole + tail.rest * tail.slices, g.stream);
        if (tail.rest && !scratch_launched(g.stream)) return 0;
        if (sum) {
            const uint32_t n = (uint32_t)(bn * rows);
            hipLaunchKernelGGL(q4_sum_slices_kernel, dim3((n + 255) / 256), dim3(256), 0, g.stream, slices, o, n,
                               (uint32_t)plan.ksplit);
        }
    }
    return 1;
}

}  // namespace
