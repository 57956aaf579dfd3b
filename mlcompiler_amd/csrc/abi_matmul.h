// Entry points of the batched Q4_0 and Q6_K matmuls and their device-resident weights.
//
// A section of the one translation unit mlc_hip.hip, which includes it once, in order, after the
// sections before it; not a header for anybody else.

extern "C" {

// ---- batched Q4_0 matmul -------------------------------------------------------------------

namespace {

bool q4_fast_shape(size_t rows, size_t cols, size_t row_stride) {
    // (the kernels address a tile's weights and a row's fragments with 32 bits)
    return rows % 64 == 0 && cols % 32 == 0 && cols <= (1u << 24) && row_stride >= cols / 32 * 18;
}

// K slices of a Q4_0 matmul on the matrix cores and the quads of blocks in each.  K is split over workgroups (of 32 rows)
// where there are too few of them for the CUs, as far as that leaves a wave fewer quads in a row: a round of quads takes
// a wave about 1.5 us, the slices' meeting inside the launch 0.8.  (Kernel times, us, one slice, or two summed by a
// launch behind -> now: 2048 x 5632 with the residual add at one request 8.2 -> 5.8 (three slices), at 32 requests 10.5 -> 8.6;
// 4096 x 4096 with it at 16 8.8 -> 7.6; 4096 x 14336 at 16 14.1 and 4.2 for sum and add -> 15.2.)
struct Q4Slices { size_t n, quads; };
Q4Slices q4_slices(size_t rows, size_t cols, size_t batch) {
    const size_t nblocks = cols / 32, quads = (nblocks + 3) / 4, n_cu = (size_t)g.n_cu, z = (batch + 15) / 16;
    size_t n = (size_t)g.opt_q4_ksplit;
    if (n == 0 && !g.opt_q4_int_operand) n = std::min(n_cu / (rows / 32), quads / 48);
    else if (n == 0) n = std::max(std::min(n_cu / (rows / 32 * z), (quads + 15) / 16), std::min(n_cu / (rows / 32), quads / 48));
    n = std::max<size_t>(1, std::min(n, nblocks / 16));
    const size_t per_slice = (quads + n - 1) / n;
    return {(quads + per_slice - 1) / per_slice, per_slice};
}

// A matmul that is a call of its own takes its rows of floats as they are and splits them itself, every workgroup all of them, where
// that takes less than a launch in front, 1.5 to 2 us and a little for long rows.  (The split is of every block by itself, as the fused
// launches have it.)  A wave splits 128 columns of every request in each of its turns, and what that takes, 0.15 us per turn and request with 16
// waves on a CU, is on the way of everybody behind it.  More than four requests: a build for eight, which splits as if there were eight, and for
// four row tiles to a workgroup would spill.  Whole calls, us, split in front / now, in brackets where the split stays in front (turns):
//   rows x columns | 1             | 4             | 5             | 8
//   2560 x 2048    | 16.4 / 14.3   | 16.1 / 15.0   | 17.0 / 15.6   | 16.9 / 16.2     (1)
//   8192 x 2048    |               |               | 18.5 / 16.9   | 18.5 / 17.5     (1, two row tiles)
//   2048 x 5632    | 17.5 / 15.7   | 17.4 / 16.3   | 19.2 / 17.7   | 19.2 / 18.4     (1)
//   2560 x 6912    |               |               | 19.8 / 18.7   | 19.7 / 19.0     (1.1)
//   11264 x 2048   | 17.9 / 16.2   | 17.9 / 17.0   | four tiles    |                 (1)
//   4096 x 14336   | 24.3 / 21.7   | 24.3 / 23.3   | (26.1 / 26.3) | (25.9 / 27.7)   (3.5)
//   28672 x 4096   | 29.2 / 27.8   | (29.5 / 29.9) | four tiles    |                 (4)
//   8192 x 8192    | 23.6 / 22.1   | (24.0 / 24.4) | (25.5 / 27.7) | (25.6 / 30.1)   (4)
//   5120 x 13824   | 27.8 / 26.0   | (27.0 / 29.2) |               |                 (6.8)
//   64000 x 4096   | 42.2 / 42.1   | (42.1 / 46.1) | four tiles    |                 (8: two rounds of workgroups)
//   128256 x 4096  | (65.4 / 69.6) | (70.2 / 78.2) | four tiles    |                 (16)
bool q4_splits_rows(size_t rows, size_t cols, size_t batch) {
    if (batch > 8) return false;
    const Q4Slices s = q4_slices(rows, cols, batch);
    if (batch > 4 && q4_tiles(kQ4Rows, rows, batch, s.n) > 2) return false;
    // (as many workgroups as CUs have 16 waves, more of them 8, two workgroups to a CU: q4_waves)
    const size_t n_cu = (size_t)g.n_cu, wgs = rows / 64 * s.n, waves = wgs > n_cu ? 8 : 16;
    const size_t rounds = wgs > n_cu ? (wgs + 2 * n_cu - 1) / (2 * n_cu) : 1;
    const size_t turns16 = rounds * std::max(waves, s.quads) * 16 / waves;   // sixteenths
    return turns16 * (batch <= 4 ? batch : 8) <= 16 * 11 + cols / 256;
}

// The split of a batch's rows into fragments: 1024 threads per row above 4096 columns, where 256 keep no row in registers.
void launch_q4_split(const float* x, _Float16* frag, float* inv_scale, size_t batch, size_t cols) {
    const unsigned threads = cols > 4096 ? 1024 : 256;
    hipLaunchKernelGGL(threads == 1024 ? q4_split_activations_kernel<1024> : q4_split_activations_kernel<256>, dim3((unsigned)batch), dim3(threads),
                       0, g.stream, x, frag, inv_scale, (uint32_t)batch, (uint32_t)cols);
}

// Copies weights to the device in the order of the library's stream (a plain hipMemcpy may return before the data is
// there, and the library's stream does not wait for it), and waits.
bool upload_weights(void* dst, const void* host, size_t bytes) {
    return hipMemcpyAsync(dst, host, bytes, hipMemcpyHostToDevice, g.stream) == hipSuccess && hipStreamSynchronize(g.stream) == hipSuccess;
}

// Gives up a matrix whose layout for the matrix cores is not complete, so that the next call starts over (hipFree waits
// for what still reads it).
void drop_weight(Ctx::Q4Weight& w) {
    for (void* p : {w.raw, w.q, w.d})
        if (p) (void)hipFree(p);
    w = Ctx::Q4Weight{};
}

// Uploads the weight matrix on first use of its name (or when its size changed).
Ctx::Q4Weight* q4_weight(const char* name, const uint8_t* host, size_t bytes, size_t rows, size_t cols,
                         size_t stride) {
    Ctx::Q4Weight& w = g.q4_weights[name];
    if (w.is(bytes, rows, cols, stride)) return &w;
    if (g_capturing) { fail("q4 matmul: the weights are not on the device yet (run the pass once uncaptured first)"); return nullptr; }
    (void)hipStreamSynchronize(g.stream);
    for (void** p : {&w.raw, &w.q, &w.d})
        if (*p) { (void)hipFree(*p); *p = nullptr; ++g.buffer_generation; }
    w = Ctx::Q4Weight{};
    void* raw = nullptr;
    if (hipMalloc(&raw, bytes) != hipSuccess) { (void)hipGetLastError(); fail("q4 matmul: hipMalloc failed"); return nullptr; }
    if (!upload_weights(raw, host, bytes)) { (void)hipFree(raw); fail("q4 matmul: upload failed"); return nullptr; }
    w.raw = raw; w.bytes = bytes; w.rows = rows; w.cols = cols; w.stride = stride;
    if (q4_fast_shape(rows, cols, stride)) {
        const size_t nb = cols / 32, quads = (nb + 3) / 4, tiles = rows / 16, units = tiles * quads * 64;
        if (hipMalloc(&w.q, units * 16) != hipSuccess || hipMalloc(&w.d, tiles * quads * 16 * 8) != hipSuccess) {
            (void)hipGetLastError();
            drop_weight(w);
            fail("q4 matmul: hipMalloc failed");
            return nullptr;
        }
        hipLaunchKernelGGL(q4_repack_kernel, dim3((unsigned)((units + 255) / 256)), dim3(256), 0, g.stream,
                           static_cast<const uint8_t*>(w.raw), static_cast<uint4*>(w.q), static_cast<uint16_t*>(w.d),
                           (uint32_t)tiles, (uint32_t)nb, (uint32_t)quads, stride);
        if (hipGetLastError() != hipSuccess) { drop_weight(w); fail("q4 matmul: repacking failed"); return nullptr; }
    }
    return &w;
}

}  // namespace

int mlc_hip_matmul_q4_0_batched(const char* weight_name, const void* weights, size_t weight_bytes,
                                const void* in, size_t batch, size_t rows, size_t cols,
                                size_t row_stride, uint32_t quant_version, void* out, int sync) {
    (void)quant_version;  // one block format: quantization.cpp:228-246 ignores it as well
    if (!init_once()) return fail("GPU unavailable");
    if (!sync && !g.pass_open) return fail("encode: no open forward pass");
    if (!in || !out || batch == 0 || rows == 0 || cols == 0) return fail("q4 matmul: null buffer or zero size");  // :6940
    if (cols < 64 || (rows % 4u) != 0) return fail("q4 matmul: needs cols >= 64 and rows % 4 == 0");          // :6942
    if (!weight_name || !weights) return fail("q4 matmul: null weights");
    const size_t nb = (cols + 31) / 32;
    if (row_stride < nb * 18 || weight_bytes < (rows - 1) * row_stride + nb * 18)
        return fail("q4 matmul: weight bytes do not cover rows x row_stride");
    if (batch * rows > 0x7FFFFFFFull || batch * cols > 0x7FFFFFFFull) return fail("q4 matmul: too many elements");
    const size_t ki = known_bytes(in), ko = known_bytes(out);
    if ((ki && batch * cols * 4 > ki) || (ko && batch * rows * 4 > ko)) return fail("q4 matmul: buffer too small");
    // (another matrix under a name that is known: a held-back matmul may read the one it replaces)
    const auto known = g.q4_weights.find(weight_name);
    if (known != g.q4_weights.end() && !known->second.is(weight_bytes, rows, cols, row_stride) && !settle()) return 0;
    // does the pending chain end in this matmul's input?  (decided before anything below can
    // replace a buffer the chain still refers to)
    const bool feeds = batch <= 64 && !g.opt_q4_force_generic && !(reinterpret_cast<uintptr_t>(out) & 15u) &&
                       q4_fast_shape(rows, cols, row_stride) && row_len_ok(cols) && rows_continue(in, batch, cols);
    // ... and is that chain  held-back matmul -> + residual -> RMSNorm?  Then the held-back matmul's
    // epilogue adds, leaves the sums of squares and writes (sum * gamma) as this matmul's fragments,
    // block-wise scaled, and this matmul finishes the norm: no launch in between.
    // (Wide matrices read block-wise scaled activations for up to 32 requests only: which launches are fused
    // beyond is pinned by tests of the launch counts.)
    const bool scales_fit = batch <= 32 || !q4_wide(rows);
    bool feeds_rms = false;
    if (feeds && scales_fit && g.gemm.active && g.opt_q4_int_operand) {
        const RowProgram& p = g.rows.p;
        const size_t row_bytes = batch * cols * 4;
        feeds_rms = gemm_adds() && p.rms && g.rows.batch == batch && g.rows.len == cols && cols / 32 <= 128 &&
                    // (as many elements as the reader's threads, over all requests: tests of the launch counts pin it)
                    batch * cols <= rows / (q4_wide(rows) ? 64 : 32) * 1024 &&
                    // Every row group of the reader writes 1024 elements of its z group's part of the norm (in whichever
                    // form it will be launched), and no element belongs to two: one slice of K,
                    std::min<size_t>(batch, 16) * cols <=
                        rows / 16 / std::max(q4_tiles(q4_wide(rows) ? kQ4Silu : kQ4Add, rows, batch, 1), q4_tiles(kQ4Plain, rows, batch, 1)) * 1024 &&
                    g.opt_q4_ksplit <= 1 &&
                    // and its buffers lie apart, too: it reads the sum and writes the norm
                    !shifted(p.rms_out, p.add_out, row_bytes) && !overlap(out, batch * rows * 4, p.add_out, row_bytes) &&
                    !overlap(out, batch * rows * 4, p.rms_out, row_bytes);
    }
    // ... or is the input the SiLU * up product that the held-back gate/up projection's epilogue
    // will write?  Then that epilogue also splits it, per (request, block of 32 columns).
    const bool feeds_silu = !feeds && scales_fit && batch <= 64 && g.opt_fuse_rows && g.opt_q4_int_operand && !g.opt_q4_force_generic &&
                            !(reinterpret_cast<uintptr_t>(out) & 15u) && q4_fast_shape(rows, cols, row_stride) &&
                            g.gemm.active && g.gemm.silu && !g.rows.active && !g.kv.active && g.gemm.silu_out == in &&
                            g.gemm.batch == batch && g.gemm.ffn_inner == cols;
    // ... or the output of the held-back decode attention?  Then the attention kernel splits it.
    const bool feeds_attn = !feeds && !feeds_silu && scales_fit && batch <= 64 && g.opt_fuse_rows && g.opt_q4_int_operand &&
                            !g.opt_q4_force_generic && !(reinterpret_cast<uintptr_t>(out) & 15u) &&
                            q4_fast_shape(rows, cols, row_stride) && g.dec.active && g.dec.o == in &&
                            g.dec.batch == batch && g.dec.cols == cols;
    const bool block_scales = feeds_silu || feeds_attn || feeds_rms;
    const Ctx::Q4Input x_from = feeds_silu ? Ctx::kXSilu : feeds_attn ? Ctx::kXAttention : feeds_rms ? Ctx::kXNorm : Ctx::kXSplit;
    // The held-back matmul writes this one's input.  Where its own came the same way (a matmul that both finishes a
    // norm and starts the next one) the two inputs take turns between two sets of buffers: some of its workgroups
    // still read the one when others are done and write the other.
    const int x_set = (feeds_silu || feeds_rms) && g.gemm.x_from == x_from ? 1 - g.gemm.x_set : 0;
    // (a held-back matmul that does not take the chain over goes out now: it may read a buffer that is replaced below)
    if (feeds && !feeds_rms ? !settle_before_rows() : !block_scales && !settle()) return 0;
    Ctx::Q4Weight* w = q4_weight(weight_name, static_cast<const uint8_t*>(weights), weight_bytes, rows, cols, row_stride);
    if (!w) return 0;

    if (!w->q || g.opt_q4_force_generic || (reinterpret_cast<uintptr_t>(out) & 15u)) {
        if (!settle()) return 0;
        const size_t waves = batch * rows;
        hipLaunchKernelGGL(q4_0_matmul_generic_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, g.stream,
                           static_cast<const uint8_t*>(w->raw), static_cast<const float*>(in),
                           static_cast<float*>(out), (uint32_t)batch, (uint32_t)rows, (uint32_t)cols,
                           (uint32_t)row_stride);
        return finish(sync);
    }

    // More than one turn of 64: all tokens in one launch.  (At 65 tokens it already takes no longer than the
    // two turns did: 43.8 against 43.0 us at 11264 x 2048, 28.7 against 35.1 at 2048 x 2048, 100 against 128
    // at 28672 x 4096.)
    if (batch > 64 && g.opt_q4_int_operand && g.opt_q4_ksplit == 0) {
        TokensArgs t{};
        t.q = static_cast<const uint2*>(w->q);
        t.d = static_cast<const _Float16*>(w->d);
        t.nblocks = (uint32_t)(cols / 32);
        if (matmul_tokens(false, t, static_cast<const float*>(in), static_cast<float*>(out), batch, rows, cols))
            return finish(sync);
    }

    // MFMA path, one pass over at most 64 requests at a time.
    const size_t nblocks = cols / 32, quads = (nblocks + 3) / 4;
    // (its workgroups read rows that others have not come to yet while the first ones store: only where the output lies apart)
    const bool rows_in = sync && g.opt_q4_int_operand && !feeds && !block_scales && aligned16(in) && q4_splits_rows(rows, cols, batch) &&
                         !overlap(in, batch * cols * 4, out, batch * rows * 4);
    for (size_t bo = 0; bo < batch; bo += 64) {
        const size_t bn = std::min<size_t>(64, batch - bo);
        const size_t bpad = (bn + 31) / 32 * 32;
        static const char* const frag_names[][2] = {{"q4_x_fragments", nullptr}, {"q4_x_fragments_silu", "q4_x_fragments_silu_2"},
                                                    {"q4_x_fragments_attention", nullptr}, {"q4_x_fragments_norm", "q4_x_fragments_norm_2"}};
        static const char* const scale_names[][2] = {{nullptr, nullptr}, {"q4_x_block_scales_silu", "q4_x_block_scales_silu_2"},
                                                     {"q4_x_block_scales_attention", nullptr}, {"q4_x_block_scales_norm", "q4_x_block_scales_norm_2"}};
        static const char* const ssq_names[] = {"q4_norm_partial_sums", "q4_norm_partial_sums_2"};
        _Float16* frag = static_cast<_Float16*>(cached_buffer(frag_names[x_from][x_set], bpad * cols * 4));
        float* inv = static_cast<float*>(cached_buffer("q4_x_inv_scale", 64 * 4));
        float* blk_scale = !block_scales ? nullptr : static_cast<float*>(cached_buffer(scale_names[x_from][x_set], bpad * nblocks * 4));
        float* ssq = feeds_rms ? static_cast<float*>(cached_buffer(ssq_names[x_set], nblocks * 64 * 4)) : nullptr;
        if (feeds_rms && !ssq) return fail("q4 matmul: scratch allocation failed");
        Q4Args norm{};   // (what this matmul needs to finish the norm)
        if (!frag || !inv || (block_scales && !blk_scale)) return fail("q4 matmul: scratch allocation failed");
        const float* xin = static_cast<const float*>(in) + bo * cols;
        float* o = static_cast<float*>(out) + bo * rows;
        if (feeds_silu) {
            g.gemm.a.split_frag = frag;
            g.gemm.a.split_blk_scale = blk_scale;
            if (!settle()) return 0;
        } else if (feeds_attn) {
            g.dec.a.split_frag = frag;
            g.dec.a.split_scale = blk_scale;
            if (!settle()) return 0;
        } else if (feeds_rms) {
            Ctx::GemmPending& m = g.gemm;
            const RowProgram& p = g.rows.p;
            m.a.add_resid = p.addend;
            m.a.add_out = p.add_out;
            m.a.add_gamma = p.rms_weight;
            m.a.add_n_gamma = p.n_weight;
            m.a.ssq_out = ssq;
            m.a.split_frag = frag;
            m.a.split_blk_scale = blk_scale;
            norm.ssq_in = ssq;
            norm.ssq_tiles = (uint32_t)nblocks;   // one partial per 32 columns of the norm's row
            norm.rms_len = (uint32_t)cols;
            norm.rms_eps = p.epsilon;
            norm.rms_src = p.add_out;
            norm.rms_out = p.rms_out;
            norm.rms_gamma = p.rms_weight;
            norm.rms_n_gamma = p.n_weight;
            g.rows.active = false;   // the two matmuls do the chain's work
            ++g.gemm_rms_fused;
            // It waits in front of this one, where the two may share a launch.  (Nothing else is pending.  The words' memory is taken now:
            // what launches the two later may be a call that allocates nothing.)
            if (!settle_front()) return 0;
            if (g.opt_q4_chain && batch <= kChainBatch && meeting_words("q4_link_words", kLinkBytes)) {
                m.active = false;
                g.front.active = true;
                g.front.block_scales = m.block_scales;
                static_cast<Q4Args&>(g.front.a) = m.a;
            } else if (!settle()) {
                return 0;
            }
        } else if (feeds) {  // the chain that produces the input also splits it (batch <= 64: one round)
            g.rows.p.frag = frag;
            g.rows.p.inv_scale = inv;
            g.rows.grid_rows = bn;
            if (!settle()) return 0;
        } else if (!rows_in) {
            launch_q4_split(xin, frag, inv, bn, cols);
        }
        // The slices' sums meet in the launch; a matmul that has no tag or no memory for that takes all of K.  (What was held
        // back has been launched, but for a matmul that waits in front of this one: that one takes no slices here, and
        // cached_buffer launches the other before it gives up a buffer.)
        Q4Slices split = feeds_rms ? Q4Slices{1, quads} : q4_slices(rows, cols, std::min<size_t>(batch, 64));
        uint64_t* words = nullptr;
        if (split.n > 1 && g.opt_q4_int_operand) {
            if (sliced_tags_left()) words = meeting_words("q4_k_meet", std::max<size_t>((split.n - 1) * bn * rows * 8, 2u << 20));
            if (!words) split = {1, quads};
        }
        const size_t ksplit = split.n, per_slice = split.quads;
        float* slices = ksplit > 1 && !words ? static_cast<float*>(cached_buffer("q4_k_slices", ksplit * bn * rows * 4)) : nullptr;
        if (ksplit > 1 && !slices && !words) return fail("q4 matmul: scratch allocation failed");
        Q4RopeArgs ra;
        Q4Args& a = ra;
        a = norm;
        a.q = static_cast<const uint4*>(w->q);
        a.d = static_cast<const uint2*>(w->d);
        a.xfrag = frag;
        a.blk_scale = blk_scale;
        a.inv_scale = inv;
        a.xrows = xin;
        a.out = slices ? slices : o;
        a.slices = (uint32_t)ksplit;
        a.meet = words;
        if (words) a.tags = next_sliced_tags();
        a.batch = (uint32_t)bn; a.rows = (uint32_t)rows; a.nblocks = (uint32_t)nblocks;
        a.nquads = (uint32_t)quads; a.quads_per_slice = (uint32_t)per_slice;
        if (g.opt_fuse_rows && g.opt_q4_int_operand && !sync && batch <= 64) {
            // held back for one call: a split + RoPE + cast of this output becomes the epilogue
            Ctx::GemmPending& m = g.gemm;
            m.active = true;
            m.silu = false;
            m.block_scales = block_scales;
            m.x_from = x_from;
            m.x_set = x_set;
            m.a = a;
            m.out = out;
            m.batch = batch;
            m.rows = rows;
            return finish(sync);
        }
        if (!g.opt_q4_int_operand) {
            const size_t z = (bn + 15) / 16, n_cu = (size_t)g.n_cu, pairs = rows / 64 * (z / 2) * ksplit;
            const int rt = rows / 16 * z * ksplit > 2 * n_cu ? 4 : 1, zt = rt == 4 && z % 2 == 0 && pairs * 8 >= n_cu * 5 ? 2 : 1;
            const auto kernel = zt == 2 ? q4_pairs_kernel<4, 2, 8> : rt == 4 ? q4_pairs_kernel<4, 1, 16> : q4_pairs_kernel<1, 1, 16>;
            hipLaunchKernelGGL(kernel, dim3((unsigned)(rows / 16 / rt), (unsigned)(z / zt), (unsigned)ksplit), dim3(zt == 2 ? 512 : 1024), 0,
                               g.stream, a);
        } else if (!launch_q4(rows_in ? kQ4Rows : kQ4Plain, block_scales || rows_in, ra)) {
            return 0;
        }
        if (slices) {
            const uint32_t n = (uint32_t)(bn * rows);
            if (g.opt_fuse_rows && batch <= 64 && rows <= 2 * kRowMaxLen) {
                // the sum over the slices starts the next chain: whatever row-local operator
                // consumes this matmul's output joins it
                rows_begin(slices, bn, rows);
                g.rows.p.n_slices = (uint32_t)ksplit;
                g.rows.p.slice_stride = n;
                g.rows.p.src_store = o;
                g.rows.cur = o;
            } else {
                hipLaunchKernelGGL(q4_sum_slices_kernel, dim3((n + 255) / 256), dim3(256), 0, g.stream, slices, o, n,
                                   (uint32_t)ksplit);
            }
        }
    }
    return finish(sync);
}

// ---- batched Q6_K matmul -------------------------------------------------------------------

namespace {

bool q6k_fast_shape(size_t rows, size_t cols, size_t row_stride) {
    // (the kernel addresses a tile's weights and a batch tile's fragments with 32 bits)
    return rows % 32 == 0 && cols % 256 == 0 && cols <= (1u << 24) && row_stride >= cols / 256 * 210;
}

// Uploads the weight matrix on first use of its name (or when its size changed); shapes the
// matrix-core kernel takes are also repacked (layout: q6k_matmul_kernels.h).
Ctx::Q6KWeight* q6k_weight(const char* name, const uint8_t* host, size_t bytes, size_t rows, size_t cols,
                           size_t stride) {
    Ctx::Q6KWeight& w = g.q6k_weights[name];
    if (w.raw && w.bytes == bytes && w.rows == rows && w.cols == cols && w.stride == stride) return &w;
    if (g_capturing) { fail("q6_k matmul: the weights are not on the device yet (run the pass once uncaptured first)"); return nullptr; }
    (void)hipStreamSynchronize(g.stream);
    for (void** p : {&w.raw, &w.qa, &w.sc, &w.d})
        if (*p) { (void)hipFree(*p); *p = nullptr; ++g.buffer_generation; }
    w = Ctx::Q6KWeight{};
    void* raw = nullptr;
    if (hipMalloc(&raw, bytes) != hipSuccess) { (void)hipGetLastError(); fail("q6_k matmul: hipMalloc failed"); return nullptr; }
    if (!upload_weights(raw, host, bytes)) { (void)hipFree(raw); fail("q6_k matmul: upload failed"); return nullptr; }
    w.raw = raw; w.bytes = bytes; w.rows = rows; w.cols = cols; w.stride = stride;
    if (q6k_fast_shape(rows, cols, stride)) {
        const size_t nb = cols / 256, tiles = rows / 32, groups = nb * 4;
        std::vector<uint8_t> qa(tiles * groups * 3 * 64 * 8);
        std::vector<uint8_t> sc(tiles * groups * 32 * 4);
        std::vector<uint16_t> d(tiles * nb * 32);
        for (size_t t = 0; t < tiles; ++t)
            for (size_t m = 0; m < 32; ++m) {
                const uint8_t* row = host + (t * 32 + m) * stride;
                for (size_t b = 0; b < nb; ++b) {
                    const uint8_t* blk = row + b * 210;
                    std::memcpy(&d[(t * nb + b) * 32 + m], blk + 208, 2);
                    for (size_t hi = 0; hi < 2; ++hi)
                        for (size_t l0i = 0; l0i < 2; ++l0i) {
                            const size_t gi = b * 4 + hi * 2 + l0i, tg = t * groups + gi;
                            for (size_t h = 0; h < 2; ++h) {
                                const size_t lane = h * 32 + m, l = l0i * 16 + h * 8;
                                std::memcpy(&qa[((tg * 3 + 0) * 64 + lane) * 8], blk + hi * 64 + l, 8);
                                std::memcpy(&qa[((tg * 3 + 1) * 64 + lane) * 8], blk + hi * 64 + 32 + l, 8);
                                std::memcpy(&qa[((tg * 3 + 2) * 64 + lane) * 8], blk + 128 + hi * 32 + l, 8);
                            }
                            for (size_t q = 0; q < 4; ++q) sc[(tg * 32 + m) * 4 + q] = blk[192 + hi * 8 + q * 2 + l0i];
                        }
                }
            }
        if (hipMalloc(&w.qa, qa.size()) != hipSuccess || hipMalloc(&w.sc, sc.size()) != hipSuccess ||
            hipMalloc(&w.d, d.size() * 2) != hipSuccess ||
            !upload_weights(w.qa, qa.data(), qa.size()) || !upload_weights(w.sc, sc.data(), sc.size()) ||
            !upload_weights(w.d, d.data(), d.size() * 2)) {
            (void)hipGetLastError();
            for (void* p : {w.raw, w.qa, w.sc, w.d})
                if (p) (void)hipFree(p);
            w = Ctx::Q6KWeight{};
            fail("q6_k matmul: repacked upload failed");
            return nullptr;
        }
    }
    return &w;
}

}  // namespace

int mlc_hip_matmul_q6_k_batched(const char* weight_name, const void* weights, size_t weight_bytes,
                                const void* in, size_t batch, size_t rows, size_t cols,
                                size_t row_stride, void* out, int sync) {
    if (!init_once()) return fail("GPU unavailable");
    if (!sync && !g.pass_open) return fail("encode: no open forward pass");
    if (!in || !out || batch == 0 || rows == 0 || cols == 0) return fail("q6_k matmul: null buffer or zero size");  // :6983
    if (cols < 64 || (rows % 4u) != 0) return fail("q6_k matmul: needs cols >= 64 and rows % 4 == 0");          // :6985
    if (!weight_name || !weights) return fail("q6_k matmul: null weights");
    const size_t nb = (cols + 255) / 256;
    if (row_stride < nb * 210 || weight_bytes < (rows - 1) * row_stride + nb * 210)
        return fail("q6_k matmul: weight bytes do not cover rows x row_stride");
    if (batch * rows > 0x7FFFFFFFull || batch * cols > 0x7FFFFFFFull) return fail("q6_k matmul: too many elements");
    const size_t ki = known_bytes(in), ko = known_bytes(out);
    if ((ki && batch * cols * 4 > ki) || (ko && batch * rows * 4 > ko)) return fail("q6_k matmul: buffer too small");
    const bool fast = q6k_fast_shape(rows, cols, row_stride) && !g.opt_q4_force_generic;
    const bool feeds = fast && batch <= 64 && row_len_ok(cols) && rows_continue(in, batch, cols);
    if (feeds ? !settle_before_rows() : !settle()) return 0;   // (a held-back matmul may read a buffer that is replaced below)
    Ctx::Q6KWeight* w = q6k_weight(weight_name, static_cast<const uint8_t*>(weights), weight_bytes, rows, cols, row_stride);
    if (!w) return 0;

    if (!fast || !w->qa) {
        if (!settle()) return 0;
        const size_t waves = batch * rows;
        hipLaunchKernelGGL(q6_k_matmul_generic_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, g.stream,
                           static_cast<const uint8_t*>(w->raw), static_cast<const float*>(in),
                           static_cast<float*>(out), (uint32_t)batch, (uint32_t)rows, (uint32_t)cols,
                           (uint32_t)row_stride);
        return finish(sync);
    }

    // more than one turn of 64: all tokens in one launch (65 tokens at 32000 x 2048: 72 us, two turns 94)
    if (batch > 64) {
        TokensArgs t{};
        t.q = static_cast<const uint2*>(w->qa);
        t.sc = static_cast<const uint32_t*>(w->sc);
        t.d = static_cast<const _Float16*>(w->d);
        t.nblocks = (uint32_t)(cols / 256);
        if (matmul_tokens(true, t, static_cast<const float*>(in), static_cast<float*>(out), batch, rows, cols))
            return finish(sync);
    }

    // matrix cores, at most 64 requests per pass
    for (size_t bo = 0; bo < batch; bo += 64) {
        const size_t bn = std::min<size_t>(64, batch - bo);
        const size_t bpad = (bn + 31) / 32 * 32;
        _Float16* frag = static_cast<_Float16*>(cached_buffer("q4_x_fragments", bpad * cols * 4));
        float* inv = static_cast<float*>(cached_buffer("q4_x_inv_scale", 64 * 4));
        if (!frag || !inv) return fail("q6_k matmul: scratch allocation failed");
        const float* xin = static_cast<const float*>(in) + bo * cols;
        if (feeds) {
            g.rows.p.frag = frag;
            g.rows.p.inv_scale = inv;
            g.rows.grid_rows = bn;
            if (!settle()) return 0;
        } else {
            launch_q4_split(xin, frag, inv, bn, cols);
        }
        Q6KArgs a;
        a.qa = static_cast<const uint2*>(w->qa);
        a.sc = static_cast<const uint32_t*>(w->sc);
        a.d = static_cast<const _Float16*>(w->d);
        a.xfrag = frag;
        a.inv_scale = inv;
        a.out = static_cast<float*>(out) + bo * rows;
        a.batch = (uint32_t)bn; a.rows = (uint32_t)rows; a.nblocks = (uint32_t)(cols / 256);
        launch_q6k_matmul(a, (size_t)g.n_cu, g.stream);
    }
    return finish(sync);
}

}  // extern "C"
