// What a workgroup of q4_matmul_kernel does, described there: the body of the kernel and of q4_matmul_workgroup
// (q4_matmul_mfma.h), which include it where it stands.  Its template parameters are NI, RT, WAVES, BS, FORM, ZT, LINK and QUADS; it reads
// the arguments w_q .. batch_z, a and link, block_x and slice (the workgroup's place), rope_args_offset and the
// LDS arrays red, scales, packed and rms_scale.
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
