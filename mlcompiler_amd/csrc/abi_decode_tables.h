// Host side of the two decode kernels: the tables of the shape-agnostic kernel, what is remembered about the
// caller's page tables (content, largest page id, shared pages), their device copy, and the launch shape of the
// tile-balanced kernel (variant, stages, grid, pair cost, arithmetic mode, scratch ordering across streams).
//
// A section of the one translation unit mlc_hip.hip, which includes it once, in order, after the
// sections before it; not a header for anybody else.

namespace {

// ---------------------------------------------------------------- tables of the shape-agnostic decode kernel

bool plan_matches(const DecodePlan& p, const uint32_t* flat, size_t n_flat, const uint32_t* off,
                  const uint32_t* seq, const uint32_t* qpos, size_t B, int causal) {
    if (!p.valid || p.B != B || p.causal != causal) return false;
    if (p.pt_flat.size() != n_flat) return false;
    if (n_flat && std::memcmp(p.pt_flat.data(), flat, n_flat * 4) != 0) return false;
    if (std::memcmp(p.pt_off.data(), off, (B + 1) * 4) != 0) return false;
    if (std::memcmp(p.seq_lens.data(), seq, B * 4) != 0) return false;
    if (std::memcmp(p.q_pos.data(), qpos, B * 4) != 0) return false;
    return true;
}

// Brings the tables of the shape-agnostic kernel onto the device (cached, see DecodePlan).
int build_plan(const uint32_t* flat, size_t n_flat, const uint32_t* off, const uint32_t* seq,
               const uint32_t* qpos, size_t B, int causal) {
    DecodePlan& p = g.plan;
    if (plan_matches(p, flat, n_flat, off, seq, qpos, B, causal)) return 1;
    p.valid = false;
    p.pt_flat.assign(flat, flat + n_flat);
    p.pt_off.assign(off, off + B + 1);
    p.seq_lens.assign(seq, seq + B);
    p.q_pos.assign(qpos, qpos + B);
    p.B = B;
    p.causal = causal;
    std::vector<uint32_t> limits(B);
    for (size_t r = 0; r < B; ++r) {
        uint64_t lim = seq[r];
        if (causal && (uint64_t)qpos[r] + 1 < lim) lim = (uint64_t)qpos[r] + 1;  // :2286
        limits[r] = (uint32_t)lim;
    }
    p.off_ptoff = align_up(n_flat * 4, 16);
    p.off_limits = p.off_ptoff + align_up(B * 4, 16);
    const size_t total = p.off_limits + align_up(B * 4, 16);
    MetaSlot& s = g.plan_slots[g.plan_next];
    if (!slot_reserve(s, total)) return 0;
    char* h = static_cast<char*>(s.host);
    if (n_flat) std::memcpy(h, flat, n_flat * 4);
    std::memcpy(h + p.off_ptoff, off, B * 4);
    std::memcpy(h + p.off_limits, limits.data(), B * 4);
    if (!slot_upload(s, total)) return 0;
    p.slot = g.plan_next;
    g.plan_next = (g.plan_next + 1) % 4;
    p.valid = true;
    return 1;
}

// Largest page id a request actually dereferences, for bounds checks against
// pools this library allocated itself.
int check_pool_bounds(const void* pool, const uint32_t* flat, const uint32_t* off,
                      const uint32_t* seq, size_t B, size_t P, size_t row_bytes,
                      const char* what) {
    const size_t bytes = known_bytes(pool);
    if (!bytes) return 1;
    for (size_t r = 0; r < B; ++r) {
        const size_t pages = (seq[r] + P - 1) / P;
        for (size_t i = 0; i < pages; ++i) {
            const size_t end = ((size_t)flat[off[r] + i] + 1) * P * row_bytes;
            if (end > bytes) return fail(std::string(what) + ": page id beyond the pool");
        }
    }
    return 1;
}

// ---------------------------------------------------------------- tile-balanced decode

// Refreshes what is remembered about the caller's page tables: their content and the largest
// page id.  The device copy is brought up to date by tables_upload.
void tables_refresh(const uint32_t* flat, size_t n_flat, const uint32_t* off, size_t B) {
    StreamTables& t = g.tables;
    const bool same_flat = t.flat.size() == n_flat && (n_flat == 0 || std::memcmp(t.flat.data(), flat, n_flat * 4) == 0);
    if (!same_flat) {
        ++t.version;
        t.flat.assign(flat, flat + n_flat);
        t.max_page = 0;
        for (size_t i = 0; i < n_flat; ++i) t.max_page = std::max(t.max_page, flat[i]);
        t.shared_pages = -1;
    }
    if (t.off.size() != B + 1 || std::memcmp(t.off.data(), off, (B + 1) * 4) != 0) {
        t.off.assign(off, off + B + 1);
        t.shared_pages = -1;
    }
}

// Does some page id occur twice among the entries the requests own ([off[r], off[r+1]), a superset
// of what a call dereferences)?  Asked only by a call that would carry the step's KV write, and
// answered once per content: one pass over a table of stamps indexed by page id (2 us for 2 100
// pages, where sorting them took 60), or by sorting where the largest id makes that table too large
// (an id may be any 32-bit number: padding, or a corrupt entry that the bounds checks refuse).
bool tables_share_pages() {
    StreamTables& t = g.tables;
    if (t.shared_pages >= 0) return t.shared_pages != 0;
    const size_t n_flat = t.flat.size(), B = t.off.size() - 1;
    bool shared = false;
    constexpr uint32_t kMostStamps = 1u << 22;
    if (n_flat && t.max_page < kMostStamps) {
        if (t.stamps.size() <= t.max_page) t.stamps.resize((size_t)t.max_page + 1, 0);
        if (++t.stamp == 0) {
            std::fill(t.stamps.begin(), t.stamps.end(), 0u);
            t.stamp = 1;
        }
        for (size_t r = 0; r < B && !shared; ++r) {
            const size_t e = std::min<size_t>(t.off[r + 1], n_flat);
            for (size_t i = t.off[r]; i < e; ++i) {
                uint32_t& st = t.stamps[t.flat[i]];
                shared |= st == t.stamp;
                st = t.stamp;
            }
        }
    } else {
        std::vector<uint32_t> owned;
        for (size_t r = 0; r < B; ++r) {
            const size_t b0 = std::min<size_t>(t.off[r], n_flat), e = std::min<size_t>(t.off[r + 1], n_flat);
            if (e > b0) owned.insert(owned.end(), t.flat.begin() + b0, t.flat.begin() + e);
        }
        std::sort(owned.begin(), owned.end());
        shared = std::adjacent_find(owned.begin(), owned.end()) != owned.end();
    }
    t.shared_pages = shared ? 1 : 0;
    return shared;
}

// Makes the device copy of the flat table (and of the per-request arrays when `meta3` is
// given: seq_lens | q_positions | offsets, B each) current.  Returns the device pointer of the
// table in *d_flat and of the arrays in *d_meta.  The arrays sit behind room for twice the
// table's entries (at least 16 Ki), so that a table that grows by a page now and then keeps both
// addresses.
int tables_upload(const uint32_t* meta3, size_t B, const uint32_t** d_flat, const uint32_t** d_meta) {
    StreamTables& t = g.tables;
    const size_t n_flat = t.flat.size();
    const size_t meta_bytes = meta3 ? 3 * B * 4 : 0;
    size_t flat_room = t.meta_off;
    if (n_flat * 4 > flat_room) flat_room = align_up(std::max<size_t>(2 * n_flat, 16384) * 4, 256);
    const size_t total = flat_room + std::max<size_t>(meta_bytes, 3 * 4096 * 4);
    bool upload = t.uploaded != t.version || !t.filled || flat_room != t.meta_off;
    if (meta3) {
        if (t.meta.size() != 3 * B || std::memcmp(t.meta.data(), meta3, meta_bytes) != 0) upload = true;
    }
    if (upload) {
        NOT_WHILE_CAPTURING("copying the decode tables to the device (run the pass once uncaptured first)");
        if (total > t.cap) {
            if (!wait_stream()) return 0;
            if (t.dev) HIP_OK(hipFree(t.dev));
            if (t.dev) ++g.buffer_generation;
            t.dev = nullptr;
            t.cap = 0;
            HIP_OK(hipMalloc(&t.dev, total));
            t.cap = total;
        }
        MetaSlot& s = g.ring[g.ring_next];
        g.ring_next = (g.ring_next + 1) % 8;
        const size_t flat_stage = align_up(n_flat * 4, 16);   // the staging slot holds the two side by side
        if (!slot_reserve(s, flat_stage + meta_bytes)) return 0;
        char* h = static_cast<char*>(s.host);
        if (n_flat) std::memcpy(h, t.flat.data(), n_flat * 4);
        if (meta3) {
            std::memcpy(h + flat_stage, meta3, meta_bytes);
            t.meta.assign(meta3, meta3 + 3 * B);
            // table and arrays in two copies: what lies between them on the device is not sent
            if (n_flat) HIP_OK(hipMemcpyAsync(t.dev, h, n_flat * 4, hipMemcpyHostToDevice, g.stream));
            HIP_OK(hipMemcpyAsync(static_cast<char*>(t.dev) + flat_room, h + flat_stage, meta_bytes,
                                  hipMemcpyHostToDevice, g.stream));
        } else {
            t.meta.clear();
            if (n_flat) HIP_OK(hipMemcpyAsync(t.dev, h, n_flat * 4, hipMemcpyHostToDevice, g.stream));
        }
        slot_mark(s);
        t.filled = true;
        t.uploaded = t.version;
        t.meta_off = flat_room;
        ++g.table_uploads;
    }
    const char* dev = static_cast<const char*>(t.dev);
    *d_flat = reinterpret_cast<const uint32_t*>(dev);
    *d_meta = meta3 ? reinterpret_cast<const uint32_t*>(dev + t.meta_off) : nullptr;
    return 1;
}

// The same for a launch whose per-request arrays travel in its arguments: a table that is already on
// the device is read there (*d_copy null); a new one is put into pinned host memory, where the launch
// reads the few ids each workgroup needs and from where it also fills the device copy for the launches
// behind it (`threads` of it, one word each).  The reads across the bus cost the launch 1.4 us (28.0
// against 26.6 us at 64 requests with 2 100 pages), where a copy in front of it cost 6 to 9 us per call.
int tables_stage(size_t threads, const uint32_t** d_flat, uint32_t** d_copy) {
    StreamTables& t = g.tables;
    const size_t n_flat = t.flat.size();
    *d_copy = nullptr;
    const uint32_t* none = nullptr;
    const bool current = t.uploaded == t.version && t.filled && n_flat * 4 <= t.meta_off;
    // (no device copy to fill yet, or one that is too small: tables_upload makes it)
    if (current || n_flat * 4 > t.meta_off || n_flat > threads) return tables_upload(nullptr, 0, d_flat, &none);
    MetaSlot& s = t.stage[t.stage_next];
    t.stage_next = (t.stage_next + 1) % 4;
    if (!slot_reserve(s, n_flat * 4)) return 0;
    std::memcpy(s.host, t.flat.data(), n_flat * 4);
    slot_mark(s);
    void* mapped = nullptr;
    HIP_OK(hipHostGetDevicePointer(&mapped, s.host, 0));
    *d_flat = static_cast<const uint32_t*>(mapped);
    *d_copy = static_cast<uint32_t*>(t.dev);
    t.meta.clear();
    t.uploaded = t.version;
    ++g.table_uploads;
    return 1;
}

// Shape of the tile-balanced launch for (G, D): query heads per wave, waves per workgroup;
// false when the kernel does not cover the shape.  On the matrix pipe every ratio up to 16 runs with
// four waves, each with room for 1, 2 or 4 heads in the epilogue.  One or two query heads per KV head
// over pages of whole tiles run on the vector pipe, in workgroups of one or two waves: it multiplies the
// fp32 numbers themselves and comes closer to float64 (2.3e-7 .. 4.4e-7 against 2.8e-7 .. 5.1e-7 of the
// output at 6 000 to 8 000 tokens), although the matrix pipe is faster (31.2 against 28.5 us a call at 32
// requests of 16 / 8 heads of 64, 44.8 against 44.1 at 8 of 32 / 16 of 128, 84.8 against 69.5 at 8 of
// 32 / 32 of 128).
// The choice depends on the shape alone: a captured pass keeps its kernel while the contexts grow, and gives
// what the same step gives when it is encoded call by call.
bool stream_variant(size_t G, size_t D, size_t P, int* hpw_out, int* nw_out) {
    if (D != 64 && D != 128) return false;
    const bool vector_pipe = G <= 2 && P % (D == 64 ? 64 : 32) == 0;
    if (g.opt_decode_mfma && g.opt_hpw_max == 0 && G >= 1 && G <= 16 && !vector_pipe) {
        *hpw_out = G <= 4 ? 1 : G <= 8 ? 2 : 4;
        *nw_out = 4;
        return true;
    }
    const long hpw_cap = g.opt_hpw_max > 0 ? g.opt_hpw_max : std::max<long>(1, (long)G / 4);
    int hpw = 8;
    while (hpw > 1 && (hpw > hpw_cap || (G % (size_t)hpw) != 0)) hpw >>= 1;
    size_t nw = G / (size_t)hpw;
    if (nw > 4 || nw == 3) {
        hpw = 8;
        while (hpw > 1 && (G % (size_t)hpw) != 0) hpw >>= 1;
        nw = G / (size_t)hpw;
    }
    if (nw > 4 || nw == 3) return false;
    *hpw_out = hpw;
    *nw_out = (int)nw;
    return true;
}

// LDS stages of the tile-balanced kernel.  Two by default: swept over 2..4 stages and 1..5
// workgroups per CU on MI355X, in both arithmetic modes, two stages and two workgroups per CU
// were fastest at 38 MB and at 1.2 GB of KV per launch (deeper stages only delay the first tile
// of every workgroup).  Batches above 64 requests keep their per-request figures in LDS as well
// and take three stages at most.
int stream_stages(size_t batch) {
    const int most = batch <= 64 ? 4 : 3;
    int nbuf = 2;
    if (g.opt_stream_stages > 0) nbuf = (int)std::min<long>(g.opt_stream_stages, most);
    return nbuf;
}

// Grid of the tile-balanced kernel: as many workgroups as stay resident (LDS decides), within
// what the scratch array holds.
unsigned stream_grid(int hpw, int nw, size_t D, int nbuf, size_t dyn_lds) {
    const size_t GP = (size_t)hpw * nw;
    const bool matrix_pipe = g.opt_decode_mfma && nw == 4 && GP <= 16;
    const size_t lds = stream_static_lds_bytes(nbuf, GP, D, matrix_pipe) + dyn_lds;
    size_t per_cu = std::max<size_t>(1, std::min<size_t>(160 * 1024 / lds, 2));
    if (g.opt_wgs_per_cu > 0) per_cu = (size_t)g.opt_wgs_per_cu;
    size_t W = (size_t)g.n_cu * per_cu;
    if (g.opt_grid_wgs > 0) W = (size_t)g.opt_grid_wgs;
    W = std::min<size_t>(W, kStreamMaxWgs);
    W = std::min<size_t>(W, kStreamPartBytes / stream_partial_bytes(GP, D, (size_t)nw));
    return (unsigned)std::max<size_t>(W, 1);
}

uint32_t stream_pair_cost(int nw) {
    if (g.opt_pair_cost >= 0) return (uint32_t)g.opt_pair_cost;
    return nw == 4 ? 2u : 0u;
}

// Page sizes the tile-balanced kernel takes: pages of whole tiles (TT = 64 tokens at head_dim 64, 32 at
// 128), and on the matrix pipe also pages that divide a tile into the slices of one or more of its four
// waves (16 and 32 tokens at head_dim 64, 8 and 16 at 128).
bool stream_page_ok(size_t D, size_t P, int hpw, int nw) {
    const size_t tile = D == 64 ? 64 : 32;
    if (P % tile == 0) return true;
    const bool matrix_pipe = g.opt_decode_mfma && nw == 4 && hpw * nw <= 16;
    return matrix_pipe && tile % P == 0 && P >= tile / 4;
}

// Arithmetic mode of the tile-balanced kernel: 0 fp32 softmax weights, 1 fp16 weights on the vector
// pipe, 2 matrix pipe (4 waves per workgroup, at most 16 heads per KV head).
int stream_pv_mode(int hpw, int nw) {
    const bool matrix_pipe = g.opt_decode_mfma && nw == 4 && hpw * nw <= 16;
    if (!g.opt_pv_fp16) return matrix_pipe ? 3 : 0;
    return matrix_pipe ? 2 : 1;
}
const char* stream_pv_name(int hpw, int nw) {
    const int m = stream_pv_mode(hpw, nw);
    return m == 3 ? "mfma-p32" : m == 2 ? "mfma" : m == 1 ? "pv16" : "pv32";
}

// Orders a launch whose workgroups wait for each other on `stream` behind the last one (see
// Ctx::scratch_stream).  The library's own stream lives as long as the library, so the event that
// marks its last launch is recorded only when another stream shows up; a caller's stream may be
// gone by then, so the event is recorded right behind a launch on one.  A captured pass runs on
// the library's stream, where its replays are ordered like any other launch there.  (A launch that a caller records into
// a graph of its own does not run now: when that graph runs is the caller's to order.)
bool caller_records(hipStream_t stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(stream, &status) == hipSuccess && status != hipStreamCaptureStatusNone;
}
int scratch_follow(hipStream_t stream) {
    if (g_capturing || (stream != g.stream && caller_records(stream))) return 1;
    if (g.scratch_in_use && g.scratch_stream != stream) {
        if (g.scratch_stream == g.stream) HIP_OK(hipEventRecord(g.scratch_ev, g.stream));
        HIP_OK(hipStreamWaitEvent(stream, g.scratch_ev, 0));
    }
    return 1;
}
int scratch_launched(hipStream_t stream) {
    if (g_capturing || (stream != g.stream && caller_records(stream))) return 1;
    g.scratch_stream = stream;
    g.scratch_in_use = true;
    if (stream != g.stream) HIP_OK(hipEventRecord(g.scratch_ev, stream));
    return 1;
}

bool launch_stream_variant(size_t D, int hpw, int nw, int nbuf, const StreamArgs& a, unsigned n_wg, size_t dyn_lds,
                           hipStream_t stream) {
    if (!scratch_follow(stream)) return false;
    const int pvm = stream_pv_mode(hpw, nw);
    bool launched = false;
#define MLC_CASE(d, h) \
    if (D == d && hpw == h) launched = launch_decode_stream_##d##_##h(nw, nbuf, pvm, a, n_wg, dyn_lds, stream);
    MLC_CASE(64, 1) MLC_CASE(64, 2) MLC_CASE(64, 4) MLC_CASE(64, 8)
    MLC_CASE(128, 1) MLC_CASE(128, 2) MLC_CASE(128, 4) MLC_CASE(128, 8)
#undef MLC_CASE
    if (!launched) g.tables.filled = false;   // (it may have been the launch that fills the tables' device copy)
    return launched && scratch_launched(stream);
}

void stream_fill_common(StreamArgs& a, const void* q, const void* k_pages, const void* v_pages, void* o,
                        size_t B, size_t H, size_t Hkv, size_t D, size_t P, int causal) {
    a.q = static_cast<const float*>(q);
    a.k_pages = static_cast<const uint4*>(k_pages);
    a.v_pages = static_cast<const uint4*>(v_pages);
    a.o = static_cast<float*>(o);
    a.part = reinterpret_cast<uint64_t*>(g.scratch_ptr);
    const TagArgs tags = next_tags(g.cap.n_decode);
    a.fault = tags.fault;
    a.spin_limit = tags.spin_limit;
    a.test_flags = tags.test_flags;
    a.tag = tags.tag;
    a.tag_dev = tags.tag_dev;
    a.batch = (uint32_t)B;
    a.num_heads = (uint32_t)H;
    a.kv_heads = (uint32_t)Hkv;
    a.page_size = (uint32_t)P;
    a.group = (uint32_t)(H / Hkv);
    const size_t tile = D == 64 ? 64 : 32;
    a.pages_per_tile = P < tile ? (uint32_t)(tile / P) : 1u;
    a.page_shift = (uint32_t)__builtin_ctzll(P);
    a.causal = causal ? 1u : 0u;
    a.capacity_pages = 0;
    a.meta = nullptr;
    a.meta_stride = 0;
    a.scale_log2e = (1.0f / std::sqrt(static_cast<float>(D))) * 1.44269504088896340736f;
    a.pair_cost = 0;  // (set by the caller once the workgroup shape is known: stream_pair_cost)
    a.new_k = a.new_v = nullptr;
    a.split_frag = nullptr;
    a.split_scale = nullptr;
    a.pt_copy = nullptr;
    a.pt_words = 0;
}

}  // namespace
