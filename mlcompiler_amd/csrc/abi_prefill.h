// Entry point of the chunked prefill attention over paged KV.
//
// A section of the one translation unit mlc_hip.hip, which includes it once, in order, after the
// sections before it; not a header for anybody else.

extern "C" {

int mlc_hip_paged_attn_prefill(const void* q_f16, const void* k_pages, const void* v_pages,
                               void* o, const uint32_t* page_tables_flat, size_t n_flat,
                               const uint32_t* page_table_offsets, const uint32_t* seq_lens,
                               const uint32_t* q_start, size_t batch, size_t chunk,
                               size_t num_heads, size_t kv_heads, size_t head_dim,
                               size_t page_size_tokens, int sync) {
    if (!init_once()) return fail("GPU unavailable");
    if (!settle()) return 0;
    if (!sync && !g.pass_open) return fail("encode: no open forward pass");
    if (!q_f16 || !k_pages || !v_pages || !o) return fail("prefill: null buffer");
    if (batch == 0 || chunk == 0 || num_heads == 0 || head_dim == 0 || page_size_tokens == 0)
        return fail("prefill: zero dimension");
    if (kv_heads == 0 || (num_heads % kv_heads) != 0) return fail("prefill: heads % kv_heads != 0");
    if (!page_table_offsets || !seq_lens || !q_start) return fail("prefill: null metadata");
    if (n_flat && !page_tables_flat) return fail("prefill: null page table");
    if (n_flat < page_table_offsets[batch]) return fail("prefill: page table shorter than offsets");
    for (size_t r = 0; r < batch; ++r) {
        const size_t pages = ((size_t)seq_lens[r] + page_size_tokens - 1) / page_size_tokens;
        if ((size_t)page_table_offsets[r] + pages > n_flat)
            return fail("prefill: page table does not cover seq_len");
    }
    {
        const size_t rows = batch * chunk * num_heads * head_dim;
        const size_t kq = known_bytes(q_f16), ko = known_bytes(o);
        if ((kq && rows * 2 > kq) || (ko && rows * 4 > ko)) return fail("prefill: q / o buffer too small");
    }
    const size_t row_bytes = kv_heads * head_dim * 2;
    if (!check_pool_bounds(k_pages, page_tables_flat, page_table_offsets, seq_lens, batch,
                           page_size_tokens, row_bytes, "prefill K") ||
        !check_pool_bounds(v_pages, page_tables_flat, page_table_offsets, seq_lens, batch,
                           page_size_tokens, row_bytes, "prefill V"))
        return 0;
    if (!prefill_shape_supported(head_dim, page_size_tokens, num_heads, kv_heads) || !aligned16(q_f16) ||
        !aligned16(k_pages) || !aligned16(v_pages) || !aligned16(o))
        return fail("prefill: unsupported shape (head_dim 64 or 128, page size a multiple of 32, heads/kv_heads in {1,2,4,8}, 16-byte aligned buffers)");

    // The tables travel inside the kernel arguments, or, where they are too large for those, are read from
    // pinned host memory: a workgroup takes 64 page ids at a time, which is nothing against the tiles
    // behind them, while a copy to the device is 6 us in front of every call.
    NOT_WHILE_CAPTURING("prefill (its tables change with every call)");
    PrefillArgs a;
    a.tables = nullptr;
    uint32_t* t = a.emb;
    const size_t words = 3 * batch + n_flat;
    if (words > kPrefillEmbWords) {
        MetaSlot& s = g.ring[g.ring_next];
        g.ring_next = (g.ring_next + 1) % 8;
        if (!slot_reserve(s, words * 4)) return 0;
        t = static_cast<uint32_t*>(s.host);
        void* mapped = nullptr;
        HIP_OK(hipHostGetDevicePointer(&mapped, s.host, 0));
        a.tables = static_cast<const uint32_t*>(mapped);
        slot_mark(s);
    }
    std::memcpy(t, page_table_offsets, batch * 4);
    std::memcpy(t + batch, seq_lens, batch * 4);
    std::memcpy(t + 2 * batch, q_start, batch * 4);
    if (n_flat) std::memcpy(t + 3 * batch, page_tables_flat, n_flat * 4);
    a.q = static_cast<const _Float16*>(q_f16);
    a.k_pages = static_cast<const _Float16*>(k_pages);
    a.v_pages = static_cast<const _Float16*>(v_pages);
    a.o = static_cast<float*>(o);
    a.batch = (uint32_t)batch;
    a.chunk = (uint32_t)chunk;
    a.num_heads = (uint32_t)num_heads;
    a.kv_heads = (uint32_t)kv_heads;
    a.page_size = (uint32_t)page_size_tokens;
    a.scale_log2e = (1.0f / std::sqrt(static_cast<float>(head_dim))) * 1.44269504088896340736f;
    a.row_blocks = 0;  // set by the launcher
    size_t max_tiles = 0;
    for (size_t r = 0; r < batch; ++r)
        max_tiles = std::max(max_tiles, (std::min<size_t>(seq_lens[r], q_start[r] + chunk) + kPfKeys - 1) / kPfKeys);
    // (one size for good: a buffer that grows ends captured passes.  A workgroup of 256 rows per CU fits, 34 MB)
    constexpr size_t kPartBytes = 36u << 20;
    const size_t wgs = prefill_wgs(batch, chunk, num_heads, kv_heads);
    uint32_t splits = prefill_splits(wgs, head_dim, max_tiles, g.n_cu, kPartBytes);
    a.part_o = splits > 1 ? static_cast<float4*>(cached_buffer("prefill_parts", kPartBytes)) : nullptr;
    if (!a.part_o) splits = 1;
    a.part_ml = reinterpret_cast<float2*>(a.part_o + (splits > 1 ? splits * wgs * kPfWaves * kPfRows * head_dim / 4 : 0));
    const bool rows64 = g.opt_prefill_rows64 &&
                        (num_heads / kv_heads < 8 || prefill_rows64_ratio8(head_dim, max_tiles, chunk, batch * kv_heads, (size_t)g.n_cu));
    launch_prefill(a, head_dim, (int)g.opt_prefill_stages, rows64, splits, g.stream);
    return finish(sync);
}

}  // extern "C"
