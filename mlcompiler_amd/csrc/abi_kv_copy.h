// Entry points that move K/V rows between the caller's buffers and the paged pools: batched scatter,
// multi-token scatter, gather.
//
// A section of the one translation unit mlc_hip.hip, which includes it once, in order, after the
// sections before it; not a header for anybody else.

namespace {

template <typename UnitT, bool TO_PAGES>
void launch_kv_copy(const KvCopyArgs& a) {
    const size_t total = (size_t)a.n_kv_heads * a.tokens * a.head_units;
    const bool wide = total >= 256 * 8 * (size_t)g.n_cu;
    const size_t per_wg = wide ? 1024 : 256;
    const dim3 grid((unsigned)((total + per_wg - 1) / per_wg)), block(256);
    if (total > 0x7FFF0000ull) hipLaunchKernelGGL((kv_copy_kernel<UnitT, TO_PAGES, 4, uint64_t>), grid, block, 0, g.stream, a);
    else if (wide) hipLaunchKernelGGL((kv_copy_kernel<UnitT, TO_PAGES, 4, uint32_t>), grid, block, 0, g.stream, a);
    else hipLaunchKernelGGL((kv_copy_kernel<UnitT, TO_PAGES, 1, uint32_t>), grid, block, 0, g.stream, a);
}

// The multi-token copies between contiguous rows and pages.
template <bool TO_PAGES>
int kv_copy(const void* src, void* dst, const uint32_t* page_table, size_t pages, size_t page_size, size_t n_kv_heads,
            size_t head_dim, size_t tokens, size_t start_slot, size_t dtype_bytes) {
    KvCopyArgs a;
    a.src = src;
    a.dst = dst;
    a.page_table = nullptr;
    a.n_kv_heads = (uint32_t)n_kv_heads;
    a.tokens = (uint32_t)tokens;
    a.page_size = (uint32_t)page_size;
    a.start_slot = (uint32_t)start_slot;
    if (pages <= kKvCopyEmbPages) {
        std::memcpy(a.emb_table, page_table, pages * 4);
    } else {
        MetaSlot& s = g.ring[g.ring_next];
        g.ring_next = (g.ring_next + 1) % 8;
        if (!slot_reserve(s, pages * 4)) return 0;
        std::memcpy(s.host, page_table, pages * 4);
        if (!slot_upload(s, pages * 4)) return 0;
        slot_mark(s);
        a.page_table = static_cast<const uint32_t*>(s.dev);
    }
    const size_t head_bytes = head_dim * dtype_bytes;
    if ((head_bytes % 16) == 0 && aligned16(src) && aligned16(dst)) {
        a.head_units = (uint32_t)(head_bytes / 16);
        launch_kv_copy<copy_u32x4, TO_PAGES>(a);
    } else {
        a.head_units = (uint32_t)head_dim;
        if (dtype_bytes == 4) launch_kv_copy<uint32_t, TO_PAGES>(a);
        else launch_kv_copy<uint16_t, TO_PAGES>(a);
    }
    return finish(1);
}

}  // namespace

extern "C" {

int mlc_hip_scatter_kv_paged_batched_f16(void* page_storage, const uint32_t* page_ids,
                                         const uint32_t* slots_in_page, size_t page_size_tokens,
                                         size_t n_kv_heads, size_t head_dim, size_t batch,
                                         const void* src, int sync) {
    if (!init_once()) return fail("GPU unavailable");
    if (!sync && !g.pass_open) return fail("encode: no open forward pass");  // :7178
    // metal_runtime.mm:7241-7243
    if (!page_storage || !src) return fail("scatter: null buffer");
    if (batch == 0 || n_kv_heads == 0 || head_dim == 0 || page_size_tokens == 0)
        return fail("scatter: zero dimension");
    if (!page_ids || !slots_in_page) return fail("scatter: null metadata");
    const size_t row_bytes = n_kv_heads * head_dim * 2;
    if (batch * row_bytes / 2 > 0x7FFFFFFFull) return fail("scatter: too many elements");
    // Beyond the reference: a slot outside the page would land in the next page.
    for (size_t r = 0; r < batch; ++r)
        if (slots_in_page[r] >= page_size_tokens) return fail("scatter: slot >= page size");
    const size_t known = known_bytes(page_storage);
    if (known) {
        for (size_t r = 0; r < batch; ++r)
            if (((size_t)page_ids[r] + 1) * page_size_tokens * row_bytes > known)
                return fail("scatter: page id beyond the pool");
    }
    const size_t known_src = known_bytes(src);
    if (known_src && batch * row_bytes > known_src) return fail("scatter: src too small");

    const bool wide = (row_bytes % 16) == 0 && aligned16(page_storage) && aligned16(src);
    Ctx::KvPending& kv = g.kv;
    // ---- does this scatter complete a pending KV write?  (only while nothing younger is pending)
    if (g.opt_fuse_rows && kv.active && !g.rows.active && kv.batch == batch && kv.row_elems == row_bytes / 2 &&
        (kv.ids.empty() || (kv.page_size == page_size_tokens &&
                            std::memcmp(kv.ids.data(), page_ids, batch * 4) == 0 &&
                            std::memcmp(kv.slots.data(), slots_in_page, batch * 4) == 0))) {
        bool joined = false;
        if (kv.rope) {
            const bool as_k = src == kv.a.k_f16 && !kv.a.k_pages && kv.a.k_rows == row_bytes / 2;
            const bool as_v = !as_k && src == kv.a.v_f16 && !kv.a.v_pages && kv.a.v_rows == row_bytes / 2;
            if ((as_k || as_v) && (reinterpret_cast<uintptr_t>(page_storage) & 3u) == 0) {
                if (kv.ids.empty()) {
                    kv.a.page_size = (uint32_t)page_size_tokens;
                    kv.page_size = page_size_tokens;
                    kv.ids.assign(page_ids, page_ids + batch);
                    kv.slots.assign(slots_in_page, slots_in_page + batch);
                }
                (as_k ? kv.a.k_pages : kv.a.v_pages) = static_cast<_Float16*>(page_storage);
                joined = true;
            }
        } else if (kv.n == 1 && kv.wide == wide && page_storage != kv.pages[0]) {
            kv.src[1] = src;
            kv.pages[1] = page_storage;
            kv.n = 2;
            joined = true;
        }
        if (joined) return finish(sync);
    }
    if (!settle()) return 0;

    kv = Ctx::KvPending{};
    kv.active = true;
    kv.src[0] = src;
    kv.pages[0] = page_storage;
    kv.n = 1;
    kv.wide = wide;
    kv.ids.assign(page_ids, page_ids + batch);
    kv.slots.assign(slots_in_page, slots_in_page + batch);
    kv.batch = batch;
    kv.row_elems = row_bytes / 2;
    kv.page_size = page_size_tokens;
    if (!g.opt_fuse_rows && !settle_kv()) return 0;  // no deferral: launched as encoded
    return finish(sync);
}

int mlc_hip_scatter_kv_paged(void* page_storage, const uint32_t* page_table, size_t n_page_table,
                             size_t page_size_tokens, size_t n_kv_heads, size_t head_dim,
                             size_t tokens, size_t start_slot, const void* src,
                             size_t dtype_bytes) {
    if (!init_once()) return fail("GPU unavailable");
    NOT_WHILE_CAPTURING("one-request scatter (it waits)");
    if (!settle()) return 0;
    // metal_runtime.mm:7839-7845
    if (!page_storage || !src) return fail("scatter_paged: null buffer");
    if (page_size_tokens == 0 || n_kv_heads == 0 || head_dim == 0 || tokens == 0)
        return fail("scatter_paged: zero dimension");
    if (dtype_bytes != 2 && dtype_bytes != 4) return fail("scatter_paged: dtype_bytes");
    if (start_slot >= page_size_tokens) return fail("scatter_paged: start_slot >= page size");
    const size_t needed = (start_slot + tokens + page_size_tokens - 1) / page_size_tokens;
    if (n_page_table < needed || !page_table) return fail("scatter_paged: page table too short");
    const size_t row_bytes = n_kv_heads * head_dim * dtype_bytes;
    const size_t known = known_bytes(page_storage);
    if (known)
        for (size_t i = 0; i < needed; ++i)
            if (((size_t)page_table[i] + 1) * page_size_tokens * row_bytes > known)
                return fail("scatter_paged: page id beyond the pool");
    const size_t known_src = known_bytes(src);
    if (known_src && tokens * row_bytes > known_src) return fail("scatter_paged: src too small");

    return kv_copy<true>(src, page_storage, page_table, needed, page_size_tokens, n_kv_heads, head_dim, tokens, start_slot, dtype_bytes);
}

int mlc_hip_gather_kv_pages(const void* page_storage, const uint32_t* page_table,
                            size_t n_page_table, size_t page_size_tokens, size_t n_kv_heads,
                            size_t head_dim, size_t num_tokens, void* dst, size_t dtype_bytes) {
    if (!init_once()) return fail("GPU unavailable");
    NOT_WHILE_CAPTURING("gather (it waits)");
    if (!settle()) return 0;
    // metal_runtime.mm:7657-7662
    if (!page_storage || !dst) return fail("gather: null buffer");
    if (page_size_tokens == 0 || n_kv_heads == 0 || head_dim == 0 || num_tokens == 0)
        return fail("gather: zero dimension");
    if (dtype_bytes != 2 && dtype_bytes != 4) return fail("gather: dtype_bytes");
    const size_t needed = (num_tokens + page_size_tokens - 1) / page_size_tokens;
    if (n_page_table < needed || !page_table) return fail("gather: page table too short");
    const size_t row_bytes = n_kv_heads * head_dim * dtype_bytes;
    const size_t known = known_bytes(page_storage);
    if (known)
        for (size_t i = 0; i < needed; ++i)
            if (((size_t)page_table[i] + 1) * page_size_tokens * row_bytes > known)
                return fail("gather: page id beyond the pool");
    const size_t known_dst = known_bytes(dst);
    if (known_dst && num_tokens * row_bytes > known_dst) return fail("gather: dst too small");

    return kv_copy<false>(page_storage, dst, page_table, needed, page_size_tokens, n_kv_heads, head_dim, num_tokens, 0, dtype_bytes);
}

}  // extern "C"
