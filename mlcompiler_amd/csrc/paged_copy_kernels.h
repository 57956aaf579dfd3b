// Paged KV write / read kernels for gfx950: the batched one-row-per-request
// scatter of the decode step and the single-request multi-token scatter / gather
// that sit either side of it.  All of them are pure copies (bit-exact by
// construction); the only design point is that a token row of all KV heads is
// contiguous in a page, so rows move as 16-byte chunks with coalesced stores.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mlc_hip {

// MSL scatter_kv_paged_batched_f16 (compiler/runtime/metal_runtime.mm:405-424):
//   page[page_ids[r]][slots[r]][kv][d] = src[r][kv][d].
// src row r (n_kv_heads*head_dim halves) and its destination row are both contiguous, so the copy
// runs in units of 16 bytes when everything is 16-byte aligned, else of 2.
// The K row and the V row of a decode step in one launch: two scatter_kv_paged_batched copies
// with the same (page id, slot) per request.  The batched step encodes them back to back
// (compiler/runtime/batched_walker.cpp:304-307); each on its own costs a launch for 32 KiB.
// The page row of every request travels inside the kernel arguments for up to kScatterEmbBatch
// requests, so that a call copies nothing to the device.
static constexpr size_t kScatterEmbBatch = 256;
struct ScatterPairArgs {
    const void* src[2];
    void* pages[2];
    const uint64_t* page_rows;  // [batch] page_id * page_size + slot on the device, or null: emb_rows
    uint32_t batch, row_units, n_tensors;
    uint64_t emb_rows[kScatterEmbBatch];
};
template <typename UnitT>
__global__ void scatter_kv_pair_kernel(const ScatterPairArgs a) {
    // n_tensors = 1: only the first copy exists (src[1] / pages[1] are null and must not be touched)
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t per = a.batch * a.row_units;
    if (gid >= a.n_tensors * per) return;
    const uint32_t which = gid / per, e = gid - which * per;
    const uint32_t req = e / a.row_units;
    const uint32_t u = e - req * a.row_units;
    const uint64_t dst_row = a.page_rows ? a.page_rows[req] : a.emb_rows[req];
    const UnitT* src = static_cast<const UnitT*>(which ? a.src[1] : a.src[0]);
    UnitT* pages = static_cast<UnitT*>(which ? a.pages[1] : a.pages[0]);
    pages[dst_row * a.row_units + u] = src[e];
}

// A prompt's rows between contiguous [kv][token][dim] (MSL scatter_kv_paged_f16/f32,
// metal_runtime.mm:468-512, and its inverse gather_kv_pages_f16/f32, :328-370) and its pages: token t
// sits at absolute slot start_slot + t of the page table.  Units are taken in page order (token, KV
// head, unit of the head's row), so one side is one contiguous stream and the other pieces of a head's
// row.  The page table travels inside the kernel arguments where it fits: a call of 1 500 tokens is
// then one launch of 3 us instead of a copy of 3 us and the launch behind it.
static constexpr size_t kKvCopyEmbPages = 960;
// (16 bytes as a vector of the compiler's own: an array of HIP's uint4 was given a home in LDS, at an address made from the
// dispatch packet, which lies in host memory.  Two scatters and two gathers of 8 heads of 128 halves, 4096 and 8192 tokens:
// 115 and 123 us -> 61 and 72, of which 48 are four calls' launch and wait.)
typedef uint32_t copy_u32x4 __attribute__((ext_vector_type(4)));
struct KvCopyArgs {
    const void* src;
    void* dst;
    const uint32_t* page_table;   // on the device, or null: emb_table
    uint32_t n_kv_heads, tokens, head_units, page_size, start_slot;
    uint32_t emb_table[kKvCopyEmbPages];
};

// UNITS per thread, all in flight together: 1 where the copy is too small to give every CU several
// workgroups otherwise, 4 above (16-byte units: 4 KiB per wave in flight).  Index: 32 bits wherever the
// unit count allows it (a 64-bit division is a hundred instructions).
template <typename UnitT, bool TO_PAGES, int UNITS, typename Index>
__global__ __launch_bounds__(256) void kv_copy_kernel(const KvCopyArgs a) {
    const Index row_units = (Index)a.n_kv_heads * a.head_units;
    const Index total = row_units * a.tokens;
    const UnitT* src = static_cast<const UnitT*>(a.src);
    UnitT* dst = static_cast<UnitT*>(a.dst);
    const Index first = (Index)blockIdx.x * (256 * UNITS) + threadIdx.x;
    UnitT v[UNITS];
    size_t to[UNITS];
#pragma unroll
    for (int i = 0; i < UNITS; ++i) {
        const Index unit = first + (Index)(i * 256) < total ? first + (Index)(i * 256) : total - 1;
        const uint32_t token = (uint32_t)(unit / row_units);
        const uint32_t in_row = (uint32_t)(unit - token * row_units);
        const uint32_t kv = in_row / a.head_units, u = in_row - kv * a.head_units;
        const uint32_t abs_slot = a.start_slot + token, page = abs_slot / a.page_size, slot = abs_slot - page * a.page_size;
        const uint32_t page_id = a.page_table ? a.page_table[page] : a.emb_table[page];
        const size_t paged = ((size_t)page_id * a.page_size + slot) * row_units + in_row;
        const size_t flat = ((size_t)kv * a.tokens + token) * a.head_units + u;
        v[i] = src[TO_PAGES ? flat : paged];
        to[i] = TO_PAGES ? paged : flat;
    }
#pragma unroll
    for (int i = 0; i < UNITS; ++i)
        if (first + (Index)(i * 256) < total) dst[to[i]] = v[i];
}

}  // namespace mlc_hip
