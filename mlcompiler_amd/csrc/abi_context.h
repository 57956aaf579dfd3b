// Library state and the helpers every entry point shares: error reporting, the context (Ctx) with its
// options, set-up, pinned metadata slots, device-resident copies of small host arrays, the operators that are
// held back to be fused with their neighbours (row chains, the KV write, the matmul with an epilogue) and the
// calls that launch them, the end of a call (finish).
//
// A section of the one translation unit mlc_hip.hip, which includes it once, in order, after the
// sections before it; not a header for anybody else.

namespace {

using namespace mlc_hip;

thread_local std::string g_err;
bool g_capture_failed = false;   // a call failed while a pass was being captured
bool g_capturing = false;        // between mlc_hip_capture_begin and mlc_hip_capture_end

int fail(const std::string& msg) {
    g_err = msg;
    if (g_capturing) g_capture_failed = true;
    return 0;
}

// For calls that allocate, copy or wait: none of that can be part of a captured pass.
#define NOT_WHILE_CAPTURING(what)                                                                   \
    do {                                                                                            \
        if (g_capturing) return fail(what ": not possible while a pass is being captured");         \
    } while (0)

#define HIP_OK(expr)                                                                  \
    do {                                                                              \
        hipError_t e_ = (expr);                                                       \
        if (e_ != hipSuccess)                                                         \
            return fail(std::string(#expr) + ": " + hipGetErrorString(e_));           \
    } while (0)

// A host-pinned + device pair used to hand small metadata to kernels.  `use` is the number of the slot's
// last use (Ctx::slot_uses, counted over all slots); it is written again once that use has run, which the
// host knows from a wait for the whole stream or for a marker (slot_reserve).
struct MetaSlot {
    void* host = nullptr;
    void* dev = nullptr;
    size_t cap = 0;
    uint64_t use = 0;
};

// Scratch memory of the tile-balanced decode kernel: the split-K partials (one slot per
// workgroup, tagged words that say by themselves whether they were written in the current
// launch, so nothing has to be cleared between launches), the replay word of captured passes,
// and, in probe builds, the time stamps.  A file-scope device array, so that no entry point
// that uses it has to allocate; every GPU the library runs on holds its own copy at its own
// address, which host code learns from hipGetSymbolAddress (the array's name is not a device
// address in host code).  Launches on one GPU share the array: they must not overlap.
constexpr size_t kScratchProbeBytes = (size_t)kStreamMaxWgs * 256;
constexpr size_t kScratchReplayWordOffset = kStreamPartBytes + kScratchProbeBytes;
constexpr size_t kScratchBytes = kScratchReplayWordOffset + 256;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// The buffers in which the K slices of matmuls meet (meeting_words) hold tagged words as well.
constexpr const char* kMeetingWords[] = {"q4_k_meet", "tokens_k_meet", "q4_link_words"};

// First launch of every captured pass: moves the replay word on, so that the launches of
// this replay (whose arguments, tag included, are the same at every replay) use tags that the
// replay before did not.
__global__ void replay_word_kernel(uint32_t* word, uint32_t step) { *word += step; }
constexpr uint32_t kReplayTagStep = 4096;   // decode launches of one captured pass, at most, and sliced matmuls with a tag

// Room for the words between two matmuls of a launch (q4_link_words): four requests of 4096 columns, eight copies, take 2.2 MB.
constexpr size_t kLinkBytes = 4u << 20;
constexpr size_t kChainBatch = 4;   // requests, at most (q4_chain_kernel: what more cost)

// Rounds that a wait for tagged words polls before it is given up (about 0.1 s).
constexpr long kSpinLimit = 200000;

// Tags: those of launches are their numbers, up to the first of these; those of launches that a caller records into a graph of
// its own lie behind, and behind them those of captured passes, at replay words up to the last.
constexpr uint32_t kLastLaunchTag = 0x3FFFFFFFu, kRecordedTag = 0x40000000u, kLastRecordedWord = 0x3FFFFFFFu,
                   kLastReplayWord = 0x80000000u - kReplayTagStep;

// Words that have been written once stay in memory until the same place is written again: before the tags start over, every
// buffer of such words is cleared (renew_tags).
__global__ void clear_words_kernel(uint4* p, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = make_uint4(0u, 0u, 0u, 0u);
}

// In front of every decode launch that a caller records into a graph of its own: numbers this replay's launch, whose arguments
// are the same at every replay.  When the numbers start over, which the host does not learn, the partials are cleared here
// (one workgroup, about a millisecond every 2^30 such launches).
__global__ __launch_bounds__(1024) void recorded_word_kernel(uint32_t* word, uint32_t step, uint4* part, uint32_t n) {
    const uint32_t last = *word;
    const bool over = last > kLastRecordedWord - step;
    if (over)
        for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) part[i] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    if (threadIdx.x == 0) *word = (over ? 0u : last) + step;
}
constexpr size_t kScratchRecordedWordOffset = kScratchReplayWordOffset + 128;

// Device copy of the flat page table (and, where the per-request arrays do not travel inside the
// kernel arguments, of those arrays) as the tile-balanced decode kernel reads it; uploaded only
// when the content changes.  One grow-only device buffer: its address stays the same from call to
// call (a captured pass keeps reading it), and a new content is copied over the old one in
// stream order, behind every launch that read the old one, from a slot of the pinned ring.
struct StreamTables {
    void* dev = nullptr;
    size_t cap = 0;
    bool filled = false;          // dev holds `flat` (version `uploaded`) and `meta`
    MetaSlot stage[4];            // pinned copies that a launch reads while it fills dev (tables_stage)
    int stage_next = 0;
    std::vector<uint32_t> flat;   // the caller's flat table as last seen
    uint64_t version = 0;         // counts the changes of `flat`
    uint64_t uploaded = ~0ull;    // version of `flat` that dev holds
    std::vector<uint32_t> meta;   // seq_lens | q_positions | offsets when they are uploaded too
    size_t meta_off = 0;          // byte offset of the arrays in dev
    uint32_t max_page = 0;        // largest page id in flat
    // does some page id occur in two requests' tables (then a row written for one request may be
    // read for another)?  -1: not computed for this content (tables_share_pages)
    int shared_pages = -1;
    std::vector<uint32_t> off;    // the caller's page_table_offsets as last seen
    std::vector<uint32_t> stamps; // by page id: the last question (stamp) in which the id was met
    uint32_t stamp = 0;
    std::vector<uint32_t> last_meta;  // seq_lens | q_positions | offsets of the last decode call (host copy)
};

// What the shape-agnostic decode kernel reads: the flat page table, the page-table offsets and the
// visible length of every request, in one device blob that is re-uploaded only when the tables
// change (the walker passes the same tables for every layer of a step).
struct DecodePlan {
    bool valid = false;
    // key
    std::vector<uint32_t> pt_flat, pt_off, seq_lens, q_pos;
    size_t B = 0;
    int causal = 0;
    // result
    size_t off_ptoff = 0, off_limits = 0;  // byte offsets in blob
    int slot = -1;
};

struct Ctx {
    bool inited = false;
    bool available = false;
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    bool pass_open = false;
    std::unordered_map<std::string, std::pair<void*, size_t>> cached;
    std::unordered_map<const void*, size_t> allocs;  // base pointer -> bytes (ours only)
    // Quantised weights, uploaded once per name (getOrCacheWeight, metal_runtime.mm:2434-2437):
    // the raw rows and, for shapes the MFMA path takes, the repacked nibbles and scales.
    struct Q4Weight {
        size_t bytes = 0, rows = 0, cols = 0, stride = 0;
        void* raw = nullptr;
        void* q = nullptr;
        void* d = nullptr;
        bool is(size_t b, size_t r, size_t c, size_t s) const { return raw && bytes == b && rows == r && cols == c && stride == s; }
    };
    std::unordered_map<std::string, Q4Weight> q4_weights;
    struct Q6KWeight {
        size_t bytes = 0, rows = 0, cols = 0, stride = 0;
        void* raw = nullptr;
        void* qa = nullptr;
        void* sc = nullptr;
        void* d = nullptr;
    };
    std::unordered_map<std::string, Q6KWeight> q6k_weights;
    long opt_q4_force_generic = 0;
    long opt_q4_int_operand = 1;  // Q4_0 matrix-core kernel: integer weights as operand, d applied per block
    long opt_q4_ksplit = 0;  // 0 = automatic
    MetaSlot ring[8];
    int ring_next = 0;
    uint64_t slot_uses = 0;    // uses of metadata slots so far
    uint64_t slots_done = 0;   // ... of which are known to have run
    // Markers: events on the library's stream, each behind the first `uses` uses.  One is recorded for every
    // second use that no wait has covered (the smallest rings have four slots), so that a caller that encodes
    // many calls without a wait waits for the oldest of them only, and one that waits now and then records none.
    struct SlotMarker {
        hipEvent_t ev = nullptr;
        uint64_t uses = 0;
    } markers[4];
    int marker_next = 0;
    uint64_t slots_marked = 0;   // uses that have a marker behind them, or have run
    // Small host arrays that callers pass again and again with the same content (norm weights,
    // the page ids of a decode step across its layers): kept on the device, uploaded only when
    // the content changes.
    struct Resident {
        std::vector<unsigned char> content;
        void* dev = nullptr;
        size_t cap = 0;
    };
    std::map<std::tuple<int, const void*, size_t>, Resident> resident;
    // Row-local operators of the open pass that have been encoded but not launched yet: a chain
    // that one row_program_kernel launch can run (walker_kernels.h).  Everything else that
    // touches the stream or device memory calls settle() first.
    struct RowPending {
        bool active = false;
        RowProgram p{};
        size_t batch = 0;            // 0 while only the flat element count is known (a lone add)
        size_t n_flat = 0;
        size_t len = 0;              // current row length
        const void* cur = nullptr;   // buffer that will hold the chain's current values
        size_t grid_rows = 0;        // rows launched
    } rows;
    // The KV write of a decode step that has been encoded but not launched: either the split +
    // RoPE + cast (whose fp16 K / V rows the batched scatters that follow it consume: they join
    // it, and the three become one launch), or a batched scatter waiting for its twin.
    struct KvPending {
        bool active = false;
        bool rope = false;
        bool from_gemm = false;             // rope form: runs as the epilogue of the pending matmul
        RopeArgs a{};                       // rope form
        const void* src[2] = {nullptr, nullptr};   // plain form: fp16 rows of the first / second scatter
        void* pages[2] = {nullptr, nullptr};
        int n = 0;
        bool wide = false;                  // plain form: 16-byte units
        std::vector<uint32_t> ids, slots;   // of the scatter(s) that joined so far
        size_t batch = 0, row_elems = 0, page_size = 0;
    } kv;
    // Who writes a Q4_0 matmul's activation fragments: the split kernel or a row chain, or the epilogue of the
    // launch in front (each with buffers of its own: the held-back matmul may still read another's).
    enum Q4Input { kXSplit, kXSilu, kXAttention, kXNorm };
    // A Q4_0 matmul of the open pass whose launch is held back for one call: when that call is
    // the split + RoPE + cast of the matmul's output (the qkv projection of a layer), the
    // matmul's epilogue does it and the two -- with the KV scatters that join -- are one launch.
    // When that call is the gate/up split + SiLU * up of the matmul's output (the gate/up
    // projection), the epilogue does that instead and the matmul is held back for one call more:
    // a Q4_0 matmul that reads the products (the down-projection) lets the epilogue also write
    // its activation fragments.  And while a residual add and an RMSNorm of the matmul's output
    // build their chain (RowPending) the matmul stays held back, too: a Q4_0 matmul that reads the
    // norm takes the chain's work over together with this one (mlc_hip_matmul_q4_0_batched).
    struct GemmPending {
        bool active = false;
        Q4Args a{};
        const void* out = nullptr;
        size_t batch = 0, rows = 0;
        bool block_scales = false;       // the activations carry one scale per (request, block)
        Q4Input x_from = kXSplit;        // who writes its activation fragments,
        int x_set = 0;                   // and in which of that producer's buffers they lie
        bool silu = false;               // the gate/up split + SiLU * up has joined
        const void* silu_out = nullptr;
        size_t ffn_inner = 0;
    } gemm;
    // The matmul in front of the held-back one, where its epilogue does the residual add and starts the norm that the
    // held-back one reads: both go out in one launch where they can (launch_chain), and this one alone before anything
    // that it reads is replaced.
    struct GemmFront {
        bool active = false;
        bool block_scales = false;
        Q4RopeArgs a{};
    } front;
    long opt_q4_chain = 1;           // 0 = always two launches
    // The tile-balanced decode attention launch of the open pass, held back for one call: when that
    // call is a Q4_0 matmul that reads the attention's output (the out-projection), the kernel
    // that writes a row of the output also writes it as that matmul's split-fp16 activations, one
    // scale exponent per (request, block of 32 columns), and the split kernel's launch goes away.
    // Everything about the call (tables, tags, the KV write it carries) was settled when it was
    // encoded; only the launch waits.
    struct DecodePending {
        bool active = false;
        StreamArgs a{};
        size_t head_dim = 0, dyn_lds = 0;
        int hpw = 0, nw = 0, nbuf = 0;
        unsigned n_wg = 0;
        const void* o = nullptr;
        size_t batch = 0, cols = 0;
    } dec;
    long decode_split_fused = 0;     // decode launches that also wrote the next matmul's activation fragments (for tests)
    long gemm_rope_fused = 0;        // matmuls launched with the RoPE epilogue (for tests)
    long gemm_silu_fused = 0;        // ... with the gate/up split + SiLU * up as epilogue
    long gemm_rms_fused = 0;         // ... with the residual add, the RMSNorm's sums and the next matmul's fragments as epilogue
    long gemm_silu_split_fused = 0;  // ... of which also wrote the next matmul's activation fragments
    std::vector<uint32_t> last_ids, last_slots;   // see place_page_rows
    size_t last_page_size = 0;
    size_t last_page_row = 0;        // the highest row of the last KV write
    long kv_fused = 0;               // KV writes that went out fused with a neighbour (for tests)
    long kv_in_decode = 0;           // ... of which inside the attention launch
    long opt_fuse_rows = 1;          // 0 = every operator is launched when it is encoded
    long row_launches = 0;           // row chains, and adds behind a held-back matmul, also in its epilogue (for tests)
    MetaSlot plan_slots[4];
    int plan_next = 0;
    DecodePlan plan;
    long opt_force_generic = 0;
    long opt_hpw_max = 0;                                      // query heads per wave, at most (0 = automatic)
    long opt_prefill_stages = 0;                               // LDS pipeline depth of the prefill kernel (0 = automatic)
    long opt_decode_mfma = 1;                                  // tile-balanced decode kernel: tile arithmetic on the matrix pipe
    long opt_prefill_rows64 = 1;                               // prefill: 64 chunk rows per wave where the GQA ratio allows it
    long opt_pv_fp16 = 0;                                      // 1 = softmax weights rounded to fp16 for P.V (default: fp32-grade)
    int last_launches = 0;
    int last_items = 0;
    char last_kernel[96] = "";   // kernel variant of the last decode launch (for benchmarks)
    int n_cu = 256;
    unsigned char* scratch_ptr = nullptr;   // device address of `scratch` on g.device
    uint32_t next_tag = 0;                  // tag of the last launch that needed one (never zero)
    uint32_t replay_word = 0;               // the replay word behind the last replay
    // Launches whose workgroups wait for each other (the decode attention, matmuls whose K slices meet inside the launch)
    // must follow each other also on different streams: decode launches share the one scratch array, and any two side
    // by side could each hold the CUs that workgroups need for which the other one's wait.  The stream of the last
    // such launch is remembered, and a launch on another stream first waits for that one (one event, created at
    // set-up; launches that stay on the library's stream cost nothing).
    hipStream_t scratch_stream = nullptr;
    bool scratch_in_use = false;
    hipEvent_t scratch_ev = nullptr;
    // One word of pinned host memory that a kernel sets (through its device address) when a
    // merge gives up waiting for another workgroup's partial; looked at wherever the host has
    // waited for the stream.
    volatile uint32_t* fault_host = nullptr;
    uint32_t* fault_dev = nullptr;
    long opt_spin_limit = kSpinLimit;       // rounds a merge of the decode attention polls before it gives up
    // Bit 0: workgroups do not publish their partials (tests of the give-up path); bit 1: a launch and a replay take more than
    // half of the tags there are (tests of what happens when they run out).
    long opt_test_flags = 0;
    StreamTables tables;
    long opt_wgs_per_cu = 0;        // tile-balanced kernel: workgroups per CU (0 = automatic)
    long opt_stream_stages = 0;     // tile-balanced kernel: LDS stages per workgroup (0 = automatic)
    long opt_grid_wgs = 0;          // tile-balanced kernel: exact grid size (0 = from workgroups per CU)
    // tile-balanced kernel: units the end of a (request, KV head) pair counts for when the ranges are
    // cut (a tile is one unit).  -1 = automatic: 2 for workgroups of four waves (swept 0..4 on
    // MI355X at the TinyLlama shape: batch 32 14.3 / 13.5 / 13.4 / 13.5 / 14.1 us, with the step's
    // KV write carried 15.5 / 14.8 / 13.9 / 14.1 / 14.6 us), 0 for the one- and two-wave workgroups
    // of GQA ratios 1 and 2, whose pair ends are cheap (there any cost was 1 to 5 % slower than 0).
    long opt_pair_cost = -1;
    long table_uploads = 0;         // page-table uploads of the tile-balanced path (for tests)
    // A captured pass: the kernel launches of the encode calls between mlc_hip_capture_begin and
    // mlc_hip_capture_end as an executable HIP graph, and what the launches read that changes from
    // decode step to decode step (device copies at fixed addresses, refreshed in place).
    struct Captured {
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;
        size_t n_nodes = 0;
        bool used_tables = false;            // a decode launch reads the device page table and arrays
        const void* tables_flat = nullptr;
        const void* tables_meta = nullptr;
        size_t B = 0, H = 0, Hkv = 0, D = 0, P = 0;
        int causal = 0;
        bool carried_kv = false;             // ... and does the step's KV write
        size_t n_decode = 0;                 // tile-balanced decode launches of the pass
        size_t n_sliced = 0;                 // matmuls of the pass whose K slices meet inside the launch
        uint32_t tag_step = 0;               // what a replay moves the replay word on by
        uint64_t buffer_generation = 0;      // Ctx::buffer_generation when the pass was captured
        const void* rows_dev = nullptr;      // device copy of the KV write's page rows
        size_t rows_batch = 0, rows_page_size = 0;
    };
    std::map<int, Captured> captures;
    // Counts the times a device buffer that the library owns (and a captured launch may have its
    // address baked in) was freed or moved: a capture taken at another count is stale.
    uint64_t buffer_generation = 0;
    int next_capture = 1;
    Captured cap;                            // the pass being captured
};

Ctx g;

bool init_once() {
    if (g.inited) return g.available;
    g.inited = true;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) {
        g_err = "no HIP device";
        return false;
    }
    if (hipGetDevice(&g.device) != hipSuccess) return false;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, g.device) != hipSuccess) return false;
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
        g_err = std::string("device is ") + prop.gcnArchName + ", library is built for gfx950";
        return false;
    }
    g.n_cu = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
    // the device address of the scratch array on this device (see its definition)
    void* sp = nullptr;
    if (hipGetSymbolAddress(&sp, HIP_SYMBOL(scratch)) != hipSuccess || !sp) {
        g_err = "hipGetSymbolAddress(scratch) failed";
        return false;
    }
    g.scratch_ptr = static_cast<unsigned char*>(sp);
    {
        void* fh = nullptr;
        void* fd = nullptr;
        if (hipHostMalloc(&fh, 64, hipHostMallocMapped) != hipSuccess || !fh ||
            hipHostGetDevicePointer(&fd, fh, 0) != hipSuccess || !fd) {
            g_err = "hipHostMalloc(fault word) failed";
            return false;
        }
        g.fault_host = static_cast<volatile uint32_t*>(fh);
        *g.fault_host = 0;
        g.fault_dev = static_cast<uint32_t*>(fd);
    }
    if (hipStreamCreateWithFlags(&g.stream, hipStreamNonBlocking) != hipSuccess) return false;
    if (hipEventCreate(&g.ev0) != hipSuccess || hipEventCreate(&g.ev1) != hipSuccess) return false;
    if (hipEventCreateWithFlags(&g.scratch_ev, hipEventDisableTiming) != hipSuccess) return false;
    for (Ctx::SlotMarker& m : g.markers)
        if (hipEventCreateWithFlags(&m.ev, hipEventDisableTiming) != hipSuccess) return false;
    g.available = true;
    return true;
}

// Waits for everything enqueued on the library's stream.
int wait_stream() {
    HIP_OK(hipStreamSynchronize(g.stream));
    // (a held-back attention launch, whose tables may lie in a slot, is not on the stream yet)
    if (!g.dec.active) g.slots_done = g.slots_marked = g.slot_uses;
    return 1;
}

int slot_reserve(MetaSlot& s, size_t bytes) {
    // (every copy of metadata to the device comes through here)
    NOT_WHILE_CAPTURING("copying metadata to the device (run the pass once uncaptured first; the planned and "
                        "generic decode kernels, one-request scatter / gather and prefill copy on every call)");
    // (everything that reads a slot is on the stream by now, unless an attention launch is held back)
    if (g.slot_uses - g.slots_marked >= 2 && !g.dec.active) {
        Ctx::SlotMarker& m = g.markers[g.marker_next];
        g.marker_next = (g.marker_next + 1) % 4;
        m.uses = 0;
        HIP_OK(hipEventRecord(m.ev, g.stream));
        m.uses = g.slots_marked = g.slot_uses;
    }
    if (s.use > g.slots_done) {
        Ctx::SlotMarker* oldest = nullptr;   // that lies behind this slot's use
        for (Ctx::SlotMarker& m : g.markers)
            if (m.uses >= s.use && (!oldest || m.uses < oldest->uses)) oldest = &m;
        if (oldest) {
            HIP_OK(hipEventSynchronize(oldest->ev));
            g.slots_done = oldest->uses;
        } else if (!wait_stream()) {
            return 0;
        }
    }
    if (bytes > s.cap) {
        size_t cap = std::max<size_t>(4096, bytes * 2);
        if (s.host) HIP_OK(hipHostFree(s.host));
        if (s.dev) HIP_OK(hipFree(s.dev));
        s.host = s.dev = nullptr;
        s.cap = 0;
        HIP_OK(hipHostMalloc(&s.host, cap, hipHostMallocDefault));
        HIP_OK(hipMalloc(&s.dev, cap));
        s.cap = cap;
    }
    return 1;
}

int slot_upload(MetaSlot& s, size_t bytes) {
    HIP_OK(hipMemcpyAsync(s.dev, s.host, bytes, hipMemcpyHostToDevice, g.stream));
    return 1;
}

// (called when what reads the slot has been enqueued, or is held back and will be before the slot's
// turn comes again)
void slot_mark(MetaSlot& s) { s.use = ++g.slot_uses; }

size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

int settle_gemm(const RopeArgs* rope);
int settle_front();
uint64_t* meeting_words(const char* name, size_t bytes);

int scratch_follow(hipStream_t stream);
int scratch_launched(hipStream_t stream);

// Tags that a launch or a replay takes, of a kind that goes up to `last`.
uint32_t tag_step(uint32_t step, uint32_t last) { return g.opt_test_flags & 2 ? last / 2 + 1 : step; }

// No tag is left that none of the words in memory can have: clears them, behind every launch that uses them, and starts over.
int renew_tags() {
    if (!scratch_follow(g.stream)) return 0;
    auto clear = [&](void* p, size_t bytes) {
        const unsigned grid = (unsigned)std::min<size_t>((bytes / 16 + 255) / 256, 1024);
        hipLaunchKernelGGL(clear_words_kernel, dim3(grid), dim3(256), 0, g.stream, static_cast<uint4*>(p), bytes / 16);
    };
    clear(g.scratch_ptr, kStreamPartBytes);
    clear(g.scratch_ptr + kScratchReplayWordOffset, 256);
    for (const char* name : kMeetingWords) {
        const auto it = g.cached.find(name);
        if (it != g.cached.end()) clear(it->second.first, it->second.second);
    }
    HIP_OK(hipGetLastError());
    g.next_tag = g.replay_word = 0;
    return scratch_launched(g.stream);
}

// Numbers a launch whose workgroups leave each other tagged words.  `in_pass` counts those of its kind in a captured pass:
// launches whose words lie in different buffers may have the same tag.
TagArgs next_tags(size_t& in_pass) {
    TagArgs t;
    t.fault = g.fault_dev;
    t.spin_limit = (uint32_t)g.opt_spin_limit;
    t.test_flags = (uint32_t)g.opt_test_flags & 1u;
    if (g_capturing) {
        // the arguments of a captured launch are the same at every replay: its tag is its number in
        // the pass plus the replay word, which the pass's first launch moves on by kReplayTagStep
        t.tag = 0x80000000u | (uint32_t)in_pass++;
        t.tag_dev = reinterpret_cast<const uint32_t*>(g.scratch_ptr + kScratchReplayWordOffset);
    } else {
        const uint32_t step = tag_step(1, kLastLaunchTag);
        if (g.next_tag > kLastLaunchTag - step) (void)renew_tags();   // (a failure shows at the launch behind it)
        g.next_tag += step;
        t.tag = g.next_tag;
        t.tag_dev = nullptr;
    }
    return t;
}
// The same for a matmul whose K slices meet.  The option cuts the wait of the decode attention, and this one only in tests of it.
TagArgs next_sliced_tags() {
    TagArgs t = next_tags(g.cap.n_sliced);
    if (!t.test_flags) t.spin_limit = (uint32_t)std::max(g.opt_spin_limit, kSpinLimit);
    return t;
}
bool sliced_tags_left() { return !g_capturing || g.cap.n_sliced < kReplayTagStep; }

// Device copy of a small host blob, uploaded only when (kind, key, bytes) has not been seen
// with this content.  The copy is ordered on the library stream, so kernels already enqueued
// that read the previous content are not disturbed.  nullptr on failure (error recorded).
const void* resident_blob(int kind, const void* key, const void* blob, size_t bytes) {
    // A caller that never repeats itself: start over -- but only while no held-back operator
    // refers to one of the copies (their launches come later).
    if (g.resident.size() > 1024 && !g.rows.active && !g.kv.active && !g.gemm.active && !g.front.active && !g.dec.active &&
        !g_capturing && g.captures.empty()) {   // (a captured pass keeps the addresses of the copies it read)
        if (!wait_stream()) return nullptr;
        for (auto& kv : g.resident)
            if (kv.second.dev) (void)hipFree(kv.second.dev);
        g.resident.clear();
    }
    Ctx::Resident& r = g.resident[std::make_tuple(kind, key, bytes)];
    if (r.dev && r.content.size() == bytes && std::memcmp(r.content.data(), blob, bytes) == 0) return r.dev;
    if (bytes > r.cap) {
        if (g_capturing) { fail("capture: a small host array is not on the device yet (run the pass once uncaptured first)"); return nullptr; }
        if (r.dev && hipFree(r.dev) != hipSuccess) { fail("resident: hipFree failed"); return nullptr; }
        if (r.dev) ++g.buffer_generation;
        r.dev = nullptr;
        r.cap = 0;
        const size_t cap = std::max<size_t>(256, align_up(bytes, 256));
        if (hipMalloc(&r.dev, cap) != hipSuccess) { r.dev = nullptr; fail("resident: hipMalloc failed"); return nullptr; }
        r.cap = cap;
    }
    // (a held-back matmul that finishes an RMSNorm reads the weights as they were: it goes out in front of the copy)
    if (r.dev && g.front.active && (g.front.a.rms_gamma == r.dev || g.front.a.add_gamma == r.dev) && !settle_front()) return nullptr;
    if (r.dev && g.gemm.active && g.gemm.a.rms_gamma == r.dev && !settle_gemm(nullptr)) return nullptr;
    r.content.clear();  // not valid until the copy has been enqueued
    MetaSlot& s = g.ring[g.ring_next];
    g.ring_next = (g.ring_next + 1) % 8;
    if (!slot_reserve(s, bytes)) return nullptr;
    std::memcpy(s.host, blob, bytes);
    if (hipMemcpyAsync(r.dev, s.host, bytes, hipMemcpyHostToDevice, g.stream) != hipSuccess) {
        fail("resident: upload failed");
        return nullptr;
    }
    slot_mark(s);
    r.content.assign(static_cast<const unsigned char*>(blob), static_cast<const unsigned char*>(blob) + bytes);
    return r.dev;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

size_t known_bytes(const void* p) {
    auto it = g.allocs.find(p);
    return it == g.allocs.end() ? 0 : it->second;
}

constexpr size_t kRowMaxLen = 16384;  // row_program_kernel: 8 groups of 8 elements per thread

bool row_len_ok(size_t len) { return len > 0 && len % 8 == 0 && len <= kRowMaxLen; }

// Rows of a Q4_0 matmul that is taken for a gate/up projection (kQ4Silu), and not for one that a residual add follows.
bool q4_wide(size_t rows) { return rows > 8192; }

// Tiles of 16 rows per workgroup of q4_matmul_kernel: as few as leave no more workgroups than CUs (one of 16 waves has
// a CU to itself), and 4 where there are more in any case: the activations that a CU fetches for a weight halve with
// every step.  (Whole calls, us, by rows > 8192 -> by this rule, and one workgroup of 32 x 32 products per 32 rows and 64
// requests: 6144 x 4096 at 17, 32, 33 and 64 requests 25.8, 27.0, 31.3, 34.2 -> 23.3, 23.6, 28.7, 29.9, 23.5, 24.5, 29.5,
// 31.4; 4096 x 4096 at 64 28.1 -> 24.8, 29.9; 4096 x 14336 at 64 70.4 -> 58.8, 62.5; 8192 x 4096 at 64 40.3 -> 32.8, 34.9.)
// The SiLU epilogue's workgroups have 4, the residual add's at least 2, and those of up to 8 requests with
// RoPE or the residual add at most 2 (the kernels of 4 do not fit the registers).
int q4_tiles(Q4Form form, size_t rows, size_t batch, size_t ksplit) {
    const size_t wgs = rows / 16 * ((batch + 15) / 16) * ksplit, n_cu = (size_t)g.n_cu;
    if (form == kQ4Silu) return 4;
    const int least = form == kQ4Add ? 2 : 1, most = form != kQ4Plain && form != kQ4Rows && batch <= 8 ? 2 : 4;
    return std::min(most, std::max(least, wgs > 2 * n_cu ? 4 : wgs > n_cu ? 2 : 1));
}

// Waves per workgroup, the same for every form of a call (they divide K).  16 fill a CU; where there are more
// workgroups than CUs, with 4 tiles each, they have 8, two workgroups to a CU, so that one's first loads overlap the
// other's products.
int q4_waves(const Q4Args& a) { return a.rows / 64 * ((a.batch + 15) / 16) * a.slices > (size_t)g.n_cu ? 8 : 16; }

int launch_chain(Q4Form form, bool block_scales, Q4RopeArgs& a);

// Launches q4_matmul_kernel in one of its forms.
int launch_q4(Q4Form form, bool block_scales, Q4RopeArgs& a) {
    if (g.front.active) {
        const int chained = launch_chain(form, block_scales, a);
        if (chained >= 0) return chained;
        if (!settle_front()) return 0;
    }
    const size_t tiles = a.rows / 16, z = (a.batch + 15) / 16, n_cu = (size_t)g.n_cu, ksplit = a.slices;
    const int rt = q4_tiles(form, a.rows, a.batch, ksplit);
    a.row_groups = (uint32_t)(tiles / rt);
    const int waves = q4_waves(a);
    // Such workgroups take four or two groups of 16 requests each, one workgroup to a CU, where those are one round of at
    // least five eighths of the CUs, or rounds of which the last is at least half full, with no group missing.  (Whole calls,
    // us, one group per workgroup -> now, and one workgroup of 32 x 32 products per 64 requests: 28672 x 4096 at 32, 49 and
    // 64 requests 46.5, 70, 74 -> 42.4, 58.4, 62, 44.4, 64.3, 66.5; 16384 x 4096 at 64 47.0 -> 38.9, 41.8; 11264 x 2048 at 32
    // 24.5 -> 23.3, 23.6.  Two groups elsewhere: 11264 x 2048 at 33, 352 workgroups, 26.3 -> 29.5; 8256 x 1024 at 32, 129
    // workgroups, 19.3 -> 19.8; 28672 x 4096 at 33, where half of 896 have one group only, 55.6 -> 63.6.)
    int zt = 1;
    for (const int n : {4, 2}) {
        const size_t wgs = tiles / 4 * ((z + n - 1) / n) * ksplit, last = wgs % n_cu;
        if (zt == 1 && waves == 8 && (form == kQ4Plain || form == kQ4Silu) && z > 1 && (n == 2 || (z == 4 && !block_scales)) &&
            (wgs <= n_cu ? wgs * 8 >= n_cu * 5 : z % n == 0 && (last == 0 || last * 2 >= n_cu)))
            zt = n;
    }
    a.z_groups = (uint32_t)((z + zt - 1) / zt);
    const dim3 grid((a.row_groups + 7) / 8 * 8 * a.z_groups, (unsigned)ksplit);
    if (ksplit > 1 && !scratch_follow(g.stream)) return 0;
    const auto launch = a.batch <= 4 ? launch_q4_matmul_1 : a.batch <= 8 ? launch_q4_matmul_2 : launch_q4_matmul_4;
    if (!launch(form, rt, waves, zt, block_scales, grid, a, g.stream)) return fail("q4 matmul: kernel variant not built");
    HIP_OK(hipGetLastError());
    return ksplit > 1 ? scratch_launched(g.stream) : 1;
}

// Launches the matmul in front of the held-back one by itself.
int settle_front() {
    if (!g.front.active) return 1;
    g.front.active = false;
    return launch_q4(kQ4Add, g.front.block_scales, g.front.a);
}

bool overlap(const void* a, size_t na, const void* b, size_t nb) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return x < y + nb && y < x + na;
}

// The matmul in front and the held-back one in one launch (q4_chain_kernel): 1, 0 on failure, -1 where they cannot be.  A wave
// of the second one holds its weights unpacked, 16 registers per row tile and quad of K, 64 of them at most: gate/up projections (four
// tiles) of up to 2048 columns, qkv projections (one or two) of up to 4096, which are as many as a norm in between has.
int launch_chain(Q4Form form, bool block_scales, Q4RopeArgs& b) {
    Q4RopeArgs& a = g.front.a;
    const size_t batch = b.batch;
    if (!g.opt_q4_chain || (form != kQ4Silu && form != kQ4Rope) || !block_scales || !g.front.block_scales || !b.ssq_in || b.ssq_in != a.ssq_out ||
        batch > kChainBatch || b.slices != 1 || q4_waves(a) != 16 || q4_waves(b) != 16 || q4_tiles(kQ4Add, a.rows, batch, a.slices) != 2)
        return -1;
    const int rt = q4_tiles(form, b.rows, batch, 1);
    if (rt * ((b.nquads + 15) / 16) > 4) return -1;
    a.row_groups = a.rows / 32;
    a.z_groups = b.z_groups = 1;
    b.row_groups = (uint32_t)(b.rows / 16 / rt);
    const uint32_t blocks = (a.row_groups + 7) / 8 * 8 * a.slices, grid = blocks + (b.row_groups + 7) / 8 * 8;
    if (blocks > 0xFFFFu || grid > 2 * (uint32_t)g.n_cu) return -1;
    // On every XCD a CU stays free of the second one's workgroups, which wait with a whole CU each (tagged_words.h: two
    // processes).  That costs nothing: where they take all CUs, the first one's hold up as many of them.  (8 layers of hidden 2048 and
    // FFN width 8192, 256 groups for gate/up, 1 to 4 requests, us, with gate/up in pairs -> by itself: 245, 253, 259, 268 -> 242, 246, 251, 256.)
    if ((b.row_groups + 7) / 8 >= (uint32_t)g.n_cu / 8) return -1;
    // The second matmul's workgroups run beside the first one's: what they write must be nothing that those read or write,
    // and what they read besides the words nothing that those write.
    const size_t row = batch * a.rows * 4;
    bool apart = true;
    const auto writes = [&](const void* p, size_t bytes) {
        if (!p) return;
        for (const void* q : {(const void*)a.out, (const void*)a.add_out, (const void*)a.add_resid}) apart = apart && !overlap(p, bytes, q, row);
        if (a.ssq_in)
            for (const void* q : {(const void*)a.rms_src, (const void*)a.rms_out}) apart = apart && !overlap(p, bytes, q, batch * a.rms_len * 4);
    };
    const auto reads = [&](const void* p, size_t bytes) {
        for (const void* q : {(const void*)a.out, (const void*)a.add_out}) apart = apart && !overlap(p, bytes, q, row);
        if (a.ssq_in) apart = apart && !overlap(p, bytes, a.rms_out, batch * a.rms_len * 4);
    };
    writes(b.out, batch * b.rows * 4);
    writes(b.rms_out, batch * b.rms_len * 4);
    if (form == kQ4Silu) {
        for (const void* p : {(const void*)b.gate, (const void*)b.up, (const void*)b.silu_out}) writes(p, batch * b.ffn_inner * 4);
    } else {
        const RopeArgs& r = b.rope;
        writes(r.q, batch * r.q_rows * 4);
        writes(r.k, batch * r.k_rows * 4);
        writes(r.v, batch * r.v_rows * 4);
        writes(r.k_f16, batch * r.k_rows * 2);
        writes(r.v_f16, batch * r.v_rows * 2);
        writes(r.k_pages, (g.last_page_row + 1) * r.k_rows * 2);
        writes(r.v_pages, (g.last_page_row + 1) * r.v_rows * 2);
        reads(r.cos_table, batch * (r.rotary_dim / 2) * 4);
        reads(r.sin_table, batch * (r.rotary_dim / 2) * 4);
    }
    const size_t bytes = q4_link_words(a.rows, b.batch) * 8 * kQ4LinkCopies;
    if (!apart || bytes > kLinkBytes || !sliced_tags_left()) return -1;
    Q4Link link;
    link.words = meeting_words("q4_link_words", kLinkBytes);   // (there since the first one was held back)
    if (!link.words) return -1;
    link.tags = next_sliced_tags();
    g.front.active = false;
    if (!scratch_follow(g.stream)) return 0;
    if (!launch_q4_chain(form, rt, blocks, grid, a, b, link, g.stream)) return fail("q4 matmul: kernel variant not built");
    HIP_OK(hipGetLastError());
    return scratch_launched(g.stream);
}

// Launches the held-back matmul, with the split + RoPE + cast of its output as epilogue when
// `rope` is given.
int settle_gemm(const RopeArgs* rope) {
    Ctx::GemmPending& m = g.gemm;
    if (!m.active) return settle_front();
    m.active = false;
    Q4RopeArgs a;
    static_cast<Q4Args&>(a) = m.a;
    Q4Form form = kQ4Plain;
    if (rope) {
        a.rope = *rope;
        form = kQ4Rope;
        ++g.gemm_rope_fused;
    } else if (m.silu) {
        m.silu = false;
        form = kQ4Silu;
        ++g.gemm_silu_fused;
        if (a.split_frag) ++g.gemm_silu_split_fused;
    } else if (a.add_resid) {
        form = kQ4Add;
    }
    return launch_q4(form, m.block_scales, a);
}

// Two buffers of one launch whose element i belongs to the same thread: do they meet at other elements than their own?
bool shifted(const void* a, const void* b, size_t bytes) { return a != b && overlap(a, bytes, b, bytes); }

// A matmul that finishes an RMSNorm reads the norm's input and writes its output in all its workgroups, in no order
// with what the others do: nothing else that the launch writes may lie there (and nothing that it reads in the output).
bool meets_norm(const Q4Args& a, const void* p, size_t bytes, bool written = true) {
    const size_t norm_bytes = (size_t)a.batch * a.rms_len * 4;
    return a.ssq_in && ((written && overlap(p, bytes, a.rms_src, norm_bytes)) || overlap(p, bytes, a.rms_out, norm_bytes));
}

// True when the held-back matmul's output is exactly the fused qkv rows a split + RoPE + cast
// call describes, so that the matmul's epilogue can do that call's work.
bool gemm_feeds_rope(const void* qkv, size_t batch, size_t qkv_rows, size_t q_rows, size_t k_rows, size_t v_rows) {
    const Ctx::GemmPending& m = g.gemm;
    return g.opt_fuse_rows && m.active && !m.silu && !g.kv.active && !g.rows.active && m.out == qkv && m.batch == batch &&
           m.rows == qkv_rows && q_rows + k_rows + v_rows == qkv_rows;
}

bool launch_stream_variant(size_t D, int hpw, int nw, int nbuf, const StreamArgs& a, unsigned n_wg, size_t dyn_lds,
                           hipStream_t stream);

// Launches the held-back decode attention.
int settle_decode() {
    Ctx::DecodePending& d = g.dec;
    if (!d.active) return 1;
    d.active = false;
    if (d.a.split_frag) ++g.decode_split_fused;
    if (!launch_stream_variant(d.head_dim, d.hpw, d.nw, d.nbuf, d.a, d.n_wg, d.dyn_lds, g.stream))
        return fail("decode: kernel variant not built");
    HIP_OK(hipGetLastError());
    return 1;
}

// The rows (page_id * page_size + slot) of one batched KV write on the device: what a captured pass and
// batches too large for the kernel arguments read (the layers of a decode step all write to the same
// rows, so only the first of them uploads).
const uint64_t* resident_page_rows(const uint32_t* page_ids, const uint32_t* slots, size_t batch, size_t page_size) {
    static thread_local std::vector<uint64_t> rows;
    rows.resize(batch);
    for (size_t r = 0; r < batch; ++r) rows[r] = (uint64_t)page_ids[r] * page_size + slots[r];
    const void* dev = resident_blob(1, nullptr, rows.data(), batch * 8);
    if (dev && g_capturing) {
        g.cap.rows_dev = dev;
        g.cap.rows_batch = batch;
        g.cap.rows_page_size = page_size;
    }
    return static_cast<const uint64_t*>(dev);
}

// Sets where a KV write's launch finds its page rows: in the kernel arguments (emb, room for `most`), or on
// the device.  They are remembered either way: mlc_hip_capture_begin brings the device copy to the rows of the
// last uncaptured KV write, so that a pass captured right after it finds them there.
bool place_page_rows(const uint32_t* page_ids, const uint32_t* slots, size_t batch, size_t page_size, uint64_t* emb, size_t most,
                     const uint64_t** dev) {
    *dev = nullptr;
    if (!g_capturing) {
        g.last_ids.assign(page_ids, page_ids + batch);
        g.last_slots.assign(slots, slots + batch);
        g.last_page_size = page_size;
    }
    g.last_page_row = 0;
    for (size_t r = 0; r < batch; ++r) g.last_page_row = std::max(g.last_page_row, (size_t)page_ids[r] * page_size + slots[r]);
    if (batch > most || g_capturing) return (*dev = resident_page_rows(page_ids, slots, batch, page_size)) != nullptr;
    for (size_t r = 0; r < batch; ++r) emb[r] = (uint64_t)page_ids[r] * page_size + slots[r];
    return true;
}

// Launches the pending KV write.
int settle_kv() {
    Ctx::KvPending& kv = g.kv;
    if (!kv.active) return 1;
    kv.active = false;
    if (kv.rope) {
        if (kv.a.k_pages || kv.a.v_pages) {
            ++g.kv_fused;
            if (!place_page_rows(kv.ids.data(), kv.slots.data(), kv.batch, kv.page_size, kv.a.emb_rows, kRopeEmbBatch, &kv.a.page_rows))
                return 0;
        }
        if (kv.from_gemm) return settle_gemm(&kv.a);
        launch_qkv_split_rope_cast(kv.a, g.stream);
        HIP_OK(hipGetLastError());
        return 1;
    }
    const unsigned block = 256;
    const uint32_t row_units = (uint32_t)(kv.row_elems * 2 / (kv.wide ? 16 : 2));
    const unsigned total = (unsigned)(kv.batch * row_units) * (unsigned)kv.n;
    const dim3 grid((total + block - 1) / block);
    if (kv.n == 2) ++g.kv_fused;
    ScatterPairArgs a{};
    a.src[0] = kv.src[0]; a.src[1] = kv.src[1];
    a.pages[0] = kv.pages[0]; a.pages[1] = kv.pages[1];
    a.batch = (uint32_t)kv.batch; a.row_units = row_units; a.n_tensors = (uint32_t)kv.n;
    if (!place_page_rows(kv.ids.data(), kv.slots.data(), kv.batch, kv.page_size, a.emb_rows, kScatterEmbBatch, &a.page_rows)) return 0;
    if (kv.wide) hipLaunchKernelGGL(scatter_kv_pair_kernel<uint4>, grid, dim3(block), 0, g.stream, a);
    else hipLaunchKernelGGL(scatter_kv_pair_kernel<uint16_t>, grid, dim3(block), 0, g.stream, a);
    HIP_OK(hipGetLastError());
    return 1;
}

// Launches what is pending, in the order it was encoded: a pending KV write is always older
// than a pending chain (whatever starts the KV write launches the chain first, and a scatter
// only joins while no chain is pending).  settle_before_rows() leaves the chain pending.
int settle_before_rows() {
    // a held-back attention launch is older than anything else: whatever was pending when it was
    // encoded has been launched, and nothing joins a chain behind it before it is launched
    if (!settle_decode()) return 0;
    // a held-back matmul is older than anything else pending, unless the pending KV write is
    // its own epilogue
    if ((g.gemm.active || g.front.active) && !(g.kv.active && g.kv.rope && g.kv.from_gemm) && !settle_gemm(nullptr)) return 0;
    return settle_kv();
}

// The held-back matmul's epilogue can do the pending chain's residual add of its output: the buffers lie apart, or exactly
// on each other where a thread has the same element of both (it reads the addend before it writes anything).
bool gemm_adds() {
    const Ctx::GemmPending& m = g.gemm;
    const RowProgram& p = g.rows.p;
    const size_t bytes = m.batch * m.rows * 4;
    return g.rows.active && m.active && !m.silu && !q4_wide(m.rows) && !g.kv.active && g.rows.batch == m.batch && g.rows.len == m.rows &&
           p.src == m.out && p.n_slices == 1 && !p.src_store && !p.silu && p.addend && !p.frag &&
           !overlap(p.addend, bytes, m.out, bytes) && !shifted(p.add_out, m.out, bytes) && !shifted(p.add_out, p.addend, bytes) &&
           !meets_norm(m.a, p.add_out, bytes) && !meets_norm(m.a, p.addend, bytes, false);
}

int settle() {
    Ctx::RowPending& r = g.rows;
    if (r.active && !r.p.rms && gemm_adds()) {
        // nothing but the add: 1.6 to 4 us for a launch of its own (counted like one)
        g.gemm.a.add_resid = r.p.addend;
        g.gemm.a.add_out = r.p.add_out;
        g.gemm.a.ssq_out = nullptr;
        g.gemm.a.split_frag = nullptr;
        r.active = false;
        ++g.row_launches;
    }
    if (!settle_before_rows()) return 0;
    if (!r.active) return 1;
    r.active = false;
    const RowProgram& p = r.p;
    // A lone add needs no rows: a flat kernel over all CUs (behind a matmul of 8192 rows: one request 1.6 us, 64
    // requests 2.6; as a row program, one workgroup per request, 2.3 and 3.6).
    if (r.batch == 0 || (p.addend && p.n_slices == 1 && !p.silu && !p.rms && !p.frag)) {
        hipLaunchKernelGGL(add_kernel, dim3((unsigned)((r.n_flat + 255) / 256)), dim3(256), 0, g.stream, p.src,
                           p.addend, p.add_out, (uint32_t)r.n_flat);
        if (r.batch) ++g.row_launches;
        HIP_OK(hipGetLastError());
        return 1;
    }
    if (r.len > kRowMaxLen) {  // only a sum over K slices can be this long (nothing joined it)
        const uint32_t n = (uint32_t)(r.batch * r.len);
        hipLaunchKernelGGL(q4_sum_slices_kernel, dim3((n + 255) / 256), dim3(256), 0, g.stream, p.src, p.src_store, n,
                           p.n_slices);
        HIP_OK(hipGetLastError());
        return 1;
    }
    const dim3 grid((unsigned)(p.frag ? r.grid_rows : r.batch));
    if (r.len <= 8 * (size_t)kRowThreads) hipLaunchKernelGGL((row_program_kernel<1>), grid, dim3(kRowThreads), 0, g.stream, p);
    else hipLaunchKernelGGL((row_program_kernel<2>), grid, dim3(kRowThreads), 0, g.stream, p);
    ++g.row_launches;
    HIP_OK(hipGetLastError());
    return 1;
}

// True when the pending chain's current values are those of `buf` as rows of `len` floats; fixes
// the row shape of a chain that so far only knew its element count.
bool rows_continue(const void* buf, size_t batch, size_t len) {
    Ctx::RowPending& r = g.rows;
    if (!g.opt_fuse_rows || !r.active || r.cur != buf || r.p.frag) return false;
    if (r.batch == 0) {
        if (r.n_flat != batch * len || !row_len_ok(len)) return false;
        r.batch = batch;
        r.len = len;
        r.p.len_src = (uint32_t)len;
        r.p.batch = (uint32_t)batch;
        return true;
    }
    return r.batch == batch && r.len == len;  // callers check that the length they go on with fits
}

// A chain's workgroups each do one row from the first operator to the last, in no order with the other rows: an operator
// may join only if its rows `p` of `len` floats meet what the chain reads and writes in the same row and column or
// not at all (written = false: what the chain writes).
bool rows_apart(const void* p, size_t len, bool written = true) {
    const Ctx::RowPending& r = g.rows;
    const RowProgram& c = r.p;
    const size_t half = c.silu ? c.len_src / 2 : c.len_src;
    auto apart = [&](const void* q, size_t q_len) {
        return !q || (p == q && len == q_len) || !overlap(p, r.batch * len * 4, q, r.batch * q_len * 4);
    };
    return apart(c.src_store, c.len_src) && (!c.silu || (apart(c.gate_out, half) && apart(c.up_out, half) && apart(c.silu_out, half))) &&
           apart(c.add_out, half) && (!written || (apart(c.n_slices == 1 ? c.src : nullptr, c.len_src) && apart(c.addend, half)));
}

// Starts a chain whose source is a plain buffer of rows.
void rows_begin(const void* src, size_t batch, size_t len) {
    Ctx::RowPending& r = g.rows;
    r = Ctx::RowPending{};
    r.active = true;
    r.p.src = static_cast<const float*>(src);
    r.p.n_slices = 1;
    r.p.len_src = (uint32_t)len;
    r.p.batch = (uint32_t)batch;
    r.batch = batch;
    r.len = len;
    r.n_flat = batch * len;
    r.cur = src;
}

// After a wait for the stream: did a launch give up on a partial?
int check_fault() {
    if (g.fault_host && *g.fault_host) {
        *g.fault_host = 0;
        return fail("a workgroup gave up waiting for another workgroup's partial result; the outputs of this "
                    "pass are not valid (launches that share the library's scratch memory must not overlap)");
    }
    return 1;
}

int finish(int sync) {
    HIP_OK(hipGetLastError());
    if (sync) {
        NOT_WHILE_CAPTURING("a call with sync = 1");
        if (!settle()) return 0;
        return wait_stream() && check_fault();
    }
    return 1;
}

}  // namespace
