// One object per number of accumulator registers that a batch group needs: -DMLC_Q4_NI=1, 2 or 4.
#include "q4_matmul_mfma.h"

namespace mlc_hip {

#define MLC_CAT2(a, b) a##b
#define MLC_CAT(a, b) MLC_CAT2(a, b)

// false: there is no such variant
bool MLC_CAT(launch_q4_matmul_, MLC_Q4_NI)(int form, int rt, int waves, int zt, bool block_scales, dim3 grid, const Q4RopeArgs& a, hipStream_t stream) {
    const Q4Args& plain = a;
#define MLC_Q4Z(ZT, FORM, RT, WAVES, ARGS)                                                                                     \
    if (form == FORM && rt == RT && waves == WAVES && zt == ZT) {                                                              \
        const auto kernel = block_scales ? q4_matmul_kernel<MLC_Q4_NI, RT, WAVES, ZT < 4, FORM, ZT> : q4_matmul_kernel<MLC_Q4_NI, RT, WAVES, false, FORM, ZT>; \
        hipLaunchKernelGGL(kernel, grid, dim3(WAVES * 64), 0, stream, a.q, a.d, a.xfrag, a.blk_scale, a.ssq_in, a.nblocks, a.quads_per_slice, \
                           a.row_groups, a.batch | a.z_groups << 16, ARGS);                                                     \
        return true;                                                                                                           \
    }
#define MLC_Q4(...) MLC_Q4Z(1, __VA_ARGS__)
    MLC_Q4(kQ4Plain, 1, 16, plain) MLC_Q4(kQ4Plain, 2, 16, plain) MLC_Q4(kQ4Plain, 4, 16, plain) MLC_Q4(kQ4Plain, 4, 8, plain)
    MLC_Q4(kQ4Silu, 4, 16, plain) MLC_Q4(kQ4Silu, 4, 8, plain)
    MLC_Q4(kQ4Rope, 1, 16, a) MLC_Q4(kQ4Rope, 2, 16, a)
    MLC_Q4(kQ4Add, 2, 16, plain)
#if MLC_Q4_NI < 4
#define MLC_Q4R(RT, WAVES)                                                                                                     \
    if (form == kQ4Rows && rt == RT && waves == WAVES && zt == 1) {                                                            \
        hipLaunchKernelGGL((q4_matmul_kernel<MLC_Q4_NI, RT, WAVES, true, kQ4Rows>), grid, dim3(WAVES * 64), 0, stream, a.q, a.d, \
                           reinterpret_cast<const _Float16*>(a.xrows), nullptr, nullptr, a.nblocks, a.quads_per_slice, a.row_groups, \
                           a.batch | a.z_groups << 16, plain);                                                                 \
        return true;                                                                                                           \
    }
    MLC_Q4R(1, 16) MLC_Q4R(2, 16)
#if MLC_Q4_NI == 1
    MLC_Q4R(4, 16) MLC_Q4R(4, 8)
#endif
#undef MLC_Q4R
    MLC_Q4(kQ4Rope, 2, 8, a)
    MLC_Q4(kQ4Add, 2, 8, plain)
#else
    MLC_Q4(kQ4Rope, 4, 16, a) MLC_Q4(kQ4Rope, 4, 8, a)
    MLC_Q4(kQ4Add, 4, 16, plain) MLC_Q4(kQ4Add, 4, 8, plain)
    MLC_Q4Z(2, kQ4Plain, 4, 8, plain) MLC_Q4Z(2, kQ4Silu, 4, 8, plain)
    if (!block_scales) { MLC_Q4Z(4, kQ4Plain, 4, 8, plain) MLC_Q4Z(4, kQ4Silu, 4, 8, plain) }
#endif
#undef MLC_Q4
#undef MLC_Q4Z
    return false;
}

#if MLC_Q4_NI == 1
// Two matmuls in one launch, `blocks` workgroups of them the first one's; false: there is no such variant
bool launch_q4_chain(int form, int rt, uint32_t blocks, uint32_t grid, const Q4Args& a, const Q4RopeArgs& b, const Q4Link& link,
                     hipStream_t stream) {
    const auto launch = [&](auto kernel, const auto& args) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(1024), 0, stream, a.q, a.d, a.xfrag, a.blk_scale, a.ssq_in, a.nblocks, a.quads_per_slice,
                           a.row_groups, a.batch | blocks << 16, args);
        return true;
    };
    const uint32_t quads = (b.nquads + 15) / 16;   // per wave of the second matmul
    if (form == kQ4Silu && rt == 4 && quads == 1) return launch(q4_chain_kernel<4, 1, kQ4Silu>, Q4ChainArgs<kQ4Silu>{a, b, link});
    if (form == kQ4Rope && rt == 1 && quads <= 2) return launch(q4_chain_kernel<1, 2, kQ4Rope>, Q4ChainArgs<kQ4Rope>{a, b, link});
    if (form == kQ4Rope && rt == 2 && quads <= 2) return launch(q4_chain_kernel<2, 2, kQ4Rope>, Q4ChainArgs<kQ4Rope>{a, b, link});
    return false;
}
#endif

}  // namespace mlc_hip
