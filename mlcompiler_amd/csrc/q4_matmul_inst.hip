// One object per number of accumulator registers that a batch group needs: -DMLC_Q4_NI=1, 2 or 4.
#include "q4_matmul_mfma.h"

namespace mlc_hip {

#define MLC_CAT2(a, b) a##b
#define MLC_CAT(a, b) MLC_CAT2(a, b)

// false: there is no such variant
bool MLC_CAT(launch_q4_matmul_, MLC_Q4_NI)(int form, int rt, int waves, bool block_scales, dim3 grid, const Q4RopeArgs& a, hipStream_t stream) {
    const Q4Args& plain = a;
#define MLC_Q4(FORM, RT, WAVES, ARGS)                                                                                          \
    if (form == FORM && rt == RT && waves == WAVES) {                                                                          \
        if (block_scales) hipLaunchKernelGGL((q4_matmul_kernel<MLC_Q4_NI, RT, WAVES, true, FORM>), grid, dim3(WAVES * 64), 0, stream, ARGS); \
        else hipLaunchKernelGGL((q4_matmul_kernel<MLC_Q4_NI, RT, WAVES, false, FORM>), grid, dim3(WAVES * 64), 0, stream, ARGS);             \
        return true;                                                                                                           \
    }
    MLC_Q4(kQ4Plain, 1, 16, plain) MLC_Q4(kQ4Plain, 2, 16, plain) MLC_Q4(kQ4Plain, 4, 16, plain) MLC_Q4(kQ4Plain, 4, 8, plain)
    MLC_Q4(kQ4Silu, 4, 16, plain) MLC_Q4(kQ4Silu, 4, 8, plain)
    MLC_Q4(kQ4Rope, 1, 16, a) MLC_Q4(kQ4Rope, 2, 16, a)
    MLC_Q4(kQ4Add, 2, 16, plain)
#if MLC_Q4_NI < 4
    MLC_Q4(kQ4Rope, 2, 8, a)
    MLC_Q4(kQ4Add, 2, 8, plain)
#else
    MLC_Q4(kQ4Rope, 4, 16, a) MLC_Q4(kQ4Rope, 4, 8, a)
    MLC_Q4(kQ4Add, 4, 16, plain) MLC_Q4(kQ4Add, 4, 8, plain)
#endif
#undef MLC_Q4
    return false;
}

}  // namespace mlc_hip
