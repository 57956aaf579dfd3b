// The kernels of the chunked prefill attention, one object per head_dim: -DMLC_D=64 or 128.
#include "paged_prefill_kernels.h"

namespace mlc_hip {

#define MLC_CAT2(a, b) a##b
#define MLC_CAT(a, b) MLC_CAT2(a, b)

void MLC_CAT(launch_prefill_, MLC_D)(const PrefillArgs& a, int stages, bool rows64, uint32_t splits, hipStream_t stream) {
    launch_prefill_d<MLC_D>(a, stages, rows64, splits, stream);
}

}  // namespace mlc_hip
