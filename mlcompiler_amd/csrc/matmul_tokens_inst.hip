// The kernels of the matmuls over many tokens, in a translation unit of their own.
#include "matmul_tokens_kernels.h"

namespace mlc_hip {

void launch_tokens_split(const float* x, _Float16* frag, float* inv_scale, uint32_t tokens, uint32_t cols, unsigned grid, hipStream_t stream) {
    if (cols > 4096) hipLaunchKernelGGL(tokens_split_kernel<1024>, dim3(grid), dim3(1024), 0, stream, x, frag, inv_scale, tokens, cols);
    else hipLaunchKernelGGL(tokens_split_kernel<256>, dim3(grid), dim3(256), 0, stream, x, frag, inv_scale, tokens, cols);
}
void launch_matmul_tokens(bool q6, const TokensArgs& a, unsigned grid, hipStream_t stream) {
    if (q6) hipLaunchKernelGGL((matmul_tokens_kernel<TokensQ6>), dim3(grid), dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((matmul_tokens_kernel<TokensQ4>), dim3(grid), dim3(256), 0, stream, a);
}

}  // namespace mlc_hip
