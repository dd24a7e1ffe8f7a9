// The decode GEMM's kernels with the q/k/v epilogue (RoPE, K/V store, query fold).
#include "ls_gemm_kernel.h"

namespace ls {

hipError_t launch_gemm_rope(const GemmParams& p, int spw, dim3 grid, hipStream_t stream) {
    return launch_epilogue<GEMM_ROPE>(p, spw, grid, stream);
}

}  // namespace ls
