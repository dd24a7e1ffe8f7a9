// The decode GEMM's kernels with the plain epilogue (bias, one rounding), and split K.
#include "ls_gemm_kernel.h"

namespace ls {

hipError_t launch_gemm_plain(const GemmParams& p, int spw, dim3 grid, hipStream_t stream) {
    return launch_epilogue<GEMM_PLAIN>(p, spw, grid, stream);
}

}  // namespace ls
