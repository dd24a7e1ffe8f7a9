// The decode GEMM's kernels with the gate/up epilogue (SiLU and multiply).
#include "ls_gemm_kernel.h"

namespace ls {

hipError_t launch_gemm_glu(const GemmParams& p, int spw, dim3 grid, hipStream_t stream) {
    return launch_epilogue<GEMM_GLU>(p, spw, grid, stream);
}

}  // namespace ls
