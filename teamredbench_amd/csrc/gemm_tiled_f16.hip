// The tiled GEMM's kernels for one input type.
#include "gemm_tiled_kernels.hpp"

namespace mb {

int gemm_tiled_launch_f16(const GemmPlan& plan, const void* A, const void* B, void* C, int64_t M, int64_t N,
                           int64_t K, float alpha, void* workspace, hipStream_t stream) {
    return launch_dtype<MB_DT_FLOAT16>(plan, A, B, C, M, N, K, alpha, workspace, stream);
}

}  // namespace mb
