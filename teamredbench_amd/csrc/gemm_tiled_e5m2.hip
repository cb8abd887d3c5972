// The tiled GEMM's kernels for one input type.
#include "gemm_tiled_kernels.hpp"

namespace mb {

int gemm_tiled_launch_e5m2(const GemmPlan& plan, const void* A, const void* B, void* C, int64_t M, int64_t N,
                           int64_t K, float alpha, void* workspace, hipStream_t stream) {
    return launch_dtype<MB_DT_FLOAT8_E5M2>(plan, A, B, C, M, N, K, alpha, workspace, stream);
}

}  // namespace mb
