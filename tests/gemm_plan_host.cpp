// Reads "dtype M N K scratch on_16" lines and prints the GEMM plan the library makes
// for each on a 256-CU part, one line of numbers per shape. Plans are host code:
// no GPU is needed. Linked to libmi355bench.so by tests/test_gemm_plans.py.
#include <cinttypes>
#include <cstdio>

#include "../teamredbench_amd/csrc/mb_common.hpp"

int main() {
    mb::DeviceProps props;
    props.cu_count = 256;
    props.is_gfx950 = true;
    int dtype, on_16;
    int64_t m, n, k;
    uint64_t scratch;
    while (std::scanf("%d %" SCNd64 " %" SCNd64 " %" SCNd64 " %" SCNu64 " %d", &dtype, &m, &n, &k, &scratch, &on_16) == 6) {
        mb::GemmPlan p;
        const int rc = mb::gemm_plan(dtype, m, n, k, props, mb::Scratch{(size_t)scratch, on_16 != 0}, &p);
        std::printf("%d %d %d %d %d %d %zu %s %s\n", rc, p.tile_m, p.tile_n, p.tile_k, p.k_stages, p.split_k, p.workspace,
                    p.implementation, p.family);
    }
    return 0;
}
