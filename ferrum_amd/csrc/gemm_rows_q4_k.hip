// The few-rows projection's kernels (gemm_rows.hpp) for Q4_K weights.
#include "gemm_rows.hpp"

namespace fh {

void launch_rows_q4_k(hipStream_t s, uint32_t dtype, const RowsPlan& plan, const RowsParams& p) {
    launch_rows_of<kQ4K>(s, dtype, plan, p);
}

}  // namespace fh
