// The few-rows projection's kernels (gemm_rows.hpp) for Q6_K weights.
#include "gemm_rows.hpp"

namespace fh {

void launch_rows_q6_k(hipStream_t s, uint32_t dtype, const RowsPlan& plan, const RowsParams& p) {
    launch_rows_of<kQ6K>(s, dtype, plan, p);
}

}  // namespace fh
