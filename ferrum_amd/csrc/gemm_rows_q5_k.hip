// The few-rows projection's kernels (gemm_rows.hpp) for Q5_K weights.
#include "gemm_rows.hpp"

namespace fh {

void launch_rows_q5_k(hipStream_t s, uint32_t dtype, const RowsPlan& plan, const RowsParams& p) {
    launch_rows_of<kQ5K>(s, dtype, plan, p);
}

}  // namespace fh
