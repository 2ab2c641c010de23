// The few-rows projection's kernels (gemm_rows.hpp) for Q8_0 weights.
#include "gemm_rows.hpp"

namespace fh {

void launch_rows_q8_0(hipStream_t s, uint32_t dtype, const RowsPlan& plan, const RowsParams& p) {
    launch_rows_of<kQ8_0>(s, dtype, plan, p);
}

}  // namespace fh
