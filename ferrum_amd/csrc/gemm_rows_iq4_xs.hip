// The few-rows projection's kernels (gemm_rows.hpp) for IQ4_XS weights.
#include "gemm_rows.hpp"

namespace fh {

void launch_rows_iq4_xs(hipStream_t s, uint32_t dtype, const RowsPlan& plan, const RowsParams& p) {
    launch_rows_of<kIQ4XS>(s, dtype, plan, p);
}

}  // namespace fh
