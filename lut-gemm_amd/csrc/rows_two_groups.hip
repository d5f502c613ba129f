// The kernel for many activation rows (rows_body.h): instances with two groups of wavefronts that share out the k-blocks
// (a translation unit of its own, so that the instances compile side by side).
#include "rows_body.h"

namespace lutgemm_kernels {

hipError_t launch_rows_two_groups(int planes, int rt, const MatvecArgs &a, const RowsGrid &g, hipStream_t s)
{
    return launch_rows_kw<2>(planes, rt, a, g, s);
}

}  // namespace lutgemm_kernels
