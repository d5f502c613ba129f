// The kernel for many activation rows (rows_body.h): instances whose wavefronts all share the k-blocks, and the dispatch.
#include "rows_body.h"

namespace lutgemm_kernels {

hipError_t launch_rows(int planes, int rt, int kw, const MatvecArgs &a, const RowsGrid &g, hipStream_t s)
{
    if (a.rows < 1 || g.row_chunks < 1 || a.rows > 16 * rt * g.row_chunks || (g.q != planes && g.q != planes - 1)) return hipErrorInvalidValue;
    return kw == 1 ? launch_rows_kw<1>(planes, rt, a, g, s) : kw == 2 ? launch_rows_two_groups(planes, rt, a, g, s) : hipErrorInvalidValue;
}

}  // namespace lutgemm_kernels
