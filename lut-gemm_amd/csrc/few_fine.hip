// The kernel for 3 to 16 activation rows (few_body.h): instances for scale groups of 32 and 64 k, at most one row per wavefront.
#include "few_body.h"

namespace lutgemm_kernels {

hipError_t launch_few_fine(int q, int has_offset, const MatvecArgs &a, const FewGrid &g, int waves, hipStream_t s)
{
    if (g.columns) return waves == kFewWavesMin ? launch_few_fine_columns(q, has_offset, a, g, s) : hipErrorInvalidValue;
    return a.rows <= waves ? launch_few_input<FewInput::kOneRow, true>(q, has_offset, a, g, waves, s) : launch_few_fine_two_rows(q, has_offset, a, g, waves, s);
}

}  // namespace lutgemm_kernels
