// The kernel for 3 to 16 activation rows (few_body.h): activations as rows, at most one per wavefront, and the dispatch.
#include "few_body.h"

namespace lutgemm_kernels {

hipError_t launch_few(int q, int has_offset, const MatvecArgs &a, const FewGrid &g, int waves, hipStream_t s)
{
    if (a.rows < 1 || a.rows > kBatchRows || waves < kFewWavesMin || g.gsub < 1 || g.gsub > 4 || g.gsub == 3 ||
        waves > few_waves_max(q + (has_offset ? 1 : 0), g.gsub))
        return hipErrorInvalidValue;
    if (g.gsub != 1) return launch_few_fine(q, has_offset, a, g, waves, s);
    if (g.columns) return waves == kFewWavesMin ? launch_few_columns(q, has_offset, a, g, s) : hipErrorInvalidValue;
    return a.rows <= waves ? launch_few_input<FewInput::kOneRow, false>(q, has_offset, a, g, waves, s) : launch_few_two_rows(q, has_offset, a, g, waves, s);
}

}  // namespace lutgemm_kernels
