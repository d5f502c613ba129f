// The kernel for 3 to 16 activation rows (few_body.h) over a work list: at most one row per wavefront, and the dispatch.
#include "few_body.h"

namespace lutgemm_kernels {

hipError_t launch_few_multi(int q, int has_offset, const MultiMatvecArgs &m, const FewGrid &g, int workgroups, int waves, hipStream_t s)
{
    if (m.count < 1 || m.count > kMaxFused || waves < kFewWavesMin || g.gsub < 1 || g.gsub > 4 || g.gsub == 3 || g.columns || g.partials || g.bias ||
        waves > few_waves_max(q + (has_offset ? 1 : 0), g.gsub))
        return hipErrorInvalidValue;
    bool two = false;   // some entry has more rows than the workgroups have wavefronts
    for (int i = 0; i < m.count; i++) {
        if (m.entry[i].rows < 1 || m.entry[i].rows > kBatchRows) return hipErrorInvalidValue;
        two = two || m.entry[i].rows > waves;
    }
    if (g.gsub != 1) return two ? launch_few_fine_multi_two_rows(q, has_offset, m, g, workgroups, waves, s) : launch_few_fine_multi(q, has_offset, m, g, workgroups, waves, s);
    return two ? launch_few_multi_two_rows(q, has_offset, m, g, workgroups, waves, s)
               : launch_few_list_input<FewInput::kOneRow, false>(q, has_offset, m, g, workgroups, waves, s);
}

}  // namespace lutgemm_kernels
