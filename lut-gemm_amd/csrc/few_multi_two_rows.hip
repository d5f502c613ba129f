// The kernel for 3 to 16 activation rows (few_body.h) over a work list: instances for two rows per wavefront.
#include "few_body.h"

namespace lutgemm_kernels {

hipError_t launch_few_multi_two_rows(int q, int has_offset, const MultiMatvecArgs &m, const FewGrid &g, int workgroups, int waves, hipStream_t s)
{
    return launch_few_list_input<FewInput::kTwoRows, false>(q, has_offset, m, g, workgroups, waves, s);
}

}  // namespace lutgemm_kernels
