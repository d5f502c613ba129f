// The kernel for 3 to 16 activation rows (few_body.h): instances whose wavefronts stage two rows each (a translation unit of
// its own, so that the instances compile side by side).
#include "few_body.h"

namespace lutgemm_kernels {

hipError_t launch_few_two_rows(int q, int has_offset, const MatvecArgs &a, const FewGrid &g, int waves, hipStream_t s)
{
    return launch_few_input<FewInput::kTwoRows, false>(q, has_offset, a, g, waves, s);
}

}  // namespace lutgemm_kernels
