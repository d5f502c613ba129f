// The kernel for 3 to 16 activation rows (few_body.h): instances for scale groups of 32 and 64 k that read activations stored as
// columns.
#include "few_body.h"

namespace lutgemm_kernels {

hipError_t launch_few_fine_columns(int q, int has_offset, const MatvecArgs &a, const FewGrid &g, hipStream_t s)
{
    return launch_few_input<FewInput::kColumns, true>(q, has_offset, a, g, kFewWavesMin, s);
}

}  // namespace lutgemm_kernels
