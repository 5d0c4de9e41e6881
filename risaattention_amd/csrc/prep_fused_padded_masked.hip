// Fused preparation of rows of fewer channels with the derived forms of a mask in its first launch (a
// translation unit of its own, compiled beside prep_fused_padded.hip).
#include "prep_fused_kernels.hpp"

namespace risa {

void launch_prepare_padded_masked(const FusedRiders& a, hipStream_t stream) { launch_by_type<true, true>(a, stream); }

}  // namespace risa
