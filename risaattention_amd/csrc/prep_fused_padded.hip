// Fused preparation of rows that hold fewer channels than the kernels' head dim (a translation unit
// of its own: as many kernels as for whole rows, compiled beside them).  Padding Q, K and V with
// zeros beforehand takes six launches and writes and reads all three once more: 45 of 148 us for
// 2 x 8 heads x 4096 tokens x 80 channels.
#include "prep_fused_kernels.hpp"

namespace risa {

void launch_prepare_padded(const FusedRiders& a, hipStream_t stream) { launch_by_type<true, false>(a, stream); }

}  // namespace risa
