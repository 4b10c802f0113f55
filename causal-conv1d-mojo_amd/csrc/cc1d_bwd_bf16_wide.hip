// cc1d_bwd_bf16_wide.hip -- the backward kernels and launchers for bf16 storage, widths 6 to 9
// (one translation unit per dtype and half of the widths, so they compile in parallel).
#include "cc1d_bwd_kernels.hpp"

namespace cc1d {

CC1D_BWD_INSTANTIATE(bf16, 6)
CC1D_BWD_INSTANTIATE(bf16, 7)
CC1D_BWD_INSTANTIATE(bf16, 8)
CC1D_BWD_INSTANTIATE(bf16, 9)

}  // namespace cc1d
