// cc1d_bwd_bf16.hip -- the backward kernels and launchers for bf16 storage, widths 2 to 5
// (one translation unit per dtype and half of the widths, so they compile in parallel).
#include "cc1d_bwd_kernels.hpp"

namespace cc1d {

CC1D_BWD_INSTANTIATE(bf16, 2)
CC1D_BWD_INSTANTIATE(bf16, 3)
CC1D_BWD_INSTANTIATE(bf16, 4)
CC1D_BWD_INSTANTIATE(bf16, 5)

}  // namespace cc1d
