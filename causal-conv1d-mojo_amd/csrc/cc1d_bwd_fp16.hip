// cc1d_bwd_fp16.hip -- the backward kernels and launchers for fp16 storage, widths 2 to 5
// (one translation unit per dtype and half of the widths, so they compile in parallel).
#include "cc1d_bwd_kernels.hpp"

namespace cc1d {

CC1D_BWD_INSTANTIATE(f16, 2)
CC1D_BWD_INSTANTIATE(f16, 3)
CC1D_BWD_INSTANTIATE(f16, 4)
CC1D_BWD_INSTANTIATE(f16, 5)

}  // namespace cc1d
