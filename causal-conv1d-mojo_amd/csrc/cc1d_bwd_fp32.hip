// cc1d_bwd_fp32.hip -- the backward kernels and launchers for float storage
// (all widths: those above 5 have no row kernels).
#include "cc1d_bwd_kernels.hpp"

namespace cc1d {

CC1D_BWD_INSTANTIATE(float, 2)
CC1D_BWD_INSTANTIATE(float, 3)
CC1D_BWD_INSTANTIATE(float, 4)
CC1D_BWD_INSTANTIATE(float, 5)
CC1D_BWD_INSTANTIATE(float, 6)
CC1D_BWD_INSTANTIATE(float, 7)
CC1D_BWD_INSTANTIATE(float, 8)
CC1D_BWD_INSTANTIATE(float, 9)

}  // namespace cc1d
