/*
 * Kernel instantiations: generalized Rodrigues, reference (FP64) form,
 * N = 2..6 levels, by assembled A2 (algo_rodr, any blob) and by rotation
 * planes (algo_rodrp, N = 3..6; team_kernel).
 */
#include "mbh_team.hpp"

namespace mbh {

#define MBH_ENTRY(LEV, C)                                                     \
    kernel_entry { MBH_ALGO_CVR_RODR, LEV, MBH_FORM_FP64, C,                  \
                   &launch_tile<algo_rodr<LEV>, C, double> }

#define MBH_PLANES(LEV, C)                                                    \
    kernel_entry { MBH_ALGO_CVR_RODR, LEV, KFORM_RODR_PLANES, C,              \
                   &launch_tile<algo_rodrp<LEV>, C, double> }

#define MBH_TEAM(LEV, FORM)                                                   \
    kernel_entry { MBH_ALGO_CVR_RODR, LEV, FORM, 1, &launch_team<LEV>,        \
                   MBH_ORDER_PLAIN }

template __global__ void team_kernel<3>(KArgs);
template __global__ void team_kernel<4>(KArgs);
template __global__ void team_kernel<5>(KArgs);
template __global__ void team_kernel<6>(KArgs);
template __global__ void tile_kernel<algo_rodr<2>, 1, double>(KArgs);
template __global__ void tile_kernel<algo_rodr<2>, 2, double>(KArgs);
template __global__ void tile_kernel<algo_rodr<3>, 1, double>(KArgs);
template __global__ void tile_kernel<algo_rodr<3>, 2, double>(KArgs);
template __global__ void tile_kernel<algo_rodr<4>, 1, double>(KArgs);
template __global__ void tile_kernel<algo_rodr<5>, 1, double>(KArgs);
template __global__ void tile_kernel<algo_rodr<6>, 1, double>(KArgs);
template __global__ void tile_kernel<algo_rodrp<3>, 1, double>(KArgs);
template __global__ void tile_kernel<algo_rodrp<3>, 2, double>(KArgs);
template __global__ void tile_kernel<algo_rodrp<4>, 1, double>(KArgs);
template __global__ void tile_kernel<algo_rodrp<5>, 1, double>(KArgs);

#if !defined(__HIP_DEVICE_COMPILE__)
const kernel_entry k_table_rodr[] = {
    MBH_ENTRY(2, 1), MBH_ENTRY(2, 2), MBH_ENTRY(3, 1), MBH_ENTRY(3, 2),
    MBH_ENTRY(4, 1), MBH_ENTRY(5, 1), MBH_ENTRY(6, 1),
    MBH_PLANES(3, 1), MBH_PLANES(3, 2), MBH_PLANES(4, 1), MBH_PLANES(5, 1),
    MBH_TEAM(3, KFORM_RODR_TEAM), MBH_TEAM(4, KFORM_RODR_TEAM),
    MBH_TEAM(5, KFORM_RODR_TEAM),
    /* (six levels: faster for every grid, see team_tiles) */
    MBH_TEAM(6, KFORM_RODR_PLANES),
};
const uint32_t k_table_rodr_n = sizeof(k_table_rodr) / sizeof(k_table_rodr[0]);
#endif

} /* namespace mbh */
