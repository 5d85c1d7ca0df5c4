// mc_fixed_dt_wide.hip — the fixed-dt kernels whose clusters live wholly in LDS
// (mc_fixed_dt.h), the builds for clusters with large hole grids: a nearest-hole
// search whose 3x3x3 block is inconclusive takes wider blocks before every hole.
#include "mc_fixed_dt.h"

namespace mcl {

hipError_t prepare_fixed_dt_wide(int lds_bytes, int max_lds)
{
    return prepare_fixed_dt_t<false, true>(lds_bytes, max_lds);
}

hipError_t launch_fixed_dt_wide(const LaunchArgs& a, int grid, int lds_bytes, int waves,
                                hipStream_t stream)
{
    return launch_fixed_dt_t<false, true>(a, grid, (unsigned)(lds_bytes + fixed_dt_waves_lds(waves)),
                                          waves, stream);
}

hipError_t fixed_dt_wide_occupancy(int lds_bytes, int waves, int* blocks_per_cu)
{
    return fixed_dt_occupancy_t<false, true>((size_t)(lds_bytes + fixed_dt_waves_lds(waves)), waves,
                                             blocks_per_cu);
}

}  // namespace mcl
