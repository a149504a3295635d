// vah_stage3d.hip -- launches of the 3+1D single-lattice stage kernels, a translation
// unit of their own so that they compile beside the 2+1D ones.
#include <hip/hip_runtime.h>

#include "../../include/vah.h"
#include "vah_stage.h"

namespace vah {

namespace {

template <bool S2, typename R>
void launch3(const StageLaunch &L, const StageParams &P) {
    if (L.wide)
        hipLaunchKernelGGL((stage_kernel<true, S2, R, kWideTileX, kWideTileWaves>), dim3(L.grid),
                           dim3(128 * kWideTileWaves), 0, L.stream, P);
    else
        hipLaunchKernelGGL((stage_kernel<true, S2, R, kTileX, kTileWaves>), dim3(L.grid), dim3(128 * kTileWaves), 0,
                           L.stream, P);
}

template <bool S2>
void variant3(const StageLaunch &L, const StageParams &P) {
    if (L.precision == VAH_FP32_SPLIT)
        launch3<S2, float>(L, P);
    else if (L.flux_mode == VAH_FLUX_SHARED)
        launch3<S2, double>(L, P);
    else
        hipLaunchKernelGGL((stage_per_cell_kernel<true, S2>), dim3(L.grid), dim3(kCellThreads), 0, L.stream, P);
}

}  // namespace

void launch_stage_3d(const StageLaunch &L, int stage, const StageParams &P) {
    if (stage == 1)
        variant3<false>(L, P);
    else
        variant3<true>(L, P);
}

}  // namespace vah
