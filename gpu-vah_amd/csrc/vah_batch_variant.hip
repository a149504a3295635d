// vah_batch_variant.hip -- instantiates the persistent batch stage kernels for
// one tile shape.  Built twice per shape with
//   -DVAH_BV_TX=<tile x> -DVAH_BV_TY=<tile y> -DVAH_BV_NW=<waves per role>
//   -DVAH_BV_FN=<name of the launch function> -DVAH_BV_FN3=<its 3+1D part>
// and -DVAH_BV_PART=2 (the launch function and the 2+1D kernels) or
// -DVAH_BV_PART=3 (the 3+1D kernels), so that the two dimensionalities can be
// compiled with different scheduler settings (the variant table in
// vah_batch.hip lists the builds).
#include "vah_batch_kernels.h"

#if !defined(VAH_BV_TX) || !defined(VAH_BV_TY) || !defined(VAH_BV_NW) || !defined(VAH_BV_FN) || \
    !defined(VAH_BV_FN3) || !defined(VAH_BV_PART)
#error "vah_batch_variant.hip needs VAH_BV_TX, VAH_BV_TY, VAH_BV_NW, VAH_BV_FN, VAH_BV_FN3 and VAH_BV_PART"
#endif

namespace vah {

namespace {

template <bool D3, bool S2, typename R>
void launch_one(const BatchLaunch &L) {
    hipLaunchKernelGGL((batch_stage_kernel<D3, S2, R, VAH_BV_TX, VAH_BV_TY, VAH_BV_NW>), dim3(L.grid),
                       dim3(128 * VAH_BV_NW), 0, L.stream, L.rec, D3 ? L.tiles3 : L.tiles2, L.counts);
}

template <bool D3, typename R>
void launch_r(const BatchLaunch &L, bool stage2) {
    if (stage2)
        launch_one<D3, true, R>(L);
    else
        launch_one<D3, false, R>(L);
}

}  // namespace

#if VAH_BV_PART == 3
void VAH_BV_FN3(const BatchLaunch &L, bool stage2, bool fp32) {
    if (fp32)
        launch_r<true, float>(L, stage2);
    else
        launch_r<true, double>(L, stage2);
}
#else
void VAH_BV_FN3(const BatchLaunch &L, bool stage2, bool fp32);

void VAH_BV_FN(const BatchLaunch &L, bool d3, bool stage2, bool fp32) {
    if (d3)
        VAH_BV_FN3(L, stage2, fp32);
    else if (fp32)
        launch_r<false, float>(L, stage2);
    else
        launch_r<false, double>(L, stage2);
}
#endif

}  // namespace vah
