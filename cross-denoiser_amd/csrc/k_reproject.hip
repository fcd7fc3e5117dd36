// Motion-vector reprojection on gfx950 as a launch of its own; the device code and what bounds it are in
// xdn_reproject.h.
#include "xdn_reproject.h"

namespace xdn {

template <int FNL, int FD, bool UNIT_OPAC>
__global__ __launch_bounds__(256) void reproject_kernel(RpBatch b)
{
    __shared__ RpShared<FNL, FD> sh;
    reproject_block<FNL, FD, UNIT_OPAC>(b, blockIdx.x, sh);
}

hipError_t launch_reproject(int n, const RpFrame *fr, int n_list, const int *dims, bool unit_opacity,
                            hipStream_t st)
{
    bool three3;
    const RpBatch b = rp_batch(n, fr, n_list, dims, three3);
    if (b.map.total == 0) return hipSuccess;
    if (three3 && unit_opacity)
        hipLaunchKernelGGL((reproject_kernel<3, 3, true>), dim3(b.map.total), dim3(256), 0, st, b);
    else if (three3)
        hipLaunchKernelGGL((reproject_kernel<3, 3, false>), dim3(b.map.total), dim3(256), 0, st, b);
    else
        hipLaunchKernelGGL((reproject_kernel<0, 0, false>), dim3(b.map.total), dim3(256), 0, st, b);
    return hipGetLastError();
}

}  // namespace xdn
