// Several 2D steps per launch of one instance with DFT regions, field probes or a Drude pole (yee2d_multi.h).
#include "yee2d_multi_kernel.h"

YEE_MULTI_KERNELS(YEE_EZ, true)
YEE_MULTI_KERNELS(YEE_HZ, true)

// A Drude pole's current from state[1] to state[0], where it lies between calls, after an odd number of launches.
__global__ void __launch_bounds__(256) yee2d_pole_copy_kernel(const float* __restrict__ from, float* __restrict__ to,
                                                              int64_t count)
{
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < count; t += (int64_t)gridDim.x * 256) to[t] = from[t];
}
