// The multi-step kernel of one instance (yee2d_multi.h): a template, instantiated by yee2d_multi.hip (fields, sources and
// flux lines) and yee2d_multi_extra.hip (DFT regions, probes and a Drude pole too).
#pragma once

#include "yee2d_multi.h"

// `plan.take` steps of one instance from n = *clock + offset, reading state set (*clock + launch) & 1. General windows
// hold VEC columns by R rows per lane; TR > 0: the windows of region 0 of a plan with an interior, all of them lean,
// hold TV by TR. Blocks are dealt to the 8 XCDs in contiguous runs of windows, so the halo that neighbouring windows
// share meets in one L2.
template <int POL, int VEC, int R, int TV, int TR, int NW, bool EXTRA>
__global__ void __launch_bounds__(64 * NW, 4) yee2d_multi_kernel(yee2d_desc desc, yee2d_multi_plan plan,
                                                                 int32_t offset, int32_t launch)
{
    typedef const __attribute__((address_space(4))) yee2d_desc ConstDesc;
    const yee2d_desc& d = *(const yee2d_desc*)(ConstDesc*)__builtin_amdgcn_kernarg_segment_ptr();
    if (d.clock != desc.clock) return;   // the argument layout is not the one assumed: do nothing
    const int block = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (block >= plan.blocks) return;
    const int64_t clock = *d.clock;
    yee::multi_block<POL, VEC, R, TV, TR, NW, EXTRA>(d, plan, block, clock, offset, launch,
                                                       EXTRA ? plan.take : plan.steps);   // equal without EXTRA
}

#define YEE_MULTI_KERNEL(POL, VEC, R, TV, TR, NW, EXTRA)                                                                 \
    template __global__ void yee2d_multi_kernel<POL, VEC, R, TV, TR, NW, EXTRA>(yee2d_desc, yee2d_multi_plan, int32_t, \
                                                                               int32_t);
#define YEE_MULTI_KERNELS(POL, EXTRA)         \
    YEE_MULTI_KERNEL(POL, 1, 8, 2, 8, 8, EXTRA) \
    YEE_MULTI_KERNEL(POL, 1, 4, 1, 0, 8, EXTRA) \
    YEE_MULTI_KERNEL(POL, 1, 2, 1, 0, 8, EXTRA)
