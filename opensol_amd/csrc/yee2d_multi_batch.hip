// Several steps per launch for batched 2D instances (E_z and H_z mixed): the windows of yee2d_multi.hip over all members.
#include "yee2d_multi.h"

// Launch `launch` of a call: every member advances by `steps` steps from step *clock + offset, or by those that its
// step limit leaves. Window b belongs to the member whose range [prefix[k], prefix[k + 1]) holds it; a member's plan is
// laid out for at least `steps` steps. State n has to end in set n & 1, and each launch a member takes part in flips its
// set: a member that has reached its limit after a number of launches of the other parity than its steps (`previous`:
// the steps of the launch before) takes one more launch of no steps, which copies its state.
template <int VEC, int R, int TV, int TR, int NW>
__global__ void __launch_bounds__(64 * NW, 4)
    yee2d_multi_batch_kernel(const yee2d_desc* __restrict__ descs, const yee2d_multi_plan* __restrict__ plans,
                             const int32_t* __restrict__ prefix, int32_t n_inst, int32_t offset, int32_t launch,
                             int32_t steps, int32_t previous)
{
    const int block = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (block >= prefix[n_inst]) return;
    int lo = 0, hi = n_inst;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (prefix[mid] <= block) lo = mid; else hi = mid;
    }
    lo = __builtin_amdgcn_readfirstlane(lo);
    typedef const __attribute__((address_space(4))) yee2d_desc ConstDesc;
    typedef const __attribute__((address_space(4))) yee2d_multi_plan ConstPlan;
    const yee2d_desc& d = *(const yee2d_desc*)((ConstDesc*)descs + lo);
    const yee2d_multi_plan& plan = *(const yee2d_multi_plan*)((ConstPlan*)plans + lo);
    const int64_t v = *d.clock;
    const int64_t clock = (int64_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32 |
                          (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
    const int64_t left = d.step_limit - clock;   // steps from the start of the call
    int take = 0;
    if (left > offset) {
        take = (int)min((int64_t)steps, left - offset);
        if (take == 0) return;   // the last launch of a call, for members that have just reached their limit
    } else if (left <= offset - previous || ((left ^ launch) & 1) == 0) {
        return;
    }
    const int index = block - __builtin_amdgcn_readfirstlane(prefix[lo]);
    if (d.polarization == YEE_EZ)
        yee::multi_block<YEE_EZ, VEC, R, TV, TR, NW, false>(d, plan, index, clock, offset, launch, take);
    else
        yee::multi_block<YEE_HZ, VEC, R, TV, 0, NW, false>(d, plan, index, clock, offset, launch, take);
}

#define YEE_MULTI_BATCH_KERNEL(VEC, R, TV, TR, NW)                                                                    \
    template __global__ void yee2d_multi_batch_kernel<VEC, R, TV, TR, NW>(                                            \
        const yee2d_desc* __restrict__, const yee2d_multi_plan* __restrict__, const int32_t* __restrict__, int32_t,   \
        int32_t, int32_t, int32_t, int32_t);
YEE_MULTI_BATCH_KERNEL(1, 8, 2, 8, 8)
YEE_MULTI_BATCH_KERNEL(1, 4, 1, 0, 8)
