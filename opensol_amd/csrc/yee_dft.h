// DFT regions of an instance: the sampled cells of a region and their accumulation (yee_dft.hip, yee3d_after.h).
#pragma once

#include "yee_device.h"

namespace yee {

// Accumulate one sampled cell `t` of region `r`. field: the new state set's component pointers; n_axis: grid extent
// per axis; axis_stride: element stride per axis.
__device__ __forceinline__ void dft_cell(const yee_dft_region& r, float* const* field, const int32_t* n_axis,
                                         const int64_t* axis_stride, int64_t sample, int64_t t)
{
    const int64_t cells = (int64_t)r.count[0] * r.count[1] * r.count[2];
    if (t >= cells) return;
    const int64_t t2 = t % r.count[2];
    const int64_t rest = t / r.count[2];
    const int64_t t1 = rest % r.count[1];
    const int64_t t0 = rest / r.count[1];
    const int64_t index[3] = {r.start[0] + t0 * r.stride[0], r.start[1] + t1 * r.stride[1],
                              r.start[2] + t2 * r.stride[2]};
    const int64_t cell = index[0] * axis_stride[0] + index[1] * axis_stride[1] + index[2] * axis_stride[2];
    for (int c = 0; c < r.n_comp; ++c) {
        const float* f = field[r.comp[c]];
        float v = f[cell];
        const int a = r.pair_axis[c];
        if (a >= 0) {
            const int64_t lower = index[a] > 0 ? cell - axis_stride[a]
                                               : (r.pair_wrap[c] ? cell + (int64_t)(n_axis[a] - 1) * axis_stride[a]
                                                                 : cell);
            v = 0.5f * (v + f[lower]);
        }
        dft_region_add(r, c, cells, t, sample, v);
    }
}

// Sample index of step n, or -1 when step n takes no DFT sample.
__device__ __forceinline__ int64_t sample_of(int64_t n, int32_t m)
{
    return ((n + 1) % m) == 0 ? (n + 1) / m - 1 : -1;
}

// Region `region` of a 2D instance after step n (cell index i * pitch + j); the region's blocks stride over its cells.
__device__ __forceinline__ void dft_region_2d(const yee2d_desc& d, int64_t n, int region, int block, int blocks)
{
    if (n >= d.step_limit) return;
    const yee_dft_region& r = d.dft[region];
    const int64_t s = sample_of(n, d.sample_interval);
    if (s < 0 || s >= r.n_samples) return;
    const int set = (int)((n & 1) ^ 1);
    const int32_t n_axis[3] = {d.nx, d.ny, 1};
    const int64_t axis_stride[3] = {d.pitch, 1, 0};
    const int64_t cells = (int64_t)r.count[0] * r.count[1] * r.count[2];
    for (int64_t t = (int64_t)block * blockDim.x + threadIdx.x; t < cells; t += (int64_t)blocks * blockDim.x)
        dft_cell(r, d.field[set], n_axis, axis_stride, s, t);
}

// Region `region` of a 3D instance after step n (cell index (i * ny + j) * nz + k).
__device__ __forceinline__ void dft_region_3d(const yee3d_desc& d, int64_t n, int region, int block, int blocks)
{
    if (n >= d.step_limit) return;
    const yee_dft_region& r = d.dft[region];
    const int64_t s = sample_of(n, d.sample_interval);
    if (s < 0 || s >= r.n_samples) return;
    const int set = (int)((n & 1) ^ 1);
    const int32_t n_axis[3] = {d.nx, d.ny, d.nz};
    const int64_t axis_stride[3] = {(int64_t)d.ny * d.nz, d.nz, 1};
    const int64_t cells = (int64_t)r.count[0] * r.count[1] * r.count[2];
    for (int64_t t = (int64_t)block * blockDim.x + threadIdx.x; t < cells; t += (int64_t)blocks * blockDim.x)
        dft_cell(r, d.field[set], n_axis, axis_stride, s, t);
}

}  // namespace yee
