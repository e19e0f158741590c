// What a 3D instance takes from the state after a step: flux-plane samples, DFT planes and field probes.
#pragma once

#include "yee_dft.h"

namespace yee3 {

// FP64 Kahan DFT sample of plane cell t (cells of plane 0 pair 0, then pair 1, then plane 1 ...) after step n, when (n + 1) % m
// == 0: E = mean of the layers edge - 1 and edge along the normal, H on layer edge - 1 (monitors3d.py:90-101).
__device__ __forceinline__ void sample_cell(const yee3d_desc& d, int64_t n, int64_t t)
{
    if (n >= d.step_limit || d.n_planes == 0) return;
    const int m = d.sample_interval > 0 ? d.sample_interval : 1;
    if ((n + 1) % m != 0) return;
    const int64_t sample = (n + 1) / m - 1;
    const int set = (int)((n & 1) ^ 1);
    for (int p = 0; p < d.n_planes; ++p) {
        const yee_flux_plane& pl = d.plane[p];
        for (int q = 0; q < 2; ++q) {
            const int na = pl.hi[q][0] - pl.lo[q][0], nb = pl.hi[q][1] - pl.lo[q][1];
            const int64_t count = (int64_t)na * nb;
            if (t >= count) {
                t -= count;
                continue;
            }
            if (sample >= pl.n_samples) return;
            const int a = pl.lo[q][0] + (int)(t / nb), b = pl.lo[q][1] + (int)(t % nb);
            const int ta = pl.normal == 0 ? 1 : 0, tb = pl.normal == 2 ? 1 : 2;   // tangential axes in grid order
            int idx[3];
            idx[ta] = a;
            idx[tb] = b;
            idx[pl.normal] = pl.edge - 1;
            const int64_t lower = ((int64_t)idx[0] * d.ny + idx[1]) * d.nz + idx[2];
            idx[pl.normal] = pl.edge;
            const int64_t upper = ((int64_t)idx[0] * d.ny + idx[1]) * d.nz + idx[2];
            const float* e = d.field[set][pl.e_comp[q]];
            const float* h = d.field[set][3 + pl.h_comp[q]];
            const double e_value = 0.5 * ((double)e[lower] + (double)e[upper]);
            const double h_value = (double)h[lower];
            const int nf = pl.n_freq;
            const double* ph = pl.phase + sample * (int64_t)nf * 2;
            for (int f = 0; f < nf; ++f) {
                const double pr = ph[2 * f], pi = ph[2 * f + 1];
                double* acc_e = pl.acc[q] + ((int64_t)(0 * nf + f) * 4) * count + t;
                double* acc_h = pl.acc[q] + ((int64_t)(1 * nf + f) * 4) * count + t;
                yee::kahan_add(acc_e, acc_e + 2 * count, pr * e_value);
                yee::kahan_add(acc_e + count, acc_e + 3 * count, pi * e_value);
                yee::kahan_add(acc_h, acc_h + 2 * count, pr * h_value);
                yee::kahan_add(acc_h + count, acc_h + 3 * count, pi * h_value);
            }
            return;
        }
    }
}

// Field probes of one instance after step n: samples[n * n_probes + k] = field[new set][component[k]][cell[k]]
// (core/monitors.py:42-130, physics/em3d/physics3d.py:425-433); the block's lanes stride over the probes.
__device__ __forceinline__ void probes_3d(const yee3d_desc& d, int64_t n)
{
    const yee_probes& p = d.probes;
    if (n >= d.step_limit || n >= p.capacity) return;
    const int set = (int)((n & 1) ^ 1);
    const int64_t cells = (int64_t)d.nx * d.ny * d.nz;
    for (int k = threadIdx.x; k < p.n_probes; k += blockDim.x) {
        const int32_t c = p.component[k];
        const int64_t cell = p.cell[k];
        // a record outside the grid or the components samples NaN rather than reading out of bounds
        p.samples[n * p.n_probes + k] = (c >= 0 && c < 6 && cell >= 0 && cell < cells)
                                            ? d.field[set][c][cell] : __builtin_nanf("");
    }
}

// Flux-plane samples of many instances after their step *clock + offset: thread t of the blocks belongs to the instance
// whose plane-cell range [prefix[k], prefix[k+1]) holds it.
__device__ __forceinline__ void sample_members(const yee3d_desc* __restrict__ descs, const int64_t* __restrict__ prefix,
                                               int32_t n_inst, int32_t offset, int block)
{
    const int64_t t = (int64_t)block * 256 + threadIdx.x;
    if (t >= prefix[n_inst]) return;
    int lo = 0, hi = n_inst;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (prefix[mid] <= t) lo = mid; else hi = mid;
    }
    typedef const __attribute__((address_space(4))) yee3d_desc ConstDesc;
    const yee3d_desc& d = *(const yee3d_desc*)((ConstDesc*)descs + lo);
    sample_cell(d, *d.clock + offset, t - prefix[lo]);
}

// Block `block` of those of `a`, after step n.
__device__ __forceinline__ void after_block(const yee3d_desc& d, const yee3d_after& a, int64_t n, int block)
{
    if (block < a.sample_blocks) {
        const int64_t t = (int64_t)block * 256 + threadIdx.x;
        if (t < a.sample_cells) sample_cell(d, n, t);
        return;
    }
    block -= a.sample_blocks;
    const int region = a.dft_blocks > 0 ? block / a.dft_blocks : d.n_dft;
    if (region < d.n_dft) yee::dft_region_3d(d, n, region, block - region * a.dft_blocks, a.dft_blocks);
    else if (d.probes.n_probes > 0) probes_3d(d, n);
}

}  // namespace yee3
