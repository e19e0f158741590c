// Running-DFT box monitors for gfx950: one launch per step (skipped at once except on sample steps) accumulates the
// FP64 spectra of every DFT region of an instance, blockIdx.y per region and a grid-stride loop over its sampled
// cells. The grid is capped at one full occupancy of the device (2048 blocks of 256 lanes), so a step that takes no
// sample costs a few microseconds however large the box is.
//
// On sample step n ((n + 1) % m == 0, sample s = (n + 1) / m - 1) each lane reads its components from the new state
// set (one float each, or two for a face pair averaged to the cell centre) and adds v * phase[s][f] to its FP64 Kahan
// (sum, compensation) pairs of the real and imaginary parts at every frequency f. Accumulators are laid out
// [component][frequency][cell][4 (sum re, sum im, comp re, comp im)], so a wavefront reads and writes 64 consecutive
// 32-byte records: the kernel streams 64 B per cell, component and frequency plus the field reads, and is HBM bound
// on the sample steps.
//
// The descriptor is read in place at the kernel-argument pointer (constant address space): the field table is
// indexed by the runtime component, which would otherwise copy the whole descriptor to private memory.
//
// Reference semantics (file:line of the reference package open_sol/):
//   2D box monitor     physics/em/monitors.py:248-322 (DFTMonitor), :152-169 (dft_sample_slice, _centre_pairs)
//   3D plane monitor   physics/em3d/monitors3d.py:165-238 (DFTPlane3D)
//   phase              physics/em/monitors.py:22-34 (exp(-j omega t) m dt)
#include "yee_dft.h"

// DFT regions of a 2D instance after step n = *clock + offset, blockIdx.y per region.
__global__ void __launch_bounds__(256) yee2d_dft_kernel(yee2d_desc desc, int32_t offset)
{
    typedef const __attribute__((address_space(4))) yee2d_desc ConstDesc;
    const yee2d_desc& d = *(const yee2d_desc*)(ConstDesc*)__builtin_amdgcn_kernarg_segment_ptr();
    if (d.clock != desc.clock) return;
    yee::dft_region_2d(d, *d.clock + offset, blockIdx.y, blockIdx.x, gridDim.x);
}

// The DFT regions of a batch's members: blockIdx.z is the member, blockIdx.y its region (the grid spans the most
// regions and the largest region of any member; the rest return at once). Descriptors are read through the constant
// address space.
__global__ void __launch_bounds__(256) yee2d_batch_dft_kernel(const yee2d_desc* __restrict__ descs, int32_t offset)
{
    typedef const __attribute__((address_space(4))) yee2d_desc ConstDesc;
    const yee2d_desc& d = *(const yee2d_desc*)((ConstDesc*)descs + blockIdx.z);
    if ((int)blockIdx.y < d.n_dft) yee::dft_region_2d(d, *d.clock + offset, blockIdx.y, blockIdx.x, gridDim.x);
}

__global__ void __launch_bounds__(256) yee3d_batch_dft_kernel(const yee3d_desc* __restrict__ descs, int32_t offset)
{
    typedef const __attribute__((address_space(4))) yee3d_desc ConstDesc;
    const yee3d_desc& d = *(const yee3d_desc*)((ConstDesc*)descs + blockIdx.z);
    if ((int)blockIdx.y < d.n_dft) yee::dft_region_3d(d, *d.clock + offset, blockIdx.y, blockIdx.x, gridDim.x);
}
