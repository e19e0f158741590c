// Vector access and the single-cell updates shared by the 2D kernels (yee2d.hip one step per launch, yee2d_multi.h
// several). Every copy of a cell, in either file, goes through these helpers and the library is built with
// -ffp-contract=on, so a recomputed value equals its owner's bit for bit.
#pragma once

#include "yee_device.h"

namespace yee {

// ------------------------------------------------------------------------------------------------ vector access
template <int VEC>
__device__ __forceinline__ void ldv(const float* __restrict__ p, float out[VEC])
{
    if constexpr (VEC == 4) {
        const float4 v = *reinterpret_cast<const float4*>(p);
        out[0] = v.x; out[1] = v.y; out[2] = v.z; out[3] = v.w;
    } else {
        const float2 v = *reinterpret_cast<const float2*>(p);
        out[0] = v.x; out[1] = v.y;
    }
}

// Stores of the new state are non-temporal (the nt cache policy): nothing reads them again in this step, and the
// next step's reads come after the whole 8192^2 state has streamed past the caches. Streaming them keeps L2 for the
// halo rows and columns that neighbouring tiles re-read: 0.3451 against 0.3520 ms per 8192^2 E_z step.
template <int VEC>
__device__ __forceinline__ void stv(float* __restrict__ p, const float v[VEC])
{
    if constexpr (VEC == 4) {
        typedef float f4 __attribute__((ext_vector_type(4)));
        const f4 x = {v[0], v[1], v[2], v[3]};
        __builtin_nontemporal_store(x, reinterpret_cast<f4*>(p));
    } else {
        typedef float f2 __attribute__((ext_vector_type(2)));
        const f2 x = {v[0], v[1]};
        __builtin_nontemporal_store(x, reinterpret_cast<f2*>(p));
    }
}

// VEC uint16 ids kept packed (two per register) until use, so a prefetch is not waited on early
template <int VEC>
__device__ __forceinline__ void ldids(const uint16_t* __restrict__ p, uint32_t out[VEC / 2])
{
    if constexpr (VEC == 4) {
        const uint2 v = *reinterpret_cast<const uint2*>(p);
        out[0] = v.x; out[1] = v.y;
    } else {
        out[0] = *reinterpret_cast<const uint32_t*>(p);
    }
}

__device__ __forceinline__ int id_at(const uint32_t* packed, int k)
{
    return (packed[k >> 1] >> (16 * (k & 1))) & 0xffff;
}

// element k of a register array without dynamic indexing (which would move the array to scratch memory)
template <int VEC>
__device__ __forceinline__ float pickv(const float v[VEC], int k)
{
    float out = v[0];
#pragma unroll
    for (int q = 1; q < VEC; ++q) out = k == q ? v[q] : out;
    return out;
}

// ------------------------------------------------------------------------------------------ single-cell updates
// E_z polarisation, c = (ca, cb, da, db): H_y on a hi-x face = da H_y + db dE_z/dx (x CPML: psi = b psi + g dE,
// H_y += db psi); H_x on a hi-y face = da H_x - db dE_z/dy (y CPML: H_x -= db psi).
__device__ __forceinline__ float ez_hy(float4 c, float hy, float de, float idx, bool layer, float b, float g,
                                       float psi_old, float* psi_new)
{
    float v = c.z * hy + c.w * de * idx;
    if (layer) {
        const float psi = b * psi_old + g * de;
        *psi_new = psi;
        v += c.w * psi;
    }
    return v;
}

__device__ __forceinline__ float ez_hx(float4 c, float hx, float de, float idy, bool layer, float b, float g,
                                       float psi_old, float* psi_new)
{
    float v = c.z * hx - c.w * de * idy;
    if (layer) {
        const float psi = b * psi_old + g * de;
        *psi_new = psi;
        v -= c.w * psi;
    }
    return v;
}

// E_z at a centre = ca E_z + cb (dH_y/dx - dH_x/dy), before its CPML corrections.
__device__ __forceinline__ float ez_centre(float4 c, float e, float dhy, float dhx, float idx, float idy)
{
    return c.x * e + c.y * (dhy * idx - dhx * idy);
}

// H_z polarisation, c = (da, db, eps_xx, eps_yy): H_z at a centre = da H_z + db (dE_x/dy - dE_y/dx)
// (x CPML: H_z -= db psi_x, y CPML: H_z += db psi_y).
__device__ __forceinline__ float hz_centre(float4 c, float hz, float dex, float dey, float idy, float idx,
                                           bool layer_x, float bx, float gx, float psi_x_old, float* psi_x_new,
                                           bool layer_y, float by, float gy, float psi_y_old, float* psi_y_new)
{
    float v = c.x * hz + c.y * (dex * idy - dey * idx);
    if (layer_x) {
        const float psi = bx * psi_x_old + gx * dey;
        *psi_x_new = psi;
        v -= c.y * psi;
    }
    if (layer_y) {
        const float psi = by * psi_y_old + gy * dex;
        *psi_y_new = psi;
        v += c.y * psi;
    }
    return v;
}

// E_x on a hi-y face = ca E_x + cb dH_z/dy; E_y on a hi-x face = ca E_y - cb dH_z/dx (before CPML).
__device__ __forceinline__ float hz_ex(float ca, float cb, float ex, float dh, float idy) { return ca * ex + cb * dh * idy; }
__device__ __forceinline__ float hz_ey(float ca, float cb, float ey, float dh, float idx) { return ca * ey - cb * dh * idx; }

// (ca, cb) of an E face between cells of two ids: mean eps / sigma (shares 1/2, fdtd_hz_2d_kernels.py:190-278) formed
// in float32, or zero when either cell is PEC (eps = -1; every E face touching a PEC cell is pinned,
// physics/em/solvers/fdtd_hz_2d.py:475-495, yee_grid.py:145-150).
__device__ __forceinline__ void mixed_face(float ea, float eb, float siga, float sigb, float dt_over_eps0, float* ca,
                                           float* cb)
{
    if (ea < 0.f || eb < 0.f) {
        *ca = 0.f;
        *cb = 0.f;
        return;
    }
    const float eps_face = 0.5f * ea + 0.5f * eb;
    const float sig_face = 0.5f * siga + 0.5f * sigb;
    const float k = sig_face * (0.5f * dt_over_eps0) / eps_face;
    const float den = 1.0f + k;
    *ca = (1.0f - k) / den;
    *cb = (dt_over_eps0 / eps_face) / den;
}

__device__ __forceinline__ int wave_index()
{
    return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

}  // namespace yee
