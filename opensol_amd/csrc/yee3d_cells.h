// Cell updates of the 3D Yee step, shared by its kernels: every copy of a value rounds the same (the library is built with
// -ffp-contract=on: an FMA forms only within one expression), so a recomputed halo equals its owner's value bit for bit
// and the kernels agree with each other.
#pragma once

#include "yee_device.h"

namespace yee3 {

constexpr float EPS0F = 8.8541878128e-12f;

// (ca, cb) of an E face between cells of ids a and b: the id's own entry when they agree, else the coefficients of the
// float32 mean eps_r and sigma_e (shares 1/2; kernels3d.py:61-85). With k = sigma dt / (2 eps):
// ca = (1 - k) / (1 + k) = (eps - sigma dt/2) / (eps + sigma dt/2) and cb = (dt / eps) / (1 + k) = dt / (eps + sigma
// dt/2), formed with one reciprocal (within 2 ulp of the reference's float32 divisions).
// PEC ids carry eps_r = -1 and (ca, cb) = (0, 0): a face between two PEC cells is pinned by the id's own entry, and a
// face between a PEC cell and another cell takes the other cell's values (kernels3d.py:61-85), i.e. its own entry.
__device__ __forceinline__ float2 mixed_face(float dt, float2 ma, float2 mb)
{
    const float eps = (0.5f * ma.x + 0.5f * mb.x) * EPS0F;
    const float loss = (0.5f * ma.y + 0.5f * mb.y) * (0.5f * dt);
    const float inv = __builtin_amdgcn_rcpf(eps + loss);
    return make_float2((eps - loss) * inv, dt * inv);
}

// psi recursion of one layer cell: b psi + g dF.
__device__ __forceinline__ float psi_next(float b, float psi, float g, float difference) { return b * psi + g * difference; }

// ---- H components (shared by owners and halo copies) ----
// H_x: -db (dEz/dy - dEy/dz); CPML y first (-), z first (+).
__device__ __forceinline__ float hx_yee(float da, float db, float hx, float dez_y, float ihy, float dey_z, float ihz)
{
    return da * hx - db * (dez_y * ihy - dey_z * ihz);
}
// H_y: -db (dEx/dz - dEz/dx); CPML x first (+), z second (-).
__device__ __forceinline__ float hy_yee(float da, float db, float hy, float dex_z, float ihz, float dez_x, float ihx)
{
    return da * hy - db * (dex_z * ihz - dez_x * ihx);
}
// H_z: -db (dEy/dx - dEx/dy); CPML x second (-), y second (+).
__device__ __forceinline__ float hz_yee(float da, float db, float hz, float dey_x, float ihx, float dex_y, float ihy)
{
    return da * hz - db * (dey_x * ihx - dex_y * ihy);
}

// CPML row of one axis at one index: psi row (-1 outside the layers), b, gain.
struct Row {
    int r;
    float b, g;
};

// The per-index record of an axis read at a wave-uniform index: through the constant address space, so it is a scalar
// load (counted apart from the vector loads of the field rows, which it would otherwise wait behind).
__device__ __forceinline__ yee3d_axis_row uniform_row(const yee3d_axis_row* rows, int index)
{
    typedef const __attribute__((address_space(4))) float ConstF;
    typedef const __attribute__((address_space(4))) int32_t ConstI;
    ConstF* f = (ConstF*)(rows) + 8 * index;
    ConstI* n = (ConstI*)(rows) + 8 * index;
    yee3d_axis_row out;
    out.inv_h = f[0];
    out.inv_e = f[1];
    out.psi_row_h = n[2];
    out.b_h = f[3];
    out.g_h = f[4];
    out.psi_row_e = n[5];
    out.b_e = f[6];
    out.g_e = f[7];
    return out;
}

__device__ __forceinline__ Row h_row(const yee3d_axis_row& a) { return Row{a.psi_row_h, a.b_h, a.g_h}; }
__device__ __forceinline__ Row e_row(const yee3d_axis_row& a) { return Row{a.psi_row_e, a.b_e, a.g_e}; }

// A lane's element of a plane: uniform pointer + byte offset.
__device__ __forceinline__ float ldp(const float* plane, uint32_t bytes)
{
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(plane) + bytes);
}
__device__ __forceinline__ void stp(float* plane, uint32_t bytes, float v)
{
    *reinterpret_cast<float*>(reinterpret_cast<char*>(plane) + bytes) = v;
}

// Symmetric mirror planes (the hi face of cell 0 / n - 2): tangential H = 0 (engine3d.py:513-518).
__device__ __forceinline__ void mirror_h(const yee3d_desc& d, int i, int j, int k, float& vx, float& vy, float& vz)
{
    if ((d.mirror[0] == YEE_MIRROR_SYMMETRIC && i == 0) || (d.mirror[1] == YEE_MIRROR_SYMMETRIC && i == d.nx - 2))
        vy = vz = 0.f;
    if ((d.mirror[2] == YEE_MIRROR_SYMMETRIC && j == 0) || (d.mirror[3] == YEE_MIRROR_SYMMETRIC && j == d.ny - 2))
        vx = vz = 0.f;
    if ((d.mirror[4] == YEE_MIRROR_SYMMETRIC && k == 0) || (d.mirror[5] == YEE_MIRROR_SYMMETRIC && k == d.nz - 2))
        vx = vy = 0.f;
}

// Pole records on cell (i, j, k): each record whose box holds the cell updates its state from E^n of its component
// and corrects the updated value with that face's cb (physics/em3d/engine3d.py:508-530).
__device__ __forceinline__ void apply_poles_3d(const yee3d_desc& d, int i, int j, int k, const float e_old[3],
                                               const float cb[3], float e_new[3])
{
    for (int p = 0; p < d.n_poles; ++p) {
        const yee3d_pole& pl = d.pole[p];
        if (i < pl.i0 || i >= pl.i1 || j < pl.j0 || j >= pl.j1 || k < pl.k0 || k >= pl.k1) continue;
        const int64_t q = ((int64_t)(i - pl.i0) * (pl.j1 - pl.j0) + (j - pl.j0)) * (pl.k1 - pl.k0) + (k - pl.k0);
        const int c = pl.component;
        const float drive = pl.drive[q];
        if (pl.kind == YEE_DRUDE) {
            float jc = pl.state[0][q];
            jc += pl.damping * jc + drive * e_old[c];
            pl.state[0][q] = jc;
            e_new[c] -= cb[c] * jc;
        } else {
            const float pc = pl.state[0][q];
            float dpc = pl.state[1][q];
            dpc += pl.damping * dpc - pl.restoring * pc + drive * e_old[c];
            pl.state[0][q] = pc + dpc;
            pl.state[1][q] = dpc;
            e_new[c] -= cb[c] * pl.inv_dt * dpc;
        }
    }
}

// Point sources on cell (i, j, k) of step n.
__device__ __forceinline__ void add_sources_3d(const yee3d_desc& d, int64_t n, int i, int j, int k, float& ex, float& ey,
                                               float& ez)
{
    for (int s = 0; s < d.n_sources; ++s) {
        const yee_point_source& src = d.source[s];
        if (src.i == i && src.j == j && src.k == k && n < src.wave_len) {
            const float add = __fmul_rn(src.weight, src.wave[n]);
            const float x = ex + add, y = ey + add, z = ez + add;   // selects, not a branch on where to add
            ex = src.component == 0 ? x : ex;
            ey = src.component == 1 ? y : ey;
            ez = src.component == 2 ? z : ez;
        }
    }
}

}  // namespace yee3
