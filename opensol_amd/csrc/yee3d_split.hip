// The 3D Yee step as two launches, H then E, for grids and batches up to kFused3D cells (yee_api.hip): a thread takes one
// cell of a plane through planes_per_tile planes, needs no halo and no barrier, and its waits are few: the old values, ids and
// layer records together, then the coefficients and psi they lead to (ids are read a plane ahead).
//
// What bounds it: small grids, the latency of these loads and of two launches; from about 2M cells, memory (76 B a cell and
// step against the fused kernel's 50; 4.6 TB/s). Lanes run over z and on into the next row, so that wavefronts are full at
// any nz and a block stores one unbroken run. Measured, us a step, against the fused kernel of wavefront tiles before it
// (62 z cells, 4 rows, 4 planes): 64^3 10.7 / 40.2, 97 x 88 x 75 18.3 / 56.7, 140 x 130 x 120 37.2 / 65.2,
// 256^3 293 / 366, 512^3 2120 / 1999.
//
// Fields and the H psi are double-buffered (step n reads set n & 1): the H launch writes H of the other set, the E launch
// reads that and writes E of it; the E psi is read and written by the one thread that owns its cell.
#include "yee3d_after.h"
#include "yee3d_cells.h"

namespace yee3 {

template <class T>
__device__ __forceinline__ const T& at(const T* base, uint32_t byte_offset)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + byte_offset);
}
__device__ __forceinline__ float ldf(const float* base, uint32_t cell) { return at(base, cell * 4u); }
__device__ __forceinline__ void stf(float* base, uint32_t cell, float v)
{
    *reinterpret_cast<float*>(reinterpret_cast<char*>(base) + cell * 4u) = v;
}

// What a face between cells of ids a and b needs beside the entry of a, loaded only where they differ.
struct Mix {
    bool mixed;
    float4 b;    // (ca, cb, eps_r, sigma_e) of b
    float2 a;    // (eps_r, sigma_e) of a
};
__device__ __forceinline__ Mix mix_of(const yee3d_desc& d, int a, int b)
{
    Mix m;
    m.mixed = a != b;
    if (m.mixed) {
        const float2 cb = at(reinterpret_cast<const float2*>(d.table + 2), (uint32_t)b * 32u);
        const float2 mb = at(reinterpret_cast<const float2*>(d.table + 4), (uint32_t)b * 32u);
        m.b = make_float4(cb.x, cb.y, mb.x, mb.y);
        m.a = at(reinterpret_cast<const float2*>(d.table + 4), (uint32_t)a * 32u);
    }
    return m;
}
__device__ __forceinline__ float2 face(const yee3d_desc& d, const Mix& m, float2 own)
{
    if (!m.mixed) return own;
    if (m.a.x < 0.f || m.b.z < 0.f) return m.a.x < 0.f ? make_float2(m.b.x, m.b.y) : own;
    return mixed_face(d.dt, m.a, make_float2(m.b.z, m.b.w));
}

// A thread's cell c = j * nz + k of a plane and its planes [i0, i1).
struct Column {
    uint32_t c;
    int j, k, i0, i1;
};

// The column of this thread in block `block` of an instance: plane cells fastest, 256 a block, in 8 runs, one an XCD
// (consecutive blocks go to the XCDs in turn), so that rows side by side share an L2.
__device__ __forceinline__ bool column_of(const yee3d_desc& d, int block, Column& out)
{
    const uint32_t plane = (uint32_t)d.ny * (uint32_t)d.nz;
    const uint32_t per_plane = ((plane + 255u) / 256u + 7u) & ~7u;
    const uint32_t chunk = (uint32_t)block / per_plane;
    const uint32_t r = (uint32_t)block - chunk * per_plane;
    const uint32_t part = (r & 7u) * (per_plane >> 3) + (r >> 3);
    out.c = part * 256u + threadIdx.x;
    if (out.c >= plane) return false;
    out.j = (int)(out.c / (uint32_t)d.nz);
    out.k = (int)(out.c - (uint32_t)out.j * (uint32_t)d.nz);
    out.i0 = (int)chunk * d.planes_per_tile;
    out.i1 = min(d.nx, out.i0 + d.planes_per_tile);
    return true;
}

// The H update of a block's columns.
__device__ __forceinline__ void h_block(const yee3d_desc& d, int64_t n, int block)
{
    Column q;
    if (!column_of(d, block, q)) return;
    const int par = (int)(n & 1), out = par ^ 1;
    const int nx = d.nx, ny = d.ny, nz = d.nz;
    const int64_t sx = (int64_t)ny * nz;
    const uint32_t c = q.c;
    const int j = q.j, k = q.k;
    const uint32_t row_up = j + 1 < ny ? c + nz : (d.periodic[1] ? (uint32_t)k : c);
    const uint32_t cell_up = k + 1 < nz ? c + 1 : (d.periodic[2] ? c - (nz - 1) : c);
    const yee3d_axis_row ay = at(d.axis_rows[1], (uint32_t)j * 32u), az = at(d.axis_rows[2], (uint32_t)k * 32u);
    const float ihy = ay.inv_h, ihz = az.inv_h;
    const Row ry = h_row(ay), rz = h_row(az);
    const bool mirrored = (d.mirror[0] | d.mirror[1] | d.mirror[2] | d.mirror[3] | d.mirror[4] | d.mirror[5]) != 0;
    float ex, ey, ez;
    int id;
    {
        const int64_t po = (int64_t)q.i0 * sx;
        id = at(d.material + po, c * 2u);
        ex = ldf(d.field[par][0] + po, c);
        ey = ldf(d.field[par][1] + po, c);
        ez = ldf(d.field[par][2] + po, c);
    }
    for (int i = q.i0; i < q.i1; ++i) {
        uint32_t c = q.c, cj = row_up, ck = cell_up;
        asm volatile("" : "+v"(c), "+v"(cj), "+v"(ck));   // 32-bit offsets from uniform pointers in every plane
        const int64_t po = (int64_t)i * sx;
        const int ip = i + 1 < nx ? i + 1 : (d.periodic[0] ? 0 : i);
        const int64_t pn = (int64_t)ip * sx;
        const float2 m = at(reinterpret_cast<const float2*>(d.table), (uint32_t)id * 32u);
        const int id_next = at(d.material + pn, c * 2u);
        const float ex_n = ldf(d.field[par][0] + pn, c), ey_xp = ldf(d.field[par][1] + pn, c),
                    ez_xp = ldf(d.field[par][2] + pn, c);
        const float ez_yp = ldf(d.field[par][2] + po, cj), ex_yp = ldf(d.field[par][0] + po, cj);
        const float ey_zp = ldf(d.field[par][1] + po, ck), ex_zp = ldf(d.field[par][0] + po, ck);
        const float hx = ldf(d.field[par][3] + po, c), hy = ldf(d.field[par][4] + po, c),
                    hz = ldf(d.field[par][5] + po, c);
        const yee3d_axis_row ax = uniform_row(d.axis_rows[0], i);
        const Row rx = h_row(ax);
        const float ihx = ax.inv_h;
        float x0 = 0.f, x1 = 0.f, y0 = 0.f, y1 = 0.f, z0 = 0.f, z1 = 0.f;
        const int64_t px = (int64_t)rx.r * sx;
        const int64_t py = (int64_t)i * d.cpml[1].n_rows * nz;
        const uint32_t qy = (uint32_t)(ry.r * nz + k);
        const int64_t pz = (int64_t)i * ny * d.cpml[2].n_rows;
        const uint32_t qz = (uint32_t)(j * d.cpml[2].n_rows + rz.r);
        if (rx.r >= 0) {
            x0 = ldf(d.cpml[0].psi_h[par][0] + px, c);
            x1 = ldf(d.cpml[0].psi_h[par][1] + px, c);
        }
        if (ry.r >= 0) {
            y0 = ldf(d.cpml[1].psi_h[par][0] + py, qy);
            y1 = ldf(d.cpml[1].psi_h[par][1] + py, qy);
        }
        if (rz.r >= 0) {
            z0 = ldf(d.cpml[2].psi_h[par][0] + pz, qz);
            z1 = ldf(d.cpml[2].psi_h[par][1] + pz, qz);
        }
        const float da = m.x, db = m.y;
        const float dez_y = ez_yp - ez, dey_z = ey_zp - ey;
        const float dex_z = ex_zp - ex, dez_x = ez_xp - ez;
        const float dey_x = ey_xp - ey, dex_y = ex_yp - ex;
        float vx = hx_yee(da, db, hx, dez_y, ihy, dey_z, ihz);
        float vy = hy_yee(da, db, hy, dex_z, ihz, dez_x, ihx);
        float vz = hz_yee(da, db, hz, dey_x, ihx, dex_y, ihy);
        if (rx.r >= 0) {   // x layers: H_y from E_z (+), H_z from E_y (-)
            const float a = psi_next(rx.b, x0, rx.g, dez_x);
            const float b = psi_next(rx.b, x1, rx.g, dey_x);
            stf(d.cpml[0].psi_h[out][0] + px, c, a);
            stf(d.cpml[0].psi_h[out][1] + px, c, b);
            vy += db * a;
            vz -= db * b;
        }
        if (ry.r >= 0) {   // y layers: H_x from E_z (-), H_z from E_x (+)
            const float a = psi_next(ry.b, y0, ry.g, dez_y);
            const float b = psi_next(ry.b, y1, ry.g, dex_y);
            stf(d.cpml[1].psi_h[out][0] + py, qy, a);
            stf(d.cpml[1].psi_h[out][1] + py, qy, b);
            vx -= db * a;
            vz += db * b;
        }
        if (rz.r >= 0) {   // z layers: H_x from E_y (+), H_y from E_x (-)
            const float a = psi_next(rz.b, z0, rz.g, dey_z);
            const float b = psi_next(rz.b, z1, rz.g, dex_z);
            stf(d.cpml[2].psi_h[out][0] + pz, qz, a);
            stf(d.cpml[2].psi_h[out][1] + pz, qz, b);
            vx += db * a;
            vy -= db * b;
        }
        if (mirrored) mirror_h(d, i, j, k, vx, vy, vz);
        stf(d.field[out][3] + po, c, vx);
        stf(d.field[out][4] + po, c, vy);
        stf(d.field[out][5] + po, c, vz);
        ex = ex_n;
        ey = ey_xp;
        ez = ez_xp;
        id = id_next;
    }
}

// The E update of a block's columns.
template <bool POLES>
__device__ __forceinline__ void e_block(const yee3d_desc& d, int64_t n, int block)
{
    Column q;
    if (!column_of(d, block, q)) return;
    const int par = (int)(n & 1), out = par ^ 1;
    const int nx = d.nx, ny = d.ny, nz = d.nz;
    const int64_t sx = (int64_t)ny * nz;
    const uint32_t c = q.c;
    const int j = q.j, k = q.k;
    const bool lo_x = !d.periodic[0], lo_y = j == 0 && !d.periodic[1], lo_z = k == 0 && !d.periodic[2];
    const uint32_t row_up = j + 1 < ny ? c + nz : (d.periodic[1] ? (uint32_t)k : c);
    const uint32_t cell_up = k + 1 < nz ? c + 1 : (d.periodic[2] ? c - (nz - 1) : c);
    const uint32_t row_down = j > 0 ? c - nz : c + (uint32_t)(ny - 1) * nz;
    const uint32_t cell_down = k > 0 ? c - 1 : c + (nz - 1);
    const yee3d_axis_row ay = at(d.axis_rows[1], (uint32_t)j * 32u), az = at(d.axis_rows[2], (uint32_t)k * 32u);
    const float iey = ay.inv_e, iez = az.inv_e;
    const Row ry = e_row(ay), rz = e_row(az);
    float hy_prev = 0.f, hz_prev = 0.f;
    if (q.i0 > 0 || !lo_x) {
        const int64_t pm = (int64_t)(q.i0 > 0 ? q.i0 - 1 : nx - 1) * sx;
        hy_prev = ldf(d.field[out][4] + pm, c);
        hz_prev = ldf(d.field[out][5] + pm, c);
    }
    const auto after = [&](int i) { return i + 1 < nx ? i + 1 : (d.periodic[0] ? 0 : i); };
    // ids a plane ahead, so that the tables are read along with the fields
    int id, id_xp, id_yp, id_zp;
    {
        const uint16_t* ids = d.material + (int64_t)q.i0 * sx;
        id = at(ids, c * 2u);
        id_yp = at(ids, row_up * 2u);
        id_zp = at(ids, cell_up * 2u);
        id_xp = at(d.material + (int64_t)after(q.i0) * sx, c * 2u);
    }
    for (int i = q.i0; i < q.i1; ++i) {
        uint32_t c = q.c, cj = row_up, ck = cell_up, bj = row_down, bk = cell_down;
        asm volatile("" : "+v"(c), "+v"(cj), "+v"(ck), "+v"(bj), "+v"(bk));   // 32-bit offsets from uniform pointers
        const int64_t po = (int64_t)i * sx;
        const float2 own = at(reinterpret_cast<const float2*>(d.table + 2), (uint32_t)id * 32u);
        const Mix mx = mix_of(d, id, id_xp), my = mix_of(d, id, id_yp), mz = mix_of(d, id, id_zp);
        const int ip = after(i), in = after(ip);
        const int id_yp2 = at(d.material + (int64_t)ip * sx, cj * 2u), id_zp2 = at(d.material + (int64_t)ip * sx, ck * 2u);
        const int id_xp2 = at(d.material + (int64_t)in * sx, c * 2u);
        const float ex = ldf(d.field[par][0] + po, c), ey = ldf(d.field[par][1] + po, c),
                    ez = ldf(d.field[par][2] + po, c);
        const float hx = ldf(d.field[out][3] + po, c), hy = ldf(d.field[out][4] + po, c),
                    hz = ldf(d.field[out][5] + po, c);
        float hx_jm = ldf(d.field[out][3] + po, bj), hz_jm = ldf(d.field[out][5] + po, bj);
        float hx_km = ldf(d.field[out][3] + po, bk), hy_km = ldf(d.field[out][4] + po, bk);
        const yee3d_axis_row ax = uniform_row(d.axis_rows[0], i);
        const Row rx = e_row(ax);
        const float iex = ax.inv_e;
        float x0 = 0.f, x1 = 0.f, y0 = 0.f, y1 = 0.f, z0 = 0.f, z1 = 0.f;
        const int64_t px = (int64_t)rx.r * sx;
        const int64_t py = (int64_t)i * d.cpml[1].n_rows * nz;
        const uint32_t qy = (uint32_t)(ry.r * nz + k);
        const int64_t pz = (int64_t)i * ny * d.cpml[2].n_rows;
        const uint32_t qz = (uint32_t)(j * d.cpml[2].n_rows + rz.r);
        if (rx.r >= 0) {
            x0 = ldf(d.cpml[0].psi_e[0] + px, c);
            x1 = ldf(d.cpml[0].psi_e[1] + px, c);
        }
        if (ry.r >= 0) {
            y0 = ldf(d.cpml[1].psi_e[0] + py, qy);
            y1 = ldf(d.cpml[1].psi_e[1] + py, qy);
        }
        if (rz.r >= 0) {
            z0 = ldf(d.cpml[2].psi_e[0] + pz, qz);
            z1 = ldf(d.cpml[2].psi_e[1] + pz, qz);
        }
        if (lo_y) hx_jm = hz_jm = 0.f;
        if (lo_z) hx_km = hy_km = 0.f;
        const float dhz_y = hz - hz_jm, dhy_z = hy - hy_km;
        const float dhx_z = hx - hx_km, dhz_x = hz - hz_prev;
        const float dhy_x = hy - hy_prev, dhx_y = hx - hx_jm;
        const float2 fx = face(d, mx, own), fy = face(d, my, own), fz = face(d, mz, own);
        float vx = fx.x * ex + fx.y * (dhz_y * iey - dhy_z * iez);
        float vy = fy.x * ey + fy.y * (dhx_z * iez - dhz_x * iex);
        float vz = fz.x * ez + fz.y * (dhy_x * iex - dhx_y * iey);
        if (rx.r >= 0) {   // x layers: E_y from H_z (-), E_z from H_y (+)
            const float a = psi_next(rx.b, x0, rx.g, dhz_x);
            const float b = psi_next(rx.b, x1, rx.g, dhy_x);
            stf(d.cpml[0].psi_e[0] + px, c, a);
            stf(d.cpml[0].psi_e[1] + px, c, b);
            vy -= fy.y * a;
            vz += fz.y * b;
        }
        if (ry.r >= 0) {   // y layers: E_x from H_z (+), E_z from H_x (-)
            const float a = psi_next(ry.b, y0, ry.g, dhz_y);
            const float b = psi_next(ry.b, y1, ry.g, dhx_y);
            stf(d.cpml[1].psi_e[0] + py, qy, a);
            stf(d.cpml[1].psi_e[1] + py, qy, b);
            vx += fx.y * a;
            vz -= fz.y * b;
        }
        if (rz.r >= 0) {   // z layers: E_x from H_y (-), E_y from H_x (+)
            const float a = psi_next(rz.b, z0, rz.g, dhy_z);
            const float b = psi_next(rz.b, z1, rz.g, dhx_z);
            stf(d.cpml[2].psi_e[0] + pz, qz, a);
            stf(d.cpml[2].psi_e[1] + pz, qz, b);
            vx -= fx.y * a;
            vy += fy.y * b;
        }
        if constexpr (POLES) {
            const float e_old[3] = {ex, ey, ez};
            const float cb[3] = {fx.y, fy.y, fz.y};
            float e_new[3] = {vx, vy, vz};
            apply_poles_3d(d, i, j, k, e_old, cb, e_new);
            vx = e_new[0];
            vy = e_new[1];
            vz = e_new[2];
        }
        add_sources_3d(d, n, i, j, k, vx, vy, vz);
        stf(d.field[out][0] + po, c, vx);
        stf(d.field[out][1] + po, c, vy);
        stf(d.field[out][2] + po, c, vz);
        hy_prev = hy;
        hz_prev = hz;
        id = id_xp;
        id_xp = id_xp2;
        id_yp = id_yp2;
        id_zp = id_zp2;
    }
}

}  // namespace yee3

// One 3D instance; the descriptor is read in place at the kernel-argument pointer. AFTER: the blocks past a.first take the
// samples of the step before, from the set that this launch only reads. As launches of their own after every step they cost
// what a small grid's update does: 97 x 88 x 75 with a flux plane, a DFT plane and probes took 28.5 us a step with
// five launches, 21 with these two.
template <bool AFTER>
__global__ void __launch_bounds__(256) yee3d_h_kernel(yee3d_desc desc, yee3d_after a, int32_t offset)
{
    typedef const __attribute__((address_space(4))) yee3d_desc ConstDesc;
    const yee3d_desc& d = *(const yee3d_desc*)(ConstDesc*)__builtin_amdgcn_kernarg_segment_ptr();
    if (d.clock != desc.clock) return;
    const int64_t n = *d.clock + offset;
    if (AFTER && (int)blockIdx.x >= a.first) {
        yee3::after_block(d, a, n - 1, (int)blockIdx.x - a.first);
        return;
    }
    if (n >= d.step_limit) return;
    yee3::h_block(d, n, blockIdx.x);
}
template __global__ void yee3d_h_kernel<false>(yee3d_desc, yee3d_after, int32_t);
template __global__ void yee3d_h_kernel<true>(yee3d_desc, yee3d_after, int32_t);

template <bool POLES>
__global__ void __launch_bounds__(256) yee3d_e_kernel(yee3d_desc desc, int32_t offset)
{
    typedef const __attribute__((address_space(4))) yee3d_desc ConstDesc;
    const yee3d_desc& d = *(const yee3d_desc*)(ConstDesc*)__builtin_amdgcn_kernarg_segment_ptr();
    if (d.clock != desc.clock) return;
    const int64_t n = *d.clock + offset;
    if (n >= d.step_limit) return;
    yee3::e_block<POLES>(d, n, blockIdx.x);
}
template __global__ void yee3d_e_kernel<false>(yee3d_desc, int32_t);
template __global__ void yee3d_e_kernel<true>(yee3d_desc, int32_t);

// The H or the E update of many instances: block b belongs to the member whose range [prefix[k], prefix[k + 1]) holds it.
// Blocks of an H launch past prefix[n_inst], rounded up to `first`, take the members' plane samples of the step before, as
// those of a single instance do (six members of 64 to 140 cells a side: 95 us a step, 101 with a
// launch of their own).
template <bool E>
__global__ void __launch_bounds__(256) yee3d_batch_half_kernel(const yee3d_desc* __restrict__ descs,
                                                              const int32_t* __restrict__ prefix,
                                                              const int64_t* __restrict__ sample_prefix, int32_t n_inst,
                                                              int32_t first, int32_t offset)
{
    const int block = blockIdx.x;
    if (!E && block >= first) {
        yee3::sample_members(descs, sample_prefix, n_inst, offset - 1, block - first);
        return;
    }
    int lo = 0, hi = n_inst;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (prefix[mid] <= block) lo = mid; else hi = mid;
    }
    typedef const __attribute__((address_space(4))) yee3d_desc ConstDesc;
    const yee3d_desc& d = *(const yee3d_desc*)((ConstDesc*)descs + lo);
    const int64_t n = *d.clock + offset;
    if (n >= d.step_limit) return;
    const int own = block - prefix[lo];
    if constexpr (!E) yee3::h_block(d, n, own);
    else if (d.n_poles > 0) yee3::e_block<true>(d, n, own);
    else yee3::e_block<false>(d, n, own);
}
template __global__ void yee3d_batch_half_kernel<false>(const yee3d_desc* __restrict__, const int32_t* __restrict__,
                                                        const int64_t* __restrict__, int32_t, int32_t, int32_t);
template __global__ void yee3d_batch_half_kernel<true>(const yee3d_desc* __restrict__, const int32_t* __restrict__,
                                                       const int64_t* __restrict__, int32_t, int32_t, int32_t);
