// Fused 3D Yee step for gfx950: one launch advances a 3D instance by one full step (H update with its CPML on every
// axis, E update with its CPML, point dipole injection); a second, small launch takes what is sampled after a step
// (yee3d_after.h).
//
// It takes instances and batches from kFused3D cells (yee_api.hip) on; smaller ones step in two launches (yee3d_split.hip).
//
// Work decomposition. Arrays are (nx, ny, nz) with z contiguous. A block of 16 wavefronts marches a tile of 64 z cells (one a
// lane) x 14 rows (one a wavefront) along planes_per_tile planes of x. The new H of the plane before stays in registers; a
// row's new H goes to the row above, and the E it loads to the row below, through LDS, so that a plane costs each wavefront
// seven loads and six stores. The H of the row below the tile and of the cells below its first z cell is formed again, by
// two further wavefronts; halo values come from the previous state, which is race-free because the fields and the H CPML psi
// are double-buffered (step n reads set n & 1 and writes set (n & 1) ^ 1); E psi is read and written only by the owner of its
// cell. A plane's loads are in flight during the step of the plane before it.
//
// Boundaries: a periodic axis wraps its indices; on a non-periodic axis indices are clamped to the grid, which makes
// the hi neighbour of the last row the row itself (face partner = the cell itself, and inv_h[n-1] = 0 cancels the
// curl term), and the lo neighbour of row 0 is forced to 0.
//
// What bounds it: memory, 26 B read and 24 B written a cell and step; 512^3 takes 1.64 ms (4.1 TB/s of these; a kernel that
// copies the same arrays takes 1.27). A wavefront's 256 B must be whole cache lines: tiles of 62 cells, as a wavefront with
// its own z halo owns, take 1.9 ms even to copy, since the lines that two blocks share are written in parts. Measured at
// 512^3 on the way here: 62-cell tiles without LDS 2.00 ms (10.6 GB moved), rows through LDS 2.02, 64-cell tiles 1.90 (the
// columns beside the tile cost a line a lane: 2.8 times the reads of L2), without the loads that another wavefront makes 1.64.
//
// Reference semantics (file:line of the reference package open_sol/):
//   H update + CPML    physics/em3d/kernels3d.py:335-400 (update_h_3d), :44-56 (edge_coefficients)
//   E update + CPML    physics/em3d/kernels3d.py:538-610 (update_e_3d), :61-85 (face_coefficients)
//   CPML rows          physics/em3d/boundaries3d.py:208-241 (cpml_slabs)
//   dipole             physics/em3d/sources3d.py:41-75
//   plane flux         physics/em3d/monitors3d.py:90-101; physics/em/monitors.py:22-34, 92-96
//   step order         physics/em3d/engine3d.py:497-554
#include "yee3d_after.h"
#include "yee3d_cells.h"
#include "yee3d_index.h"

namespace yee3 {

constexpr int LANES = yee3idx::kLanes;
constexpr int OWNED = yee3idx::kOwned;
constexpr int ROWS = yee3idx::kRows;
constexpr int WAVES = ROWS + 2;    // a block's wavefronts: the halo row, the owned rows, the halo column
constexpr int LDS_IDS = 512;       // ids whose table is staged in LDS: (da, db, ca, cb) + (eps_r, sigma_e), 12 KiB

__shared__ float4 lds3_coef[LDS_IDS];
__shared__ float2 lds3_mat[LDS_IDS];
// What a plane's step hands on within the block, two planes in turn so that one barrier a plane is enough: the new (H_x,
// H_z) of a row for the row above it; (E_x, E_z) and the id of the next plane of a row for the row below it; the new (H_x,
// H_y) of the cell below a row's first one along z; (E_x, E_y) of the next plane of a row's first cell, and (E_x, E_y, id)
// of the next plane of the cell above its last one.
__shared__ float2 lds3_h[2][ROWS + 1][LANES], lds3_e[2][ROWS + 1][LANES];
__shared__ int lds3_id[2][ROWS + 1][LANES];
__shared__ float2 lds3_below[2][ROWS + 1], lds3_first[2][ROWS + 1];
__shared__ float4 lds3_above[2][ROWS + 1];

// Orders the block's LDS accesses; global loads and stores stay in flight (no thread reads what another one stores).
__device__ __forceinline__ void barrier_lds()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// Stage the table of one instance in LDS (whole block; the barrier is the caller's).
__device__ __forceinline__ void stage_tables(const yee3d_desc& d)
{
    if (d.n_materials > LDS_IDS) return;
    for (int k = threadIdx.x; k < d.n_materials; k += blockDim.x) {
        const float* t = d.table + 8 * k;
        lds3_coef[k] = make_float4(t[0], t[1], t[2], t[3]);
        lds3_mat[k] = make_float2(t[4], t[5]);
    }
}

template <bool LDS>
__device__ __forceinline__ float4 coef(const yee3d_desc& d, int id)
{
    if constexpr (LDS) return lds3_coef[id];
    else return *reinterpret_cast<const float4*>(d.table + 8 * id);
}

template <bool LDS>
__device__ __forceinline__ float2 mat(const yee3d_desc& d, int id)
{
    if constexpr (LDS) return lds3_mat[id];
    else return *reinterpret_cast<const float2*>(d.table + 8 * id + 4);
}

// The face coefficients between cells of ids a (whose entry is `own`) and b.
template <bool LDS>
__device__ __forceinline__ float2 face(const yee3d_desc& d, int a, int b, const float4& own)
{
    if (a == b) return make_float2(own.z, own.w);
    const float2 ma = mat<LDS>(d, a), mb = mat<LDS>(d, b);
    if (ma.x < 0.f || mb.x < 0.f) {
        const float4 c = ma.x < 0.f ? coef<LDS>(d, b) : own;
        return make_float2(c.z, c.w);
    }
    return mixed_face(d.dt, ma, mb);
}

using yee3idx::fold;

// What the step of one plane reads, loaded a plane ahead: E and the id of the next plane (also of the row above the tile, by
// its last row), the old H, and the psi of the layers that the cell lies in.
struct Plane {
    float ex, ey, ez, exu, ezu, hx, hy, hz;
    int id, idu;
    float hp[6];   // x, y, z layers, two each
};

// The value of the lane above (lane 63: 0) and below (lane 0: 0).
__device__ __forceinline__ int lane_above(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, true); }
__device__ __forceinline__ float lane_above(float v) { return __int_as_float(lane_above(__float_as_int(v))); }
__device__ __forceinline__ float lane_below(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}

// Raw buffer access to one plane of an array: its base and size sit in a buffer resource (scalar registers), the lane's
// byte offset in a vector register. An access past the plane reads 0 and writes nothing, so a lane that takes no part has
// the offset OFF instead of a branch around it. (Branches cost more than the accesses here: where paths with and without a
// store join, the wait for an older load has to assume that there was none, and waits for the stores as well.)
typedef __amdgpu_buffer_rsrc_t Rsrc;
constexpr int RSRC_DWORD3 = 0x00020000;   // 32-bit data format, no swizzle (gfx9 buffer resource word 3)
constexpr uint32_t OFF = 0xfffffffeu;     // past any plane, also halved (ids)

__device__ __forceinline__ Rsrc plane_rsrc(const void* base, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, RSRC_DWORD3);
}
__device__ __forceinline__ float ldf(Rsrc r, uint32_t bytes, uint32_t plane = 0)
{
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)bytes, (int)plane, 0));
}
__device__ __forceinline__ int ldid(Rsrc r, uint32_t bytes, uint32_t plane = 0)
{
    return (int)__builtin_amdgcn_raw_buffer_load_b16(r, (int)bytes, (int)plane, 0);
}
__device__ __forceinline__ void stf(Rsrc r, uint32_t bytes, uint32_t plane, float v)
{
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, (int)bytes, (int)plane, 0);
}

typedef const __attribute__((address_space(4))) yee3d_desc ConstDesc;

// One block tile: planes [i0, i1), rows tj * ROWS .. + ROWS - 1 (wavefronts 1..ROWS, one row each), z cells tk * OWNED ..
// + OWNED - 1 (one a lane). Wavefront 0 holds the halo row below. The last wavefront holds the columns beside the tile, 16
// lanes each: the cells below the first z cell (rows 1..ROWS + 1; their H_x and H_y) and above the last one (rows 0..ROWS;
// their E_x, E_y). Each of its loads costs a cache line per lane, so it loads no more than that. Every wavefront reaches every barrier.
// EDGE: any tile. Else no cell of it, halo included, lies in a layer, on a mirror plane, beside a wrap or under a source, and
// the planes i0 - 1..i1 follow each other: each array is one buffer resource for the whole tile, a plane an offset in it.
template <bool LDS, bool POLES, bool EDGE>
__device__ __forceinline__ void tile3d(ConstDesc* desc, int64_t n, int i0, int i1, int tj, int tk)
{
    const yee3d_desc& d = *(const yee3d_desc*)desc;
    const int lane = threadIdx.x & (LANES - 1), wave = wave_index();
    const int nx = d.nx, ny = d.ny, nz = d.nz;
    const bool px = d.periodic[0] != 0, py = d.periodic[1] != 0, pz = d.periodic[2] != 0;
    const int64_t sx = (int64_t)ny * nz;
    const uint32_t plane_bytes = (uint32_t)sx * 4u;
    const int par = (int)(n & 1);

    const bool column = wave == WAVES - 1, last_row = wave == ROWS;
    const int side = lane >> 4;   // of the columns: 0 below, 1 above, 2 and 3 none
    const int kraw = yee3idx::lane_z(tk, !column ? lane : side == 0 ? -1 : LANES);
    const int jraw = yee3idx::row_y(tj, !column ? wave : side == 1 ? lane & 15 : 1 + min(lane & 15, ROWS));
    const int k = fold(kraw, nz, pz), j = fold(jraw, ny, py), ju = fold(jraw + 1, ny, py);
    const bool lone = column || lane == LANES - 1;   // the cell above along z is no other lane's
    const bool k_zero = !pz && kraw < 0, row_zero = !py && jraw < 0;   // below cell 0 of a non-periodic axis: H reads 0
    const bool own = wave > 0 && !column && jraw < ny && yee3idx::lane_owns(lane, kraw, nz);
    const yee3d_axis_row az = d.axis_rows[2][k], ay = d.axis_rows[1][j];
    const Row rz_h = h_row(az), rz_e = e_row(az), ry_h = h_row(ay), ry_e = e_row(ay);
    const float ihy = ay.inv_h, iey = ay.inv_e, ihz = az.inv_h, iez = az.inv_e;
    const uint32_t own_bytes = column && (side > 1 || (lane & 15) > ROWS) ? OFF : (uint32_t)(j * nz + k) * 4u;
    const uint32_t ez_bytes = column && side == 1 ? OFF : own_bytes;
    const uint32_t h_bytes = column && (side == 1 || lane >= ROWS) ? OFF : own_bytes, hz_bytes = column ? OFF : own_bytes;
    const uint32_t up_bytes = (uint32_t)(ju * nz + k) * 4u, store_bytes = own ? own_bytes : OFF;
    // offsets in a plane of the psi arrays of the y and z layers (used in the layers only)
    const uint32_t y_bytes_h = (uint32_t)(ry_h.r * nz + k) * 4u, y_bytes_e = (uint32_t)(ry_e.r * nz + k) * 4u;
    const uint32_t z_bytes_h = (uint32_t)(j * d.cpml[2].n_rows + rz_h.r) * 4u;
    const uint32_t z_bytes_e = (uint32_t)(j * d.cpml[2].n_rows + rz_e.r) * 4u;
    const bool layers = EDGE && __ballot(ry_h.r >= 0 || ry_e.r >= 0 || rz_h.r >= 0 || rz_e.r >= 0) != 0;
    const bool mirrored = EDGE && (d.mirror[0] | d.mirror[1] | d.mirror[2] | d.mirror[3] | d.mirror[4] | d.mirror[5]) != 0;
    bool sources = false;   // whether a source lies in this wavefront's row
    for (int s = 0; EDGE && s < d.n_sources; ++s)
        sources = sources || __ballot(own && d.source[s].j == j && d.source[s].k == k) != 0;

    const float *fex = d.field[par][0], *fey = d.field[par][1], *fez = d.field[par][2], *fhx = d.field[par][3],
                *fhy = d.field[par][4], *fhz = d.field[par][5];
    float *oex = d.field[par ^ 1][0], *oey = d.field[par ^ 1][1], *oez = d.field[par ^ 1][2], *ohx = d.field[par ^ 1][3],
          *ohy = d.field[par ^ 1][4], *ohz = d.field[par ^ 1][5];
    const uint16_t* ids = d.material;
    const yee3d_axis_row* rows_x = d.axis_rows[0];
    // the resource that holds plane i of an array, and the plane's offset in it
    const int64_t base = EDGE ? 0 : (int64_t)(i0 - 1) * sx;
    const uint32_t span = EDGE ? plane_bytes : (uint32_t)(i1 - i0 + 2) * plane_bytes;
    auto res = [&](const float* a, int i) { return plane_rsrc(a + (EDGE ? (int64_t)i * sx : base), span); };
    auto res_id = [&](int i) { return plane_rsrc(ids + (EDGE ? (int64_t)i * sx : base), span >> 1); };
    auto at = [&](int i) { return EDGE ? 0u : (uint32_t)(i - i0 + 1) * plane_bytes; };

    // E and the id of plane i
    auto load_e = [&](int i, float& x, float& y, float& z, int& m, float& xu, float& zu, int& mu) {
        if (last_row) {   // before the others: the wait for those does not have to assume it away
            xu = ldf(res(fex, i), up_bytes, at(i));
            zu = ldf(res(fez, i), up_bytes, at(i));
            mu = ldid(res_id(i), up_bytes >> 1, at(i) >> 1);
        }
        x = ldf(res(fex, i), own_bytes, at(i));
        y = ldf(res(fey, i), own_bytes, at(i));
        z = ldf(res(fez, i), ez_bytes, at(i));
        m = ldid(res_id(i), own_bytes >> 1, at(i) >> 1);
    };
    // the loads of plane i's step
    auto load = [&](int i, int next, const yee3d_axis_row& ax, Plane& p) {
        load_e(next, p.ex, p.ey, p.ez, p.id, p.exu, p.ezu, p.idu);
        p.hx = ldf(res(fhx, i), h_bytes, at(i));
        p.hy = ldf(res(fhy, i), h_bytes, at(i));
        p.hz = ldf(res(fhz, i), hz_bytes, at(i));
        if (!EDGE || (ax.psi_row_h < 0 && !layers)) return;
        ConstDesc* fresh = desc;   // pointers of the layers are read where they are used: with the others they do not fit
        asm volatile("" : "+s"(fresh));
        const yee3d_desc& e = *(const yee3d_desc*)fresh;
        if (ax.psi_row_h >= 0 && own_bytes != OFF) {
            const int64_t q = (int64_t)ax.psi_row_h * sx;
            p.hp[0] = ldp(e.cpml[0].psi_h[par][0] + q, own_bytes);
            p.hp[1] = ldp(e.cpml[0].psi_h[par][1] + q, own_bytes);
        }
        if (ry_h.r >= 0) {
            const int64_t q = (int64_t)i * e.cpml[1].n_rows * nz;
            p.hp[2] = ldp(e.cpml[1].psi_h[par][0] + q, y_bytes_h);
            p.hp[3] = ldp(e.cpml[1].psi_h[par][1] + q, y_bytes_h);
        }
        if (rz_h.r >= 0) {
            const int64_t q = (int64_t)i * ny * e.cpml[2].n_rows;
            p.hp[4] = ldp(e.cpml[2].psi_h[par][0] + q, z_bytes_h);
            p.hp[5] = ldp(e.cpml[2].psi_h[par][1] + q, z_bytes_h);
        }
    };

    float ex, ey, ez;                       // E of the current plane
    int id;
    float exu, ezu, exa, eya;               // and of the row above, and (lone) of the cell above along z
    int idu, ida;
    float hy_prev = 0.f, hz_prev = 0.f;     // new H_y, H_z of the plane before
    int turn = 0;

    // Hands on E of a plane: written before the barrier, read after it.
    auto give = [&](float x, float y, float z, int m) {
        if (!column) {
            lds3_e[turn][wave][lane] = make_float2(x, z);
            lds3_id[turn][wave][lane] = m;
            if (lane == 0) lds3_first[turn][wave] = make_float2(x, y);
        } else if (side == 1 && (lane & 15) <= ROWS) {
            lds3_above[turn][lane & 15] = make_float4(x, y, __int_as_float(m), 0.f);
        }
    };
    auto take = [&](float xu, float zu, int mu) {
        const float2 up = lds3_e[turn][min(wave + 1, ROWS)][lane];
        const int up_id = lds3_id[turn][min(wave + 1, ROWS)][lane];
        const float4 above = lds3_above[turn][min(wave, ROWS)];
        exu = last_row ? xu : up.x;
        ezu = last_row ? zu : up.y;
        idu = last_row ? mu : up_id;
        const float2 next = lds3_first[turn][min(lane + 1, ROWS)];   // of the columns: the cell above along z is the row's first
        exa = column ? next.x : above.x;
        eya = column ? next.y : above.y;
        ida = __float_as_int(above.z);
    };

    // New H of plane i; the owners write it, and E of the plane (whole; i >= i0).
    auto step = [&](int i, bool whole, const yee3d_axis_row& ax, const Plane& p) {
        ConstDesc* fresh = desc;
        asm volatile("" : "+s"(fresh));
        const yee3d_desc& e = *(const yee3d_desc*)fresh;
        const int out = par ^ 1;
        float ep[6];   // psi of the E update, in flight during the H update
        if (EDGE && whole && (layers || ax.psi_row_e >= 0)) {
            if (own && ax.psi_row_e >= 0) {
                const int64_t q = (int64_t)ax.psi_row_e * sx;
                ep[0] = ldp(e.cpml[0].psi_e[0] + q, own_bytes);
                ep[1] = ldp(e.cpml[0].psi_e[1] + q, own_bytes);
            }
            if (own && ry_e.r >= 0) {
                const int64_t q = (int64_t)i * e.cpml[1].n_rows * nz;
                ep[2] = ldp(e.cpml[1].psi_e[0] + q, y_bytes_e);
                ep[3] = ldp(e.cpml[1].psi_e[1] + q, y_bytes_e);
            }
            if (own && rz_e.r >= 0) {
                const int64_t q = (int64_t)i * ny * e.cpml[2].n_rows;
                ep[4] = ldp(e.cpml[2].psi_e[0] + q, z_bytes_e);
                ep[5] = ldp(e.cpml[2].psi_e[1] + q, z_bytes_e);
            }
        }
        const bool store = whole && own;
        const float4 c = coef<LDS>(d, id);
        const float da = c.x, db = c.y, ihx = ax.inv_h;
        const float above_x = lane_above(ex), above_y = lane_above(ey), above_z = lane_above(ez);
        const float ex_zp = lone ? exa : above_x, ey_zp = lone ? eya : above_y, ez_yp = column ? above_z : ezu;
        const float dez_y = ez_yp - ez, dey_z = ey_zp - ey;
        const float dex_z = ex_zp - ex, dez_x = p.ez - ez;
        const float dey_x = p.ey - ey, dex_y = exu - ex;
        float vx = hx_yee(da, db, p.hx, dez_y, ihy, dey_z, ihz);
        float vy = hy_yee(da, db, p.hy, dex_z, ihz, dez_x, ihx);
        float vz = hz_yee(da, db, p.hz, dey_x, ihx, dex_y, ihy);
        if (EDGE && ax.psi_row_h >= 0) {   // x layers: H_y from E_z (+), H_z from E_y (-)
            const float a = psi_next(ax.b_h, p.hp[0], ax.g_h, dez_x);
            const float b = psi_next(ax.b_h, p.hp[1], ax.g_h, dey_x);
            if (store) {
                const int64_t q = (int64_t)ax.psi_row_h * sx;
                stp(e.cpml[0].psi_h[out][0] + q, own_bytes, a);
                stp(e.cpml[0].psi_h[out][1] + q, own_bytes, b);
            }
            vy += db * a;
            vz -= db * b;
        }
        if (EDGE && ry_h.r >= 0) {   // y layers: H_x from E_z (-), H_z from E_x (+)
            const float a = psi_next(ry_h.b, p.hp[2], ry_h.g, dez_y);
            const float b = psi_next(ry_h.b, p.hp[3], ry_h.g, dex_y);
            if (store) {
                const int64_t q = (int64_t)i * e.cpml[1].n_rows * nz;
                stp(e.cpml[1].psi_h[out][0] + q, y_bytes_h, a);
                stp(e.cpml[1].psi_h[out][1] + q, y_bytes_h, b);
            }
            vx -= db * a;
            vz += db * b;
        }
        if (EDGE && rz_h.r >= 0) {   // z layers: H_x from E_y (+), H_y from E_x (-)
            const float a = psi_next(rz_h.b, p.hp[4], rz_h.g, dey_z);
            const float b = psi_next(rz_h.b, p.hp[5], rz_h.g, dex_z);
            if (store) {
                const int64_t q = (int64_t)i * ny * e.cpml[2].n_rows;
                stp(e.cpml[2].psi_h[out][0] + q, z_bytes_h, a);
                stp(e.cpml[2].psi_h[out][1] + q, z_bytes_h, b);
            }
            vx += db * a;
            vy -= db * b;
        }
        if (EDGE && mirrored) mirror_h(e, i, j, k, vx, vy, vz);
        if (whole) {
            stf(res(ohx, i), store_bytes, at(i), vx);
            stf(res(ohy, i), store_bytes, at(i), vy);
            stf(res(ohz, i), store_bytes, at(i), vz);
            if (!column)
                lds3_h[turn][wave][lane] = EDGE && row_zero ? make_float2(0.f, 0.f) : make_float2(vx, vz);
            else if (side == 0 && lane < ROWS)
                lds3_below[turn][lane + 1] = EDGE && k_zero ? make_float2(0.f, 0.f) : make_float2(vx, vy);
        }
        give(p.ex, p.ey, p.ez, p.id);
        const int id_up = idu, id_far = ida;
        barrier_lds();
        take(p.exu, p.ezu, p.idu);
        if (whole) {
            const float2 row = lds3_h[turn][min(max(wave - 1, 0), ROWS)][lane], first = lds3_below[turn][min(wave, ROWS)];
            const float below_x = lane_below(vx), below_y = lane_below(vy);
            const float hx_km = lane == 0 ? first.x : below_x, hy_km = lane == 0 ? first.y : below_y;
            const int id_above = lane_above(id), id_zp = lone ? id_far : id_above;
            const float dhz_y = vz - row.y, dhy_z = vy - hy_km;
            const float dhx_z = vx - hx_km, dhz_x = vz - hz_prev;
            const float dhy_x = vy - hy_prev, dhx_y = vx - row.x;
            const float iex = ax.inv_e;
            float2 fx = make_float2(c.z, c.w), fy = fx, fz = fx;
            if (__ballot((id != p.id) | (id != id_up) | (id != id_zp)) != 0) {
                fx = face<LDS>(d, id, p.id, c);
                fy = face<LDS>(d, id, id_up, c);
                fz = face<LDS>(d, id, id_zp, c);
            }
            float wx = fx.x * ex + fx.y * (dhz_y * iey - dhy_z * iez);
            float wy = fy.x * ey + fy.y * (dhx_z * iez - dhz_x * iex);
            float wz = fz.x * ez + fz.y * (dhy_x * iex - dhx_y * iey);
            if (EDGE && own && ax.psi_row_e >= 0) {   // x layers: E_y from H_z (-), E_z from H_y (+)
                const int64_t q = (int64_t)ax.psi_row_e * sx;
                const float a = psi_next(ax.b_e, ep[0], ax.g_e, dhz_x);
                const float b = psi_next(ax.b_e, ep[1], ax.g_e, dhy_x);
                stp(e.cpml[0].psi_e[0] + q, own_bytes, a);
                stp(e.cpml[0].psi_e[1] + q, own_bytes, b);
                wy -= fy.y * a;
                wz += fz.y * b;
            }
            if (EDGE && own && ry_e.r >= 0) {   // y layers: E_x from H_z (+), E_z from H_x (-)
                const int64_t q = (int64_t)i * e.cpml[1].n_rows * nz;
                const float a = psi_next(ry_e.b, ep[2], ry_e.g, dhz_y);
                const float b = psi_next(ry_e.b, ep[3], ry_e.g, dhx_y);
                stp(e.cpml[1].psi_e[0] + q, y_bytes_e, a);
                stp(e.cpml[1].psi_e[1] + q, y_bytes_e, b);
                wx += fx.y * a;
                wz -= fz.y * b;
            }
            if (EDGE && own && rz_e.r >= 0) {   // z layers: E_x from H_y (-), E_y from H_x (+)
                const int64_t q = (int64_t)i * ny * e.cpml[2].n_rows;
                const float a = psi_next(rz_e.b, ep[4], rz_e.g, dhy_z);
                const float b = psi_next(rz_e.b, ep[5], rz_e.g, dhx_z);
                stp(e.cpml[2].psi_e[0] + q, z_bytes_e, a);
                stp(e.cpml[2].psi_e[1] + q, z_bytes_e, b);
                wx -= fx.y * a;
                wy += fy.y * b;
            }
            if constexpr (POLES) {
                const float e_old[3] = {ex, ey, ez};
                const float cb[3] = {fx.y, fy.y, fz.y};
                float e_new[3] = {wx, wy, wz};
                if (own) apply_poles_3d(e, i, j, k, e_old, cb, e_new);
                wx = e_new[0];
                wy = e_new[1];
                wz = e_new[2];
            }
            if (EDGE && sources && own) add_sources_3d(e, n, i, j, k, wx, wy, wz);
            stf(res(oex, i), store_bytes, at(i), wx);
            stf(res(oey, i), store_bytes, at(i), wy);
            stf(res(oez, i), store_bytes, at(i), wz);
        }
        hy_prev = vy;
        hz_prev = vz;
        ex = p.ex;
        ey = p.ey;
        ez = p.ez;
        id = p.id;
        turn ^= 1;
    };

    // the first plane whose H is formed here: i0 - 1 for H_y, H_z of the plane before (0 below a non-periodic cell 0)
    const bool before = !EDGE || i0 > 0 || px;
    const int first = before ? (i0 > 0 ? i0 - 1 : nx - 1) : i0;
    auto after = [&](int i) { return i + 1 < nx ? i + 1 : (px ? 0 : nx - 1); };
    Plane a, b;
    yee3d_axis_row ax = uniform_row(rows_x, first), ax_next = uniform_row(rows_x, before ? i0 : after(i0));
    load_e(first, ex, ey, ez, id, b.exu, b.ezu, b.idu);
    load(first, before ? i0 : after(i0), ax, a);
    give(ex, ey, ez, id);
    barrier_lds();
    take(b.exu, b.ezu, b.idu);
    turn ^= 1;
    int i = i0;
    if (before) {
        load(i0, after(i0), ax_next, b);
        step(first, false, ax, a);
        a = b;
        ax = ax_next;
        ax_next = uniform_row(rows_x, after(i0));
    }
    // The next plane's loads are in flight during a plane's step; the last plane has nothing left to load.
    while (i + 1 < i1) {
        const yee3d_axis_row ax_far = uniform_row(rows_x, min(i + 2, nx - 1));
        load(i + 1, after(i + 1), ax_next, b);
        step(i, true, ax, a);
        a = b;
        ++i;
        ax = ax_next;
        ax_next = ax_far;
    }
    step(i, true, ax, a);
}

// Whether a block tile is an inner one (inner_tile3d). Stages the tables; ends in a barrier of the whole block.
__device__ __forceinline__ bool inner_block(const yee3d_desc& d, int i0, int i1, int tj, int tk)
{
    stage_tables(d);
    const int j0 = yee3idx::row_y(tj, 0), j1 = min(d.ny, yee3idx::row_y(tj, ROWS + 1) + 1);
    const int k0 = yee3idx::lane_z(tk, -1), k1 = min(d.nz, yee3idx::lane_z(tk, OWNED) + 1);
    bool edge = i0 < 1 || i1 >= d.nx || j0 < 0 || j1 >= d.ny || k0 < 0 || k1 >= d.nz ||
                (int64_t)d.ny * d.nz * 4 * (i1 - i0 + 2) >= OFF;
    if (!edge) {
        auto layer = [&](int axis, int i) {
            const yee3d_axis_row& r = d.axis_rows[axis][i];
            return r.psi_row_h >= 0 || r.psi_row_e >= 0;
        };
        const int t = threadIdx.x;
        for (int i = i0 - 1 + t; i <= i1; i += blockDim.x) edge = edge || layer(0, i);
        if (j0 + t < j1) edge = edge || layer(1, j0 + t);
        if (k0 + t < k1) edge = edge || layer(2, k0 + t);
        if (t < d.n_sources) {
            const yee_point_source& s = d.source[t];
            edge = edge || (s.i >= i0 && s.i < i1 && s.j >= j0 && s.j < j1 && s.k >= k0 && s.k < k1);
        }
        // symmetric mirror planes: the hi face of cell 0 / n - 2
        edge = edge || (d.mirror[0] && i0 < 2) || (d.mirror[1] && i1 > d.nx - 2) || (d.mirror[2] && j0 < 1) ||
               (d.mirror[3] && j1 > d.ny - 2) || (d.mirror[4] && k0 < 1) || (d.mirror[5] && k1 > d.nz - 2);
    }
    return !__syncthreads_or(edge);
}

// The tile of block `block` of one instance: z tile fastest, then y tile, then x chunk.
template <bool POLES>
__device__ __forceinline__ void step_block(ConstDesc* desc, int64_t n, int block)
{
    const yee3d_desc& d = *(const yee3d_desc*)desc;
    const int tiles_j = yee3idx::tiles_along(d.ny, yee3idx::kRows), tiles_k = yee3idx::tiles_along(d.nz, OWNED);
    const yee3idx::TileCoords c = yee3idx::tile_coords(block, tiles_j, tiles_k);
    const int i0 = c.ic * d.planes_per_tile;
    const int i1 = min(d.nx, i0 + d.planes_per_tile);
    const bool inner = inner_block(d, i0, i1, c.tj, c.tk) && !POLES;   // and the barrier that the tables need
    const bool lds = d.n_materials <= LDS_IDS;
    if (inner && lds)
        tile3d<true, false, false>(desc, n, i0, i1, c.tj, c.tk);
    else if (lds)
        tile3d<true, POLES, true>(desc, n, i0, i1, c.tj, c.tk);
    else
        tile3d<false, POLES, true>(desc, n, i0, i1, c.tj, c.tk);
}

// Consecutive workgroups go to the 8 XCDs in turn: block b of a grid of a multiple of 8 takes part b % 8 of the tiles, so
// that tiles side by side share an L2.
__device__ __forceinline__ int xcd_block() { return (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3); }

}  // namespace yee3

// One 3D instance, one tile per block. The descriptor is read in place at the kernel-argument pointer.
template <bool POLES>
__global__ void __launch_bounds__(64 * yee3::WAVES) yee3d_step_kernel(yee3d_desc desc, int32_t blocks, int32_t offset)
{
    yee3::ConstDesc* d = (yee3::ConstDesc*)__builtin_amdgcn_kernarg_segment_ptr();
    if (d->clock != desc.clock) return;
    const int block = yee3::xcd_block();
    if (block >= blocks) return;
    const int64_t n = *d->clock + offset;
    if (n >= d->step_limit) return;
    yee3::step_block<POLES>(d, n, block);
}

// Many 3D instances of uneven sizes in one launch: block b belongs to the instance whose block range
// [prefix[k], prefix[k+1]) holds it, so a block stages one instance's table. Each instance runs on its own clock
// and stops at its own step limit; members with dispersive poles take the E update that carries them.
__global__ void __launch_bounds__(64 * yee3::WAVES) yee3d_batch_kernel(const yee3d_desc* __restrict__ descs,
                                                          const int32_t* __restrict__ prefix, int32_t n_inst,
                                                          int32_t offset)
{
    const int block = yee3::xcd_block();
    if (block >= prefix[n_inst]) return;
    int lo = 0, hi = n_inst;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (prefix[mid] <= block) lo = mid; else hi = mid;
    }
    // Read the descriptor through the constant address space: its fields become scalar loads, as a kernel argument's.
    yee3::ConstDesc* d = (yee3::ConstDesc*)descs + lo;
    const int64_t n = *d->clock + offset;
    if (n >= d->step_limit) return;
    const int own = block - prefix[lo];
    if (d->n_poles > 0)   // the E update with the member's dispersive-pole records (block-uniform: one member per block)
        yee3::step_block<true>(d, n, own);
    else
        yee3::step_block<false>(d, n, own);
}

template __global__ void yee3d_step_kernel<false>(yee3d_desc, int32_t, int32_t);
template __global__ void yee3d_step_kernel<true>(yee3d_desc, int32_t, int32_t);

// Samples after step n = *clock + offset (after_block). The descriptor is read in place.
__global__ void __launch_bounds__(256) yee3d_after_kernel(yee3d_desc desc, yee3d_after a, int32_t offset)
{
    typedef const __attribute__((address_space(4))) yee3d_desc ConstDesc;
    const yee3d_desc& d = *(const yee3d_desc*)(ConstDesc*)__builtin_amdgcn_kernarg_segment_ptr();
    if (d.clock != desc.clock) return;
    yee3::after_block(d, a, *d.clock + offset, blockIdx.x);
}

// Samples of many instances after their step *clock + offset, in one launch (sample_members).
__global__ void __launch_bounds__(256) yee3d_batch_sample_kernel(const yee3d_desc* __restrict__ descs,
                                                                const int64_t* __restrict__ prefix, int32_t n_inst,
                                                                int32_t offset)
{
    yee3::sample_members(descs, prefix, n_inst, offset, blockIdx.x);
}

namespace yee3 {

// Mirror face `face` (0 x_lo .. 5 z_hi) of one instance after step n, cell t of the face: symmetric, the normal E on
// the plane (the hi face of cell 0 / n - 2) = 0; antisymmetric, the ghost cell's (0 / n - 1) tangential E = minus its
// inner neighbour's (1 / n - 2) (physics/em3d/engine3d.py:531-540). The host launches the symmetric faces first, then
// the antisymmetric ones in face order, as the reference writes its zero rows before its images.
__device__ __forceinline__ void mirror_cell(const yee3d_desc& d, int64_t n, int face, int64_t t)
{
    if (n >= d.step_limit) return;
    const int a = face >> 1, hi = face & 1;
    const int b = a == 0 ? 1 : 0, c = a == 2 ? 1 : 2;   // the two tangential axes, in grid order
    const int32_t ext[3] = {d.nx, d.ny, d.nz};
    if (t >= (int64_t)ext[b] * ext[c]) return;
    int idx[3];
    idx[b] = (int)(t / ext[c]);
    idx[c] = (int)(t % ext[c]);
    const int64_t stride[3] = {(int64_t)d.ny * d.nz, d.nz, 1};
    const int set = (int)((n & 1) ^ 1);
    if (d.mirror[face] == YEE_MIRROR_SYMMETRIC) {
        idx[a] = hi ? ext[a] - 2 : 0;
        d.field[set][a][idx[0] * stride[0] + idx[1] * stride[1] + idx[2]] = 0.f;
    } else if (d.mirror[face] == YEE_MIRROR_ANTISYMMETRIC) {
        idx[a] = hi ? ext[a] - 1 : 0;
        const int64_t ghost = idx[0] * stride[0] + idx[1] * stride[1] + idx[2];
        const int64_t inner = ghost + (hi ? -stride[a] : stride[a]);
        d.field[set][b][ghost] = -d.field[set][b][inner];
        d.field[set][c][ghost] = -d.field[set][c][inner];
    }
}

}  // namespace yee3

// Mirror face `face` after step n = *clock + offset, one lane per cell of the face. The descriptor is read in place at
// the kernel-argument pointer: the field table is indexed by runtime axes.
__global__ void __launch_bounds__(256) yee3d_mirror_kernel(yee3d_desc desc, int32_t face, int32_t offset)
{
    typedef const __attribute__((address_space(4))) yee3d_desc ConstDesc;
    const yee3d_desc& d = *(const yee3d_desc*)(ConstDesc*)__builtin_amdgcn_kernarg_segment_ptr();
    if (d.clock != desc.clock) return;
    yee3::mirror_cell(d, *d.clock + offset, face, (int64_t)blockIdx.x * blockDim.x + threadIdx.x);
}

// Face `face` of the batch's members whose mirror there is of `kind`: blockIdx.y is the member, blockIdx.x * 256 +
// lane the face cell (the grid spans the largest face; the rest return at once). The host launches the kinds and faces
// in the single-instance order.
__global__ void __launch_bounds__(256) yee3d_batch_mirror_kernel(const yee3d_desc* __restrict__ descs, int32_t face,
                                                                int32_t kind, int32_t offset)
{
    typedef const __attribute__((address_space(4))) yee3d_desc ConstDesc;
    const yee3d_desc& d = *(const yee3d_desc*)((ConstDesc*)descs + blockIdx.y);
    if (d.mirror[face] == kind)
        yee3::mirror_cell(d, *d.clock + offset, face, (int64_t)blockIdx.x * blockDim.x + threadIdx.x);
}

// The probes of a batch's members: block k serves member k (members without probes return at once).
__global__ void __launch_bounds__(256) yee3d_batch_probe_kernel(const yee3d_desc* __restrict__ descs, int32_t offset)
{
    typedef const __attribute__((address_space(4))) yee3d_desc ConstDesc;
    const yee3d_desc& d = *(const yee3d_desc*)((ConstDesc*)descs + blockIdx.x);
    if (d.probes.n_probes > 0) yee3::probes_3d(d, *d.clock + offset);
}

// Advance the clocks of a 3D batch by k steps, each bounded by its instance's step limit.
__global__ void yee_clock_advance_batch3d(const yee3d_desc* __restrict__ descs, int32_t n_inst, int64_t k)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_inst) {
        int64_t* clock = descs[i].clock;
        const int64_t v = *clock + k;
        *clock = v < descs[i].step_limit ? v : descs[i].step_limit;
    }
}
