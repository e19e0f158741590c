// Several 2D Yee steps per launch for gfx950: a block holds a window of the grid in registers, advances it by `steps`
// steps and writes the part of it that is still valid, so the state streams from and to HBM once per launch instead of
// once per step, and a small grid pays one launch for many steps.
//
// Work decomposition. A block of NW wavefronts holds a window of 64 * VEC columns by NW * R rows: a
// lane holds VEC adjacent columns of R rows (E_z, H_x, H_y and, in windows that reach a CPML layer, their psi). Each
// step makes one more row and column on every side of the window invalid; the block owns what is left after `steps`
// steps, and the halo around it is recomputed from the state before the launch, so no block reads what another one
// writes. Neighbours along y are lane shifts (DPP), neighbours along x are registers of the same lane, and the one row
// that passes between wavefronts per half step goes through LDS; the rows that do not need it are computed on the near
// side of the barrier.
//
// What bounds it. A step costs 174 instructions for the 8 cells of a lean E_z lane of one column (a tall one holds 16), 30 to
// 43 a cell in general windows; a large grid is bound by the windows' loads and stores (43 ns per 128 x 64 window of 10
// steps, 172 KB: 4 TB/s, with 35 ns at 0 steps extrapolated), a small one by the two rounds of loads before the first step
// (about 4 us of the 9 a 7-step launch takes). Two blocks of 8 wavefronts a CU, so that one loads while the other steps: one
// block of 16 wavefronts and 128 x 128 cells took 88 us a step at 8192^2 where this took 65 (10 steps a launch; 61 now).
// One step a launch moves the whole state and took 343. Material tables: read once, into one coefficient a cell or face, when all
// materials are lossless with one mu_r (the usual case); the general form keeps or looks up all four.
//
// The state arrays stay double-buffered: launch k of a call reads set (clock + k) & 1 and writes the other one, and the
// host makes the number of launches odd for an odd number of steps, so state n ends in set n & 1.
//
// Two forms of a window: the lean one lies, halo included, inside the grid and outside every CPML layer; the general
// one takes grid edges, periodic wraps and CPML. Cells outside the grid take a table entry of zeros, so they stay 0
// without selects. Sheet sources and flux lines are applied in both.
//
// EXTRA windows also take the DFT regions, the field probes and a Drude pole of an E_z instance, which one-step launches
// serve with two kernels more a step: a sampled cell or probe is taken from the registers of the window that owns it, the
// pole's current lives in registers beside E_z (its drive in LDS) and passes from launch to launch through two arrays in
// turn. They are instantiations of their own: the current costs the registers of half a field.
#pragma once

#include "yee2d_cells.h"

namespace yee {

__shared__ float4 lds_coef[kMultiIds];
__shared__ float4 lds_row[2 * kMultiRowsMax];             // x constants of a window row: (inv, b, g, psi bits) of h and of e
__shared__ float lds_wave[YEE_MAX_SOURCES * kMultiMax];   // source values of the launch's steps
__shared__ float lds_profile[YEE_MAX_SOURCES * 128];      // source profiles along the window (0 past their span)
__shared__ float lds_up[kMultiWavesMax * 128];            // the row each wavefront hands down (its lowest)
__shared__ float lds_down[kMultiWavesMax * 128];          // the row each wavefront hands up (its highest)
__shared__ float lds_sigma[kMultiIds / 2];                // H_z: sigma_e per id
__shared__ float lds_drive[kMultiCells];                  // Drude pole: drive of the window's cells, by lane

// value of the next / previous lane (0 past the wavefront's ends, which only halo columns see)
__device__ __forceinline__ float lane_next(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));   // wave_shl:1
}
__device__ __forceinline__ float lane_prev(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));   // wave_shr:1
}

// A float at a wave-uniform address, through the constant address space: a scalar load.
__device__ __forceinline__ float uniform_float(const float* p)
{
    typedef const __attribute__((address_space(4))) float ConstF;
    return *(ConstF*)p;
}

__device__ __forceinline__ float4 coef_at(uint32_t byte_offset)
{
    return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(lds_coef) + byte_offset);
}

// Sheet sources and flux lines (bits of d.source, d.monitor) that reach a window: a source with any of its cells (or any
// window that wraps around a periodic axis), a flux line with owned ones.
struct WindowRecords {
    uint32_t sources, monitors, regions;   // regions: DFT regions with owned cells (EXTRA)
};

struct Window {
    int i0, i1, c0, c1;   // owned rows and columns
    int w0, k0;           // first row and column, halo included
    int rows;             // rows of the window
};

__device__ __forceinline__ WindowRecords window_records(const yee2d_desc& d, const Window& w, int columns)
{
    WindowRecords out{0, 0, 0};
    const bool wrap_x = d.periodic_x != 0 && (w.w0 < 0 || w.w0 + w.rows > d.nx);
    const bool wrap_y = d.periodic_y != 0 && (w.k0 < 0 || w.k0 + columns > d.ny);
    for (int s = 0; s < d.n_sources; ++s) {
        const yee_line_source& src = d.source[s];
        const bool row = src.axis == 1;
        const int r0 = row ? src.line : src.lo, r1 = row ? src.line + 1 : src.hi;
        const int k0 = row ? src.lo : src.line, k1 = row ? src.hi : src.line + 1;
        if ((wrap_x || (r0 < w.w0 + w.rows && r1 > w.w0)) && (wrap_y || (k0 < w.k0 + columns && k1 > w.k0)))
            out.sources |= 1u << s;
    }
    for (int m = 0; m < d.n_monitors; ++m) {
        const yee_flux_line& mon = d.monitor[m];
        const bool row = mon.normal == 0;
        const int r0 = row ? mon.position : mon.lo, r1 = row ? mon.position + 1 : mon.hi;
        const int k0 = row ? mon.lo : mon.position, k1 = row ? mon.hi : mon.position + 1;
        if (r0 < w.i1 && r1 > w.i0 && k0 < w.c1 && k1 > w.c0) out.monitors |= 1u << m;
    }
    return out;
}

// DFT regions with sampled cells among the owned ones (by their bounding boxes).
__device__ __forceinline__ uint32_t window_regions(const yee2d_desc& d, const Window& w)
{
    uint32_t out = 0;
    for (int k = 0; k < d.n_dft; ++k) {
        const yee_dft_region& g = d.dft[k];
        if (g.start[0] < w.i1 && g.start[0] + g.stride[0] * (g.count[0] - 1) >= w.i0 && g.start[1] < w.c1 &&
            g.start[1] + g.stride[1] * (g.count[1] - 1) >= w.c0)
            out |= 1u << k;
    }
    return out;
}

// Whether a window, halo included, may meet the box of a Drude pole (one that wraps around a periodic axis may).
__device__ __forceinline__ bool window_pole(const yee2d_desc& d, const Window& w, int columns)
{
    if (d.n_poles == 0) return false;
    const yee_pole& p = d.pole[0];
    const bool wrap_x = d.periodic_x != 0 && (w.w0 < 0 || w.w0 + w.rows > d.nx);
    const bool wrap_y = d.periodic_y != 0 && (w.k0 < 0 || w.k0 + columns > d.ny);
    return (wrap_x || (p.i0 < w.w0 + w.rows && p.i1 > w.w0)) && (wrap_y || (p.j0 < w.k0 + columns && p.j1 > w.k0));
}

template <int VEC>
__device__ __forceinline__ void load_n(const float* __restrict__ p, float out[VEC])
{
    if constexpr (VEC == 1) out[0] = p[0];
    else ldv<VEC>(p, out);
}

template <int VEC>
__device__ __forceinline__ void store_n(float* __restrict__ p, const float v[VEC])
{
    if constexpr (VEC == 1) __builtin_nontemporal_store(v[0], p);
    else stv<VEC>(p, v);
}

// `v` where `bits` are set, 0 where none are: what a recursion takes where there is no psi. Its factors are 0 there as well,
// but 0 times an infinite difference is NaN, and an overflowed field stays what the one-step kernels make of it. An AND with
// bits in a vector register: 300 steps of 1031 x 773 E_z take 0.83 ms so, 0.79 without it, 0.98 with selects on lane masks or
// scalar branches around the recursions, which the general windows have no scalar registers left for (8192^2 E_z, 40 steps:
// 2.39, 2.38 and 2.65 ms). Windows that reach no y layer have forms without its recursions (0.84 and 2.48 ms if they had not;
// 1370 steps of 270 x 120 cells, periodic along y, 2.16 and 2.26).
__device__ __forceinline__ float keep_bits(uint32_t bits, float v) { return __uint_as_float(bits & __float_as_uint(v)); }
__device__ __forceinline__ float keep_bits(float bits, float v) { return keep_bits(__float_as_uint(bits), v); }
// `v` where `bits` are set, `old` where none are.
__device__ __forceinline__ float pick_bits(uint32_t bits, float v, float old)
{
    return __uint_as_float((bits & __float_as_uint(v)) | (~bits & __float_as_uint(old)));
}

// Columns of a lane and their y constants; the lean form knows that all of them are inside the grid's bulk, and without YL
// none lies in a y layer.
template <int VEC, bool EDGE, bool YL>
struct LaneColumns {
    static_assert(!EDGE || VEC == 1, "general windows hold one column a lane: two beside each other may fold apart");
    int j;                   // first column before folding
    bool owner;
    uint32_t at[VEC];        // column of the grid (a stand-in of 0 outside it)
    bool in[VEC], last[VEC]; // inside the grid; the last column of a bounded axis
    bool stays[VEC];         // fx keeps its value: the last column of a bounded axis, or outside the grid
    int ry_h[VEC], ry_e[VEC];
    float inv_e[VEC], inv_h[VEC], b_h[VEC], g_h[VEC], b_e[VEC], g_e[VEC];
    uint32_t psi_h[VEC], psi_e[VEC], moves[VEC];   // all bits set, or none: has a psi row; not `stays` (keep_bits)

    // positions, and the loads that need nothing loaded before
    __device__ __forceinline__ void begin(const yee2d_desc& d, const Window& w)
    {
        const int lane = threadIdx.x & (YEE_WAVE - 1);
        j = w.k0 + VEC * lane;
        owner = j >= w.c0 && j < w.c1;
        at[0] = (uint32_t)j;
        if constexpr (EDGE) {
            const int ny = d.ny;
            const bool py = d.periodic_y != 0;
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                int c = j + k;
                if (py) {
                    c %= ny;
                    c = c < 0 ? c + ny : c;
                }
                in[k] = c >= 0 && c < ny;
                at[k] = in[k] ? (uint32_t)c : 0u;
                last[k] = c == ny - 1 && !py;
                stays[k] = last[k] || !in[k];
                inv_e[k] = d.inv_dy_e[at[k]];
                inv_h[k] = d.inv_dy_h[at[k]];
                ry_h[k] = ry_e[k] = -1;
                if constexpr (YL) {
                    ry_h[k] = d.cpml[1].row_h[at[k]];
                    ry_e[k] = d.cpml[1].row_e[at[k]];
                }
            }
        }
    }

    // the loads that follow the psi rows of the columns
    __device__ __forceinline__ void constants(const yee2d_desc& d)
    {
        if constexpr (YL) {
            const yee_cpml_axis& cy = d.cpml[1];
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                if (!in[k]) ry_e[k] = -1;
                if (stays[k]) ry_h[k] = -1;
                const int h = max(ry_h[k], 0), e = max(ry_e[k], 0);
                b_h[k] = cy.b_h[h];
                g_h[k] = cy.g_h[h];
                b_e[k] = cy.b_e[e];
                g_e[k] = cy.g_e[e];
            }
        }
    }

    // after constants(): 0 for the columns without a psi row
    __device__ __forceinline__ void finish()
    {
        if constexpr (YL) {
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                b_h[k] = ry_h[k] >= 0 ? b_h[k] : 0.f;
                g_h[k] = ry_h[k] >= 0 ? g_h[k] : 0.f;
                b_e[k] = ry_e[k] >= 0 ? b_e[k] : 0.f;
                g_e[k] = ry_e[k] >= 0 ? g_e[k] : 0.f;
                psi_h[k] = ry_h[k] >= 0 ? ~0u : 0u;
                psi_e[k] = ry_e[k] >= 0 ? ~0u : 0u;
                // not lane masks in scalar registers, which are full
                asm volatile("" : "+v"(psi_h[k]), "+v"(psi_e[k]));
            }
        }
        if constexpr (EDGE) {
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                moves[k] = stays[k] ? 0u : ~0u;
                asm volatile("" : "+v"(moves[k]));
            }
        }
    }

    // column of the grid of element k, -1 outside
    __device__ __forceinline__ int column(int k) const
    {
        if constexpr (EDGE) return in[k] ? (int)at[k] : -1;
        else return j + k;
    }

    __device__ __forceinline__ void read(const float* __restrict__ row, float out[VEC]) const
    {
        load_n<VEC>(row + at[0], out);
    }
};

// The material tables of one instance in LDS (whole block, no barrier here), with a zero entry after the last id (E_z).
// H_z: entries a (da, db, eps_xx, eps_yy) first, the face coefficients b of
// equal ids kMultiIds / 2 further, sigma_e beside them. Returns whether this thread saw a material that is not simple:
// simple ones are lossless and not PEC (ca = 1) and share da = 1 and the db of the first one, so a cell or face needs
// one coefficient, which the window keeps in a register, and a step reads no table.
template <int POL, int NW>
__device__ __forceinline__ bool stage_multi_tables(const yee2d_desc& d)
{
    const float4* a = reinterpret_cast<const float4*>(d.table);
    bool odd = false;
    for (int k = threadIdx.x; k <= d.n_materials; k += 64 * NW) {
        if (k == d.n_materials) {
            lds_coef[k] = make_float4(0.f, 0.f, 0.f, 0.f);
            break;
        }
        const float4 u = a[k], first = a[0];
        lds_coef[k] = u;
        if constexpr (POL == YEE_HZ) {
            const float4 v = *reinterpret_cast<const float4*>(d.table2 + 8 * k);
            lds_coef[kMultiIds / 2 + k] = v;
            lds_sigma[k] = d.table2[8 * k + 4];
            odd = odd || v.x != 1.f || v.z != 1.f || u.x != 1.f || u.y != first.y;
        } else {
            odd = odd || u.x != 1.f || u.z != 1.f || u.w != first.w;
        }
    }
    return odd;
}

// What a window loads first, before its form (FULL or not) and state set are known.
template <int VEC, int R, bool EDGE, bool YL>
struct WindowEarly {
    static constexpr int IDS = VEC == 1 ? VEC : VEC / 2;   // one to a register, or two
    LaneColumns<VEC, EDGE, YL> col;
    uint32_t ids[R + 1][IDS];    // ids of the rows (H_z: and of the one after them)
    float inv_h, inv_e;          // lane r: x constants of row r (windows with x layers)
    int row_h, row_e;

    __device__ __forceinline__ uint32_t id(int r, int k) const
    {
        if constexpr (IDS == VEC) return ids[r][k];
        else return k & 1 ? ids[r][k >> 1] >> 16 : ids[r][k >> 1] & 0xffffu;
    }
};

// A window of either polarisation: c is the field at the cell centres (E_z or H_z), fx the one on the hi-y faces (H_x or
// E_x) and fy the one on the hi-x faces (H_y or E_y). EDGE: the general form; XL, YL: rows, columns of it lie in an x, a y CPML
// layer; FULL: materials that are not simple (stage_multi_tables). Simple forms keep 1 * x in the updates: exact, and the
// rounding of each expression stays that of the general one.
template <int POL, int VEC, int R, int NW, bool EDGE, bool XL, bool YL, bool FULL, bool EXTRA, bool POLE>
struct MultiWindow {
    static constexpr bool HZ = POL == YEE_HZ;
    using Early = WindowEarly<VEC, R, EDGE, YL>;
    const yee2d_desc& d;
    const Window& w;
    LaneColumns<VEC, EDGE, YL> col;
    int wave, q0;            // this wavefront and its first row
    int par;
    int64_t n;               // step count before the launch
    uint32_t stays;          // bit r: fy of row q0 + r keeps its value: past a bounded axis' last row, or outside the grid
    int ph[XL ? R : 1], pe[XL ? R : 1];   // x psi rows, -1 for none
    float idx, idy, db;      // bulk inverse spacings; the one db of simple materials
    float c[R][VEC], fx[R][VEC], fy[R][VEC];
    uint32_t id[FULL ? R : 1];   // table offsets, two to a register
    // coefficients of the E updates: cb of the cells in cbx (simple E_z); of the E_x and E_y faces (H_z)
    float cax[FULL && HZ ? R : 1][VEC], cay[FULL && HZ ? R : 1][VEC];
    float cbx[HZ || !FULL ? R : 1][VEC], cby[HZ ? R : 1][VEC];
    float yh[YL ? R : 1][VEC], ye[YL ? R : 1][VEC], xh[XL ? R : 1][VEC], xe[XL ? R : 1][VEC];
    // Drude pole: current of the cells, the rows (bits) and elements (bits) inside its box
    float jp[POLE ? R : 1][VEC];
    uint32_t pole_rows, pole_cols;
    float damping;
    // Probes (EXTRA): lane p holds probe p as component << 16 | row of the wavefront << 8 | column of the window
    // (bits of probes_mine: those on owned cells of this wavefront), or the value of one outside the grid (probes_stray)
    uint64_t probes_mine, probes_stray;
    uint32_t probe;

    __device__ __forceinline__ MultiWindow(const yee2d_desc& desc, const Window& window) : d(desc), w(window) {}

    // row of the grid of row q (periodic wrap), -1 outside
    static __device__ __forceinline__ int fold_row(const yee2d_desc& d, int q)
    {
        if (!EDGE || (uint32_t)q < (uint32_t)d.nx) return q;
        if (!d.periodic_x) return -1;
        q %= d.nx;
        return q < 0 ? q + d.nx : q;
    }
    __device__ __forceinline__ int fold_row(int q) const { return fold_row(d, q); }

    // The first round of loads: column constants and psi rows, ids, x constants and psi rows.
    static __device__ __forceinline__ void early(const yee2d_desc& d, const Window& w, Early& out)
    {
        const int q0 = w.w0 + wave_index() * R;
        out.col.begin(d, w);
#pragma unroll
        for (int r = 0; r < R + 1; ++r) {
            if (r == R && !HZ) break;
            const uint16_t* row = d.material + (int64_t)max(0, fold_row(d, q0 + r)) * d.pitch;
            if constexpr (VEC == 1) {
#pragma unroll
                for (int k = 0; k < VEC; ++k) out.ids[r][k] = row[out.col.at[k]];
            } else {
                ldids<VEC>(row + out.col.at[0], out.ids[r]);
            }
        }
        if constexpr (XL) {
            const int q = q0 + min((int)(threadIdx.x & (YEE_WAVE - 1)), R - 1);
            const bool inside = (uint32_t)q < (uint32_t)d.nx;   // an axis with layers is not periodic
            const int f = inside ? q : 0;
            out.inv_h = d.inv_dx_h[f];
            out.inv_e = d.inv_dx_e[f];
            out.row_h = d.cpml[0].row_h[f];
            out.row_e = d.cpml[0].row_e[f];
            if (!inside) out.row_h = out.row_e = -1;
        }
    }

    static __device__ __forceinline__ float uniform(float v)
    {
        return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
    }

    // Fields and psi of the window; nothing here uses a loaded value, so all loads are in flight together.
    __device__ __forceinline__ void load()
    {
        const yee_cpml_axis& cx = d.cpml[0];
        const yee_cpml_axis& cy = d.cpml[1];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int f = max(0, fold_row(q0 + r));
            const int64_t base = (int64_t)f * d.pitch;
            col.read(d.field[par][0] + base, c[r]);
            col.read(d.field[par][1] + base, fx[r]);
            col.read(d.field[par][2] + base, fy[r]);
            if constexpr (YL) {
                const int64_t yrow = (int64_t)f * cy.n_rows;
#pragma unroll
                for (int k = 0; k < VEC; ++k) {
                    yh[r][k] = cy.psi_h[par][yrow + max(col.ry_h[k], 0)];
                    ye[r][k] = cy.psi_e[par][yrow + max(col.ry_e[k], 0)];
                }
            }
            if constexpr (XL) {
                if (ph[r] >= 0) col.read(cx.psi_h[par] + (int64_t)ph[r] * d.pitch, xh[r]);
                if (pe[r] >= 0) col.read(cx.psi_e[par] + (int64_t)pe[r] * d.pitch, xe[r]);
            }
        }
    }

    // The loaded window as the steps take it: zeros outside the grid and where there is no psi, ids as table offsets or
    // the coefficients they stand for.
    __device__ __forceinline__ void finish(const Early& early)
    {
        col.finish();
        uint32_t ids[R + 1][VEC];
#pragma unroll
        for (int r = 0; r < R + 1; ++r) {
            if (r == R && !HZ) break;
#pragma unroll
            for (int k = 0; k < VEC; ++k) ids[r][k] = early.id(r, k);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            bool inside = true;
            if constexpr (EDGE) {
                inside = fold_row(q0 + r) >= 0;
#pragma unroll
                for (int k = 0; k < VEC; ++k) {
                    const bool cell = inside && col.in[k];
                    c[r][k] = cell ? c[r][k] : 0.f;
                    fx[r][k] = cell ? fx[r][k] : 0.f;
                    fy[r][k] = cell ? fy[r][k] : 0.f;
                    if constexpr (!HZ) ids[r][k] = cell ? ids[r][k] : (uint32_t)d.n_materials;   // the zero entry
                    if constexpr (YL) {
                        yh[r][k] = cell && col.ry_h[k] >= 0 ? yh[r][k] : 0.f;
                        ye[r][k] = cell && col.ry_e[k] >= 0 ? ye[r][k] : 0.f;
                    }
                    if constexpr (XL) {
                        xh[r][k] = cell && ph[r] >= 0 ? xh[r][k] : 0.f;
                        xe[r][k] = cell && pe[r] >= 0 ? xe[r][k] : 0.f;
                    }
                }
            }
            if constexpr (HZ) {
                const int id_next = __builtin_amdgcn_update_dpp(0, (int)ids[r][0], 0x130, 0xf, 0xf, true);
#pragma unroll
                for (int k = 0; k < VEC; ++k) {
                    const bool cell = !EDGE || (inside && col.in[k]);
                    const uint32_t right = k < VEC - 1 ? ids[r][k < VEC - 1 ? k + 1 : k] : (uint32_t)id_next;
                    float ca, cb;
                    face(ids[r][k], right, 0, &ca, &cb);
                    // faces outside the grid and past a bounded axis' last column keep their value
                    const bool x_free = cell && !(EDGE && col.last[k]);
                    cbx[r][k] = x_free ? cb : 0.f;
                    if constexpr (FULL) cax[r][k] = x_free ? ca : 1.f;
                    face(ids[r][k], ids[r + 1][k], 1, &ca, &cb);
                    const bool y_free = cell && !((stays >> r) & 1);
                    cby[r][k] = y_free ? cb : 0.f;
                    if constexpr (FULL) cay[r][k] = y_free ? ca : 1.f;
                }
            }
            if constexpr (!HZ && !FULL) {
#pragma unroll
                for (int k = 0; k < VEC; ++k) cbx[r][k] = lds_coef[ids[r][k]].y;
            }
            if constexpr (FULL) {
                id[r] = ids[r][0] << 4;
                if constexpr (VEC == 2) id[r] |= ids[r][1] << 20;
            }
        }
    }

    // (ca, cb) of the E face between cells of ids a and b (comp 0: E_x, 1: E_y)
    __device__ __forceinline__ void face(uint32_t a, uint32_t b, int comp, float* ca, float* cb) const
    {
        if (a == b) {
            const float4 s = lds_coef[kMultiIds / 2 + a];
            *ca = comp == 0 ? s.x : s.z;
            *cb = comp == 0 ? s.y : s.w;
            return;
        }
        const float4 va = lds_coef[a], vb = lds_coef[b];
        mixed_face(comp == 0 ? va.z : va.w, comp == 0 ? vb.z : vb.w, lds_sigma[a], lds_sigma[b], d.dt_over_eps0, ca, cb);
    }

    __device__ __forceinline__ float4 coef(int r, int k) const
    {
        return coef_at(k ? id[r] >> 16 : (VEC == 2 ? id[r] & 0xffffu : id[r]));
    }

    // element k's neighbours along y in a row: the next column, the previous one
    static __device__ __forceinline__ float right(const float v[VEC], int k, float next)
    {
        return k < VEC - 1 ? v[k < VEC - 1 ? k + 1 : k] : next;
    }
    static __device__ __forceinline__ float left(const float v[VEC], int k, float prev)
    {
        return k == 0 ? prev : v[k > 0 ? k - 1 : 0];
    }

    // The drive of a cell (read and written by its own lane only).
    static __device__ __forceinline__ float& drive(int r, int k)
    {
        return lds_drive[(r * 64 * NW + threadIdx.x) * VEC + k];
    }

    // Current and drive of the cells inside the pole's box; launch `launch` of a call reads state[launch & 1].
    __device__ __forceinline__ void load_pole(int launch)
    {
        pole_rows = pole_cols = 0;
        const yee_pole& p = d.pole[0];
        damping = uniform(p.damping);
        const float* __restrict__ state = p.state[launch & 1];
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            const int at = col.column(k);
            pole_cols |= (uint32_t)(at >= p.j0 && at < p.j1) << k;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int f = fold_row(q0 + r);
#pragma unroll
            for (int k = 0; k < VEC; ++k) jp[r][k] = drive(r, k) = 0.f;
            if (f < p.i0 || f >= p.i1) continue;
            pole_rows |= 1u << r;
            const int64_t base = (int64_t)(f - p.i0) * (p.j1 - p.j0) - p.j0;
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                if (!((pole_cols >> k) & 1)) continue;
                jp[r][k] = state[base + col.column(k)];
                drive(r, k) = p.drive[base + col.column(k)];
            }
        }
    }

    __device__ __forceinline__ void store_pole(int launch) const
    {
        if (!col.owner) return;
        const yee_pole& p = d.pole[0];
        float* __restrict__ state = p.state[(launch & 1) ^ 1];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int q = q0 + r;
            if (!((pole_rows >> r) & 1) || q < w.i0 || q >= w.i1) continue;
            const int64_t base = (int64_t)(q - p.i0) * (p.j1 - p.j0) - p.j0;
#pragma unroll
            for (int k = 0; k < VEC; ++k)
                if ((pole_cols >> k) & 1) state[base + col.column(k)] = jp[r][k];
        }
    }

    // (ca, cb, da, db) of an E_z cell
    __device__ __forceinline__ float4 ez_coef(int r, int k) const
    {
        if constexpr (FULL) return coef(r, k);
        else return make_float4(1.f, cbx[HZ ? 0 : r][k], 1.f, db);
    }

    // E_z: H of row r from E of the row above it
    __device__ __forceinline__ void ez_h_row(int r, const float above[VEC])
    {
        const float4 x = XL ? lds_row[2 * (wave * R + r)] : float4{};
        const float next = lane_next(c[r][0]);
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            const float4 m = ez_coef(r, k);
            const float de_x = above[k] - c[r][k];
            const float de_y = right(c[r], k, next) - c[r][k];
            float unused;
            if constexpr (EDGE) {
                float v = ez_hy(m, fy[r][k], de_x, XL ? x.x : idx, false, 0.f, 0.f, 0.f, &unused);
                if constexpr (XL) {
                    xh[r][k] = x.y * xh[r][k] + x.z * keep_bits(x.w, de_x);
                    v += m.w * xh[r][k];
                }
                fy[r][k] = (stays >> r) & 1 ? fy[r][k] : v;
                float u = ez_hx(m, fx[r][k], de_y, col.inv_h[k], false, 0.f, 0.f, 0.f, &unused);
                if constexpr (YL) {
                    yh[r][k] = col.b_h[k] * yh[r][k] + col.g_h[k] * keep_bits(col.psi_h[k], de_y);
                    u -= m.w * yh[r][k];
                }
                fx[r][k] = pick_bits(col.moves[k], u, fx[r][k]);
            } else {
                fy[r][k] = ez_hy(m, fy[r][k], de_x, idx, false, 0.f, 0.f, 0.f, &unused);
                fx[r][k] = ez_hx(m, fx[r][k], de_y, idy, false, 0.f, 0.f, 0.f, &unused);
            }
        }
    }

    // E_z: E of row r from H_y of the row below it
    __device__ __forceinline__ void ez_e_row(int r, const float below[VEC])
    {
        const float4 x = XL ? lds_row[2 * (wave * R + r) + 1] : float4{};
        const float ie = XL ? x.x : idx;
        const float prev = lane_prev(fx[r][VEC - 1]);
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            const float4 m = ez_coef(r, k);
            const float dhy = fy[r][k] - below[k];
            const float dhx = fx[r][k] - left(fx[r], k, prev);
            float v = ez_centre(m, c[r][k], dhy, dhx, ie, EDGE ? col.inv_e[k] : idy);
            if constexpr (XL) {
                xe[r][k] = x.y * xe[r][k] + x.z * keep_bits(x.w, dhy);
                v += m.y * xe[r][k];
            }
            if constexpr (YL) {
                ye[r][k] = col.b_e[k] * ye[r][k] + col.g_e[k] * keep_bits(col.psi_e[k], dhx);
                v -= m.y * ye[r][k];
            }
            if constexpr (POLE) {
                // cells outside the box have no current and no drive: their E passes unread (it may be infinite)
                const float e_n = (pole_rows >> r) & 1 && (pole_cols >> k) & 1 ? c[r][k] : 0.f;
                float jc = jp[r][k];
                jc += damping * jc + drive(r, k) * e_n;
                jp[r][k] = jc;
                v -= m.y * jc;
            }
            c[r][k] = v;
        }
    }

    // H_z: H of row r from E_y of the row below it
    __device__ __forceinline__ void hz_h_row(int r, const float below[VEC])
    {
        const float4 x = XL ? lds_row[2 * (wave * R + r) + 1] : float4{};
        const float ie = XL ? x.x : idx;
        const float prev = lane_prev(fx[r][VEC - 1]);
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            float4 m = make_float4(1.f, db, 0.f, 0.f);
            if constexpr (FULL) m = coef(r, k);   // (da, db, eps_xx, eps_yy)
            const float dex = fx[r][k] - left(fx[r], k, prev);
            const float dey = fy[r][k] - below[k];
            float no_x, no_y;
            c[r][k] = hz_centre(m, c[r][k], dex, dey, EDGE ? col.inv_e[k] : idy, ie, false, 0.f, 0.f, 0.f, &no_x, false,
                                0.f, 0.f, 0.f, &no_y);
            if constexpr (XL) {
                xe[r][k] = x.y * xe[r][k] + x.z * keep_bits(x.w, dey);
                c[r][k] -= m.y * xe[r][k];
            }
            if constexpr (YL) {
                ye[r][k] = col.b_e[k] * ye[r][k] + col.g_e[k] * keep_bits(col.psi_e[k], dex);
                c[r][k] += m.y * ye[r][k];
            }
        }
    }

    // H_z: E_x of row r
    __device__ __forceinline__ void hz_ex_row(int r)
    {
        const float next = lane_next(c[r][0]);
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            // faces that keep their value have cb = 0, which an infinite difference would not survive
            float dh = right(c[r], k, next) - c[r][k];
            if constexpr (EDGE) dh = keep_bits(col.moves[k], dh);
            fx[r][k] = hz_ex(FULL ? cax[FULL ? r : 0][k] : 1.f, cbx[r][k], fx[r][k], dh, EDGE ? col.inv_h[k] : idy);
            if constexpr (YL) {
                yh[r][k] = col.b_h[k] * yh[r][k] + col.g_h[k] * keep_bits(col.psi_h[k], dh);
                fx[r][k] += cbx[r][k] * yh[r][k];
            }
        }
    }

    // H_z: E_y of row r from H_z of the row above it
    __device__ __forceinline__ void hz_ey_row(int r, const float above[VEC])
    {
        const float4 x = XL ? lds_row[2 * (wave * R + r)] : float4{};
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            float dh = above[k] - c[r][k];
            if constexpr (EDGE) dh = keep_bits(((stays >> r) & 1) - 1u, dh);
            fy[r][k] = hz_ey(FULL ? cay[FULL ? r : 0][k] : 1.f, cby[r][k], fy[r][k], dh, XL ? x.x : idx);
            if constexpr (XL) {
                xh[r][k] = x.y * xh[r][k] + x.z * keep_bits(x.w, dh);
                fy[r][k] -= cby[r][k] * xh[r][k];
            }
        }
    }

    // The rows of this wavefront (bits) that source `s` acts on: its line, or the rows of its span.
    __device__ __forceinline__ uint32_t source_rows(int s) const
    {
        const yee_line_source& src = d.source[s];
        const bool line = src.axis == 1;
        const int lo = line ? src.line : src.lo, hi = line ? src.line + 1 : src.hi;
        uint32_t rows = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int f = fold_row(q0 + r);
            rows |= (uint32_t)(f >= lo && f < hi) << r;
        }
        return rows;
    }

    // The values of the launch's steps and the profile along the window (whole block; before the first barrier of the
    // steps): a step then reads LDS instead of a chain of global loads.
    __device__ __forceinline__ void stage_sources(uint32_t sources, int steps) const
    {
        for (uint32_t left = sources; left; left &= left - 1) {
            const int s = __builtin_ctz(left);
            const yee_line_source& src = d.source[s];
            const bool line = src.axis == 1;
            const int t = threadIdx.x;
            if (t < steps) lds_wave[s * kMultiMax + t] = wave_value(src, n + t);
            if (t < (line ? 64 * VEC : w.rows)) {
                const int n_axis = line ? d.ny : d.nx;
                int f = (line ? w.k0 : w.w0) + t;
                if (EDGE && (line ? d.periodic_y : d.periodic_x)) {
                    f %= n_axis;
                    f = f < 0 ? f + n_axis : f;
                }
                lds_profile[s * 128 + t] = f >= src.lo && f < src.hi ? src.profile[f - src.lo] : 0.f;
            }
        }
    }

    // Source `s` on step `step` of the launch after the update of its field: field += float32(value * profile) in `rows`.
    // Lines along y act on c (E_z, H currents) or E_y, lines along x on c or E_x.
    // (One field a call: a run-time choice between register arrays would move them to scratch memory.)
    __device__ __forceinline__ void add_line(float (&field)[R][VEC], int s, uint32_t rows, int step) const
    {
        const int lane = threadIdx.x & (YEE_WAVE - 1);
        const int lo = d.source[s].lo, hi = d.source[s].hi;
        const float v = lds_wave[s * kMultiMax + step];
        float add[VEC];
        bool in[VEC];   // within the span: past it an infinite value times the profile's 0 would be NaN
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            add[k] = __fmul_rn(v, lds_profile[s * 128 + VEC * lane + k]);
            in[k] = col.column(k) >= lo && col.column(k) < hi;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (!((rows >> r) & 1)) continue;
#pragma unroll
            for (int k = 0; k < VEC; ++k) field[r][k] = in[k] ? field[r][k] + add[k] : field[r][k];
        }
    }
    __device__ __forceinline__ void add_column(float (&field)[R][VEC], int s, uint32_t rows, int step) const
    {
        const int column = d.source[s].line;
        const float v = lds_wave[s * kMultiMax + step];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (!((rows >> r) & 1)) continue;
            const float add = __fmul_rn(v, lds_profile[s * 128 + wave * R + r]);
            // the two columns apart, in code that cannot be merged: merged, the choice between them becomes an indexed
            // access and the field moves to scratch memory
            if (col.column(0) == column) {
                field[r][0] += add;
                asm volatile("; column 0" : "+v"(field[r][0]));
            }
            if constexpr (VEC > 1) {
                if (col.column(1) == column) {
                    field[r][1] += add;
                    asm volatile("; column 1" : "+v"(field[r][1]));
                }
            }
        }
    }
    __device__ __forceinline__ void add_source(int s, uint32_t rows, int step)
    {
        const yee_line_source& src = d.source[s];
        if (src.axis == 1) {
            if (HZ && src.field == YEE_SOURCE_E) add_line(fy, s, rows, step);
            else add_line(c, s, rows, step);
        } else {
            if (HZ && src.field == YEE_SOURCE_E) add_column(fx, s, rows, step);
            else add_column(c, s, rows, step);
        }
    }

    __device__ __forceinline__ void add_sources(uint32_t mine, int kind, int step)
    {
        for (uint32_t left = mine; left; left &= left - 1) {
            const int s = __builtin_ctz(left);
            if (d.source[s].field == kind) add_source(s, source_rows(s), step);
        }
    }

    // flux-line samples of the owned rows after `done` steps: (E_z, H_y or H_x), (E_y or E_x, H_z)
    __device__ __forceinline__ void sample(uint32_t monitors, int64_t done) const
    {
        const int64_t index = done / d.sample_interval - 1;
        for (uint32_t left = monitors; left; left &= left - 1) {
            const yee_flux_line& mon = d.monitor[__builtin_ctz(left)];
            const bool line = mon.normal == 0;
            const int lo = max(max(line ? mon.position : mon.lo, w.i0), q0);
            const int hi = min(min(line ? mon.position + 1 : mon.hi, w.i1), q0 + R);
            for (int q = lo; q < hi; ++q) {
                float vc[VEC], vf[VEC];
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (q == q0 + r) {
#pragma unroll
                        for (int k = 0; k < VEC; ++k) {
                            vc[k] = c[r][k];
                            vf[k] = line ? fy[r][k] : fx[r][k];
                        }
                    }
#pragma unroll
                for (int k = 0; k < VEC; ++k) {
                    const int at = col.column(k);
                    if (col.owner && (line ? at >= mon.lo && at < mon.hi : at == mon.position))
                        dft_accumulate(mon, index, line ? at - mon.lo : q - mon.lo, HZ ? vf[k] : vc[k],
                                       HZ ? vc[k] : vf[k]);
                }
            }
        }
    }

    // Row q0 + r (r uniform) of field `component`: selects, because an indexed access, or a choice between the arrays,
    // would move the fields to scratch memory.
    __device__ __forceinline__ void pick(int component, int r, float out[VEC]) const
    {
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            float a = c[0][k], b = fx[0][k], e = fy[0][k];
#pragma unroll
            for (int q = 1; q < R; ++q) {
                a = q == r ? c[q][k] : a;
                b = q == r ? fx[q][k] : b;
                e = q == r ? fy[q][k] : e;
            }
            out[k] = component == 0 ? a : component == 1 ? b : e;
        }
    }

    // DFT regions' samples of the owned cells after `done` steps. A mean with the lower neighbour along x needs the row
    // that the wavefront below holds: every wavefront of the block takes part in that exchange.
    __device__ __forceinline__ void sample_regions(uint32_t regions, int64_t done, float* down, const float* from_below)
    {
        const int64_t index = done / d.sample_interval - 1;
        float row[VEC];
#pragma unroll
        for (int k = 0; k < VEC; ++k) down[k] = fy[R - 1][k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < VEC; ++k) row[k] = from_below[k];
        __syncthreads();
        for (uint32_t rest = regions; rest; rest &= rest - 1) {
            const yee_dft_region& g = d.dft[__builtin_ctz(rest)];
            if (index >= g.n_samples) continue;
            const int64_t cells = (int64_t)g.count[0] * g.count[1];
            const int step = g.stride[0];
            const int first = max(max(w.i0, q0), g.start[0]);
            const int end = min(min(w.i1, q0 + R), g.start[0] + step * (g.count[0] - 1) + 1);
            int64_t along[VEC];   // sampled column of element k, -1 for none
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                const int at = col.column(k), from = at - g.start[1];
                const bool hit = col.owner && at < d.ny && from >= 0 && from % g.stride[1] == 0 &&
                                 from / g.stride[1] < g.count[1];
                along[k] = hit ? from / g.stride[1] : -1;
            }
            int t0 = (first - g.start[0] + step - 1) / step;
            for (int q = g.start[0] + t0 * step; q < end; q += step, ++t0) {
                const int r = q - q0;
                for (int s = 0; s < g.n_comp; ++s) {
                    float v[VEC], low[VEC];
                    pick(g.comp[s], r, v);
                    const bool self = !g.pair_wrap[s];   // the lower neighbour of index 0 is the cell itself
                    const float prev = lane_prev(v[VEC - 1]);
                    if (g.pair_axis[s] == 0) {
                        pick(2, r - 1, low);
#pragma unroll
                        for (int k = 0; k < VEC; ++k) {
                            low[k] = r == 0 ? row[k] : low[k];
                            low[k] = q == 0 && self ? v[k] : low[k];
                        }
                    } else {
#pragma unroll
                        for (int k = 0; k < VEC; ++k) low[k] = col.column(k) == 0 && self ? v[k] : left(v, k, prev);
                    }
#pragma unroll
                    for (int k = 0; k < VEC; ++k) {
                        if (along[k] < 0) continue;
                        const float x = g.pair_axis[s] >= 0 ? 0.5f * (v[k] + low[k]) : v[k];
                        dft_region_add(g, s, cells, (int64_t)t0 * g.count[1] + along[k], index, x);
                    }
                }
            }
        }
    }

    // The probes of this wavefront, at most 64 (the host's rule); the window of cell (0, 0) takes those outside the grid.
    __device__ __forceinline__ void find_probes()
    {
        probes_mine = probes_stray = 0;
        probe = 0;
        if (d.probes.n_probes == 0) return;
        const int p = threadIdx.x & (YEE_WAVE - 1);
        bool mine = false, stray = false;
        if (p < d.probes.n_probes) {
            const int64_t cell = d.probes.cell[p];
            const int32_t component = d.probes.component[p];
            const bool known = component >= 0 && component < 3 && cell >= 0 && cell < (int64_t)d.nx * d.pitch;
            const int32_t i = known ? (int32_t)(cell / d.pitch) : 0;
            const int32_t j = known ? (int32_t)(cell - (int64_t)i * d.pitch) : 0;
            stray = !known || j >= d.ny;   // past the grid: NaN; a padding column: what it holds (0)
            mine = !stray && i >= max(q0, w.i0) && i < min(q0 + R, w.i1) && j >= w.c0 && j < w.c1;
            stray = stray && wave == 0 && w.i0 == 0 && w.c0 == 0;
            if (mine) probe = (uint32_t)component << 16 | (uint32_t)(i - q0) << 8 | (uint32_t)(j - w.k0);
            if (stray) probe = __float_as_uint(known ? d.field[par][component][cell] : __builtin_nanf(""));
        }
        probes_mine = __ballot(mine);
        probes_stray = __ballot(stray);
    }

    // Probe samples of step `step` (row `step` of the table).
    __device__ __forceinline__ void sample_probes(int64_t step) const
    {
        if (step >= d.probes.capacity) return;
        float* const row = d.probes.samples + step * d.probes.n_probes;
        const int lane = threadIdx.x & (YEE_WAVE - 1);
        if ((probes_stray >> lane) & 1) row[lane] = __uint_as_float(probe);
        for (uint64_t left = probes_mine; left; left &= left - 1) {
            const int p = __builtin_ctzll(left);
            const uint32_t word = __builtin_amdgcn_readlane(probe, p);
            const int component = word >> 16, r = (word >> 8) & 0xff, column = word & 0xff;
            float v[VEC];
            pick(component, r, v);
            if (lane == column / VEC) row[p] = VEC > 1 && column % VEC ? v[VEC - 1] : v[0];
        }
    }

    __device__ __forceinline__ void store()
    {
        if (!col.owner) return;
        const yee_cpml_axis& cx = d.cpml[0];
        const yee_cpml_axis& cy = d.cpml[1];
        const int out = par ^ 1;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int q = q0 + r;
            if (q < w.i0 || q >= w.i1) continue;
            const int64_t base = (int64_t)q * d.pitch + col.j;
            store_n<VEC>(d.field[out][0] + base, c[r]);
            store_n<VEC>(d.field[out][1] + base, fx[r]);
            store_n<VEC>(d.field[out][2] + base, fy[r]);
            if constexpr (YL) {
                const int64_t yrow = (int64_t)q * cy.n_rows;
#pragma unroll
                for (int k = 0; k < VEC; ++k) {
                    if (col.ry_h[k] >= 0 && !col.last[k]) cy.psi_h[out][yrow + col.ry_h[k]] = yh[r][k];
                    if (col.ry_e[k] >= 0) cy.psi_e[out][yrow + col.ry_e[k]] = ye[r][k];
                }
            }
            if constexpr (XL) {
                if (ph[r] >= 0 && q < d.nx - 1) store_n<VEC>(cx.psi_h[out] + (int64_t)ph[r] * d.pitch + col.j, xh[r]);
                if (pe[r] >= 0) store_n<VEC>(cx.psi_e[out] + (int64_t)pe[r] * d.pitch + col.j, xe[r]);
            }
        }
    }

    // Two half steps; the row each needs from the neighbouring wavefront goes through LDS, and the rows that do not need
    // it are computed before the barrier. (up is written before the first barrier and read after it, down before and
    // after the second, so one buffer of each is enough: the other barrier lies between a read and the next write.)
    __device__ __forceinline__ void ez_step(float* up, float* down, const float* from_above, const float* from_below)
    {
        float row[VEC];
#pragma unroll
        for (int k = 0; k < VEC; ++k) up[k] = c[0][k];
#pragma unroll
        for (int r = 0; r < R - 1; ++r) ez_h_row(r, c[r + 1]);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < VEC; ++k) row[k] = from_above[k];
        ez_h_row(R - 1, row);
#pragma unroll
        for (int k = 0; k < VEC; ++k) down[k] = fy[R - 1][k];
#pragma unroll
        for (int r = R - 1; r > 0; --r) ez_e_row(r, fy[r - 1]);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < VEC; ++k) row[k] = from_below[k];
        ez_e_row(0, row);
    }

    __device__ __forceinline__ void hz_step(float* up, float* down, const float* from_above, const float* from_below,
                                            uint32_t mine, int step)
    {
        float row[VEC];
#pragma unroll
        for (int k = 0; k < VEC; ++k) down[k] = fy[R - 1][k];
#pragma unroll
        for (int r = R - 1; r > 0; --r) hz_h_row(r, fy[r - 1]);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < VEC; ++k) row[k] = from_below[k];
        hz_h_row(0, row);
        if (mine) add_sources(mine, YEE_SOURCE_H, step);
#pragma unroll
        for (int k = 0; k < VEC; ++k) up[k] = c[0][k];
#pragma unroll
        for (int r = 0; r < R; ++r) hz_ex_row(r);
#pragma unroll
        for (int r = 0; r < R - 1; ++r) hz_ey_row(r, c[r + 1]);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < VEC; ++k) row[k] = from_above[k];
        hz_ey_row(R - 1, row);
    }

    // The second round of loads, behind the first one's results (Early): constants by psi row, fields and psi.
    __device__ __forceinline__ void begin(const Early& early, int64_t n_start, int set, int launch)
    {
        n = n_start;
        par = set;
        wave = wave_index();
        q0 = w.w0 + wave * R;
        stays = 0;
        if (EDGE && !d.periodic_x) {
#pragma unroll
            for (int r = 0; r < R; ++r) stays |= (uint32_t)(q0 + r < 0 || q0 + r >= d.nx - 1) << r;
        }
        idx = uniform(d.inv_dx_bulk);
        idy = uniform(d.inv_dy_bulk);
        col = early.col;
        col.constants(d);
        if constexpr (XL) {
            // lane r holds the constants of row r; every lane takes part, so that the loads are plain
            const yee_cpml_axis& cx = d.cpml[0];
            const int lane = threadIdx.x & (YEE_WAVE - 1);
            const int h = max(early.row_h, 0), e = max(early.row_e, 0);
            const float4 a = make_float4(early.inv_h, cx.b_h[h], cx.g_h[h], 0.f);
            const float4 b = make_float4(early.inv_e, cx.b_e[e], cx.g_e[e], 0.f);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                ph[r] = __builtin_amdgcn_readlane(early.row_h, r);
                pe[r] = __builtin_amdgcn_readlane(early.row_e, r);
            }
            load();
            if (lane < R) {
                const bool layer_h = early.row_h >= 0, layer_e = early.row_e >= 0;
                lds_row[2 * (wave * R + lane)] = make_float4(a.x, layer_h ? a.y : 0.f, layer_h ? a.z : 0.f,
                                                             __uint_as_float(layer_h ? ~0u : 0u));
                lds_row[2 * (wave * R + lane) + 1] = make_float4(b.x, layer_e ? b.y : 0.f, layer_e ? b.z : 0.f,
                                                                 __uint_as_float(layer_e ? ~0u : 0u));
            }
        } else {
            load();
        }
        if constexpr (EXTRA) find_probes();
        if constexpr (POLE) load_pole(launch);
    }

    __device__ __forceinline__ void run(int steps, const Early& early, const WindowRecords& records, int launch)
    {
        if (records.sources) stage_sources(records.sources, steps);
        finish(early);
        if constexpr (!FULL) db = uniform(HZ ? lds_coef[0].y : lds_coef[0].w);
        uint32_t mine = 0;   // sources on rows of this wavefront
        for (uint32_t left = records.sources; left; left &= left - 1)
            if (source_rows(__builtin_ctz(left))) mine |= left & -left;
        const int lane = threadIdx.x & (YEE_WAVE - 1);
        float* const up = lds_up + wave * 128 + VEC * lane;
        float* const down = lds_down + wave * 128 + VEC * lane;
        const float* const from_above = lds_up + (wave + 1 < NW ? wave + 1 : wave) * 128 + VEC * lane;
        const float* const from_below = lds_down + (wave > 0 ? wave - 1 : 0) * 128 + VEC * lane;
        int left = records.monitors | records.regions ? d.sample_interval - (int)(n % d.sample_interval) : 0;   // steps to the next sample
        for (int s = 0; s < steps; ++s) {
            if constexpr (HZ) hz_step(up, down, from_above, from_below, mine, s);
            else ez_step(up, down, from_above, from_below);
            if (mine) add_sources(mine, YEE_SOURCE_E, s);
            if ((records.monitors | records.regions) && --left == 0) {
                sample(records.monitors, n + s + 1);
                if constexpr (EXTRA)
                    if (records.regions) sample_regions(records.regions, n + s + 1, down, from_below);
                left = d.sample_interval;
            }
            if constexpr (EXTRA)
                if (probes_mine | probes_stray) sample_probes(n + s);
        }
        store();
        if constexpr (POLE) store_pole(launch);
    }
};

// One window of `steps` steps: a first round of loads with the tables among them, the choice of the form, a second round
// behind the first one's results, the steps and the stores. The two rounds are what a launch waits for before it steps.
template <int POL, int VEC, int R, int NW, bool EDGE, bool XL, bool YL, bool EXTRA>
__device__ __forceinline__ void run_window(const yee2d_desc& d, const Window& w, int64_t clock, int32_t offset,
                                           int32_t launch, int steps)
{
    WindowRecords records = window_records(d, w, 64 * VEC);
    if constexpr (EXTRA) records.regions = window_regions(d, w);
    WindowEarly<VEC, R, EDGE, YL> early;
    MultiWindow<POL, VEC, R, NW, EDGE, XL, YL, false, EXTRA, false>::early(d, w, early);
    const bool odd = stage_multi_tables<POL, NW>(d);
    clock = (int64_t)__builtin_amdgcn_readfirstlane((int)(clock >> 32)) << 32 |
            (uint32_t)__builtin_amdgcn_readfirstlane((int)clock);
    const int64_t n = clock + offset;
    const int set = (int)((clock + launch) & 1);
    const bool full = __syncthreads_or(odd);
    const auto run = [&](auto& window) {
        window.begin(early, n, set, launch);
        window.run(steps, early, records, launch);
    };
    if constexpr (EXTRA && POL == YEE_EZ) {
        if (window_pole(d, w, 64 * VEC)) {
            if (full) {
                MultiWindow<POL, VEC, R, NW, EDGE, XL, YL, true, true, true> window(d, w);
                run(window);
            } else {
                MultiWindow<POL, VEC, R, NW, EDGE, XL, YL, false, true, true> window(d, w);
                run(window);
            }
            return;
        }
    }
    if (full) {
        MultiWindow<POL, VEC, R, NW, EDGE, XL, YL, true, EXTRA, false> window(d, w);
        run(window);
    } else {
        MultiWindow<POL, VEC, R, NW, EDGE, XL, YL, false, EXTRA, false> window(d, w);
        run(window);
    }
}

// Window `block` of one instance, in the form its place asks for: `steps` steps (at most plan.steps, which the windows'
// halo is laid out for).
template <int POL, int VEC, int R, int TV, int TR, int NW, bool EXTRA>
__device__ __forceinline__ void multi_block(const yee2d_desc& d, const yee2d_multi_plan& plan, int block, int64_t clock,
                                            int32_t offset, int32_t launch, int steps)
{
    const int t = plan.steps;
    int region = 0;
    for (int k = 1; k < plan.n_regions; ++k)
        if (block >= plan.region[k].first) region = k;
    const yee2d_multi_region& g = plan.region[region];
    const int index = block - g.first;
    const int ti = __builtin_amdgcn_readfirstlane(index / g.tiles_j), tj = index - ti * g.tiles_j;
    const bool tall = TR > 0 && plan.interior && region == 0;
    const int columns = 64 * (tall ? TV : VEC);
    Window w;
    w.rows = NW * (tall ? TR : R);
    w.i0 = g.i0 + ti * g.rows;
    w.i1 = min(g.i1, w.i0 + g.rows);
    w.c0 = g.j0 + tj * g.columns;
    w.c1 = min(g.j1, w.c0 + g.columns);
    w.w0 = w.i0 - t;
    w.k0 = w.c0 - yee2d_multi_halo(t, tall ? TV : VEC);
    if constexpr (TR > 0) {
        if (tall) {
            run_window<POL, TV, TR, NW, false, false, false, EXTRA>(d, w, clock, offset, launch, steps);
            return;
        }
    }
    // layers of an axis without psi rows have none to step
    const bool x_layers = d.cpml[0].n_rows > 0 && (w.w0 < d.layer_x_lo || w.w0 + w.rows > d.layer_x_hi);
    const bool y_layers = d.cpml[1].n_rows > 0 && (w.k0 < d.layer_y_lo || w.k0 + columns > d.layer_y_hi);
    const bool lean = w.w0 >= 0 && w.w0 >= d.layer_x_lo && w.w0 + w.rows < d.nx && w.w0 + w.rows <= d.layer_x_hi &&
                      w.k0 >= 0 && w.k0 >= d.layer_y_lo && w.k0 + columns < d.ny && w.k0 + columns <= d.layer_y_hi;
    if (lean)
        run_window<POL, VEC, R, NW, false, false, false, EXTRA>(d, w, clock, offset, launch, steps);
    else if (x_layers && y_layers)
        run_window<POL, VEC, R, NW, true, true, true, EXTRA>(d, w, clock, offset, launch, steps);
    else if (x_layers)
        run_window<POL, VEC, R, NW, true, true, false, EXTRA>(d, w, clock, offset, launch, steps);
    else if (y_layers)
        run_window<POL, VEC, R, NW, true, false, true, EXTRA>(d, w, clock, offset, launch, steps);
    else
        run_window<POL, VEC, R, NW, true, false, false, EXTRA>(d, w, clock, offset, launch, steps);
}

}  // namespace yee
