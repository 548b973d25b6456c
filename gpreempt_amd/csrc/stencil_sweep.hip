// A direction sweep of miniWeather in one launch.
//
// Kernel by kernel a sweep reads and writes the 82 MB state (3200 x 1600 cells) eight times per Runge-Kutta stage and
// is bound by that: 280 us per sweep.  But a sweep couples cells along its own direction only, and a stage reaches two
// cells to either side.  So a wavefront takes a stretch of 64 * CELLS consecutive cells along the sweep, six of them at
// either end belonging to its neighbours, and carries them through the three stages in registers: lane l holds cells
// CELLS * l .. CELLS * l + CELLS - 1, the cells and fluxes of the next lanes come by DPP wave shifts, and the state is
// read and written once.  What bounds it now is the arithmetic: 125 vector instructions per cell and stage, for an
// eighth more cells than there are.  82 us per preemptible sweep, 100 (x) and 88 (z) for the two that also leave state_tmp
// and the fluxes (86, 109 and 93 before products and sums were fused and the viscosity's division went to the host); two cells per
// lane, since four take 140-200 registers (x 100-130 us, z 154-175).  More wavefronts by fewer registers (five to a SIMD for
// four): spills, 8260 -> 8570 us for twenty steps and their output; a workgroup per claim for the x sweeps' 11200 tiles: level.
//
// x: rows are contiguous, a wavefront loads and stores its stretch itself.  z: a workgroup brings 16 columns of a
// stretch in through LDS (64-byte runs of every row; a column is contiguous there), and its wavefronts take a column
// at a time.
#include "launch_tiles.hpp"
#include "stencil_bodies.hpp"

namespace gp {

constexpr int SW_HALO = 6;  // three stages of two cells

// the sweep's parameters, and what a stage takes from its length and the cell's: divisions made once on the host
struct SweepArgs : gp_mw_sweep_params {
    float hv_coef[3];  // -MW_HV_BETA * d / (16 * dt[stage])
};

// the value of the lane below / above (lane 0 / 63: 0; those cells are the neighbours' anyway)
__device__ __forceinline__ float from_below(float x) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x138, 0xf, 0xf, true)); }
__device__ __forceinline__ float from_above(float x) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x130, 0xf, 0xf, true)); }

// The fluxes through the lower faces of a lane's cells, and through the upper face of its last one (f[CELLS]).
// point(j, stencil, fluxes) computes one.
template <int CELLS, class Point>
__device__ __forceinline__ void sweep_fluxes(const float (&c)[MW_VARS][CELLS], float (&f)[MW_VARS][CELLS + 1], Point &&point) {
    static_assert(CELLS >= 2, "two cells of the lane below");
    float w[MW_VARS][CELLS + 3];  // cells -2 .. CELLS
#pragma unroll
    for (int ll = 0; ll < MW_VARS; ++ll) {
        w[ll][0] = from_below(c[ll][CELLS - 2]);
        w[ll][1] = from_below(c[ll][CELLS - 1]);
#pragma unroll
        for (int j = 0; j < CELLS; ++j) w[ll][2 + j] = c[ll][j];
        w[ll][CELLS + 2] = from_above(c[ll][0]);
    }
#pragma unroll
    for (int j = 0; j < CELLS; ++j) {
        float s[MW_VARS][4], out[MW_VARS];
#pragma unroll
        for (int ll = 0; ll < MW_VARS; ++ll)
#pragma unroll
            for (int q = 0; q < 4; ++q) s[ll][q] = w[ll][j + q];
        point(j, s, out);
#pragma unroll
        for (int ll = 0; ll < MW_VARS; ++ll) f[ll][j] = out[ll];
    }
#pragma unroll
    for (int ll = 0; ll < MW_VARS; ++ll) f[ll][CELLS] = from_above(f[ll][0]);
}


// ---- x --------------------------------------------------------------------------------------------------------------
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
constexpr int SX_CELLS = 2, SX_OUT = 64 * SX_CELLS - 2 * SW_HALO;

template <bool LAST>
__device__ __forceinline__ void sweep_x(const SweepArgs &p, int item) {
#pragma clang fp contract(off)
    const int nx = p.nx, nz = p.nz, pieces = (nx + SX_OUT - 1) / SX_OUT;
    const int lane = threadIdx.x & 63;
    const int k = __builtin_amdgcn_readfirstlane(item / pieces), piece = __builtin_amdgcn_readfirstlane(item % pieces);
    if (k >= nz) return;
    const int lo = (int)((long)nx * piece / pieces), hi = (int)((long)nx * (piece + 1) / pieces);
    const unsigned W = (unsigned)(nx + 2 * MW_HS), plane = (unsigned)(nz + 2 * MW_HS) * W, row = (unsigned)(k + MW_HS) * W + MW_HS;
    const int first = lo - SW_HALO + SX_CELLS * lane;  // this lane's cells; beyond the ends the row goes round
    float init[MW_VARS][SX_CELLS], cur[MW_VARS][SX_CELLS], f[MW_VARS][SX_CELLS + 1];
    if (lo >= SW_HALO && lo - SW_HALO + 64 * SX_CELLS <= nx) {
#pragma unroll
        for (int ll = 0; ll < MW_VARS; ++ll) {
            const f32x2u v = *reinterpret_cast<const f32x2u *>(p.in + ll * plane + row + (unsigned)first);
#pragma unroll
            for (int j = 0; j < SX_CELLS; ++j) init[ll][j] = v[j];
        }
    } else {
        unsigned at[SX_CELLS];
#pragma unroll
        for (int j = 0; j < SX_CELLS; ++j) {
            int i = (first + j) % nx;
            at[j] = row + (unsigned)(i < 0 ? i + nx : i);
        }
#pragma unroll
        for (int ll = 0; ll < MW_VARS; ++ll)
#pragma unroll
            for (int j = 0; j < SX_CELLS; ++j) init[ll][j] = p.in[ll * plane + at[j]];
    }
#pragma unroll
    for (int ll = 0; ll < MW_VARS; ++ll)
#pragma unroll
        for (int j = 0; j < SX_CELLS; ++j) cur[ll][j] = init[ll][j];
    // column i of this lane's cells, as the halo columns of `to` (cells nx-2, nx-1 in front, 0, 1 behind)
    auto halo = [&](float *to, const float (&c)[MW_VARS][SX_CELLS]) {
#pragma unroll
        for (int j = 0; j < SX_CELLS; ++j) {
            const int i = first + j;
            if (i < lo || i >= hi) continue;
            for (int ll = 0; ll < MW_VARS; ++ll) {
                if (i >= nx - 2) to[ll * plane + row + (unsigned)(i - nx)] = c[ll][j];
                if (i < 2) to[ll * plane + row + (unsigned)(i + nx)] = c[ll][j];
            }
        }
    };
    const bool ends = lo < 2 || hi > nx - 2;
    if (ends) halo(p.state, init);
    const float dx_inv = 1.0f / p.dx, h0 = p.hydro[k + MW_HS], h1 = p.hydro[nz + 2 * MW_HS + k + MW_HS];
#pragma unroll 1
    for (int stage = 0; stage < 3; ++stage) {
        const float dt = p.dt[stage], hv_coef = p.hv_coef[stage];
        sweep_fluxes<SX_CELLS>(cur, f, [&](int, const float (&s)[MW_VARS][4], float (&out)[MW_VARS]) { mw_flux_x_point(s, h0, h1, hv_coef, out); });
        if (LAST && stage == 2) {  // the faces below the cells, and the row's last one
            const unsigned fplane = (unsigned)(nz + 1) * (unsigned)(nx + 1), frow = (unsigned)k * (unsigned)(nx + 1);
    #pragma unroll
            for (int j = 0; j < SX_CELLS; ++j) {
                const int i = first + j;
                if (i < lo || i >= hi) continue;
                for (int ll = 0; ll < MW_VARS; ++ll) {
                    p.flux[ll * fplane + frow + (unsigned)i] = f[ll][j];
                    if (i == nx - 1) p.flux[ll * fplane + frow + (unsigned)nx] = f[ll][j + 1];
                }
            }
        }
#pragma unroll
        for (int ll = 0; ll < MW_VARS; ++ll)
#pragma unroll
            for (int j = 0; j < SX_CELLS; ++j) {
                const float tend = mw_div(-(f[ll][j + 1] - f[ll][j]), p.dx, dx_inv);
                cur[ll][j] = init[ll][j] + dt * tend;
            }
        if (stage == 1) {
            if (ends) halo(p.state_tmp, cur);
            if constexpr (LAST) {
#pragma unroll
                for (int j = 0; j < SX_CELLS; ++j)
                    if (first + j >= lo && first + j < hi)
                        for (int ll = 0; ll < MW_VARS; ++ll) p.state_tmp[ll * plane + row + (unsigned)(first + j)] = cur[ll][j];
            }
        }
    }
    if (first >= lo && first + SX_CELLS <= hi) {
#pragma unroll
        for (int ll = 0; ll < MW_VARS; ++ll) {
            f32x2u v;
#pragma unroll
            for (int j = 0; j < SX_CELLS; ++j) v[j] = cur[ll][j];
            *reinterpret_cast<f32x2u *>(p.out + ll * plane + row + (unsigned)first) = v;
        }
    } else {
#pragma unroll
        for (int j = 0; j < SX_CELLS; ++j)
            if (first + j >= lo && first + j < hi)
                for (int ll = 0; ll < MW_VARS; ++ll) p.out[ll * plane + row + (unsigned)(first + j)] = cur[ll][j];
    }
}

// ---- z --------------------------------------------------------------------------------------------------------------
constexpr int SZ_CELLS = 2, SZ_ROWS = 64 * SZ_CELLS, SZ_OUT = SZ_ROWS - 2 * SW_HALO, SZ_COLS = 16;
constexpr int SZ_STRIDE = SZ_ROWS + 4;  // of a column in LDS: 16 columns of 4 rows fall into 64 different banks
constexpr size_t SZ_LDS = sizeof(float) * MW_VARS * SZ_COLS * SZ_STRIDE;

template <bool LAST>
__device__ __forceinline__ void sweep_z(const SweepArgs &p, int tile, float *lds) {
#pragma clang fp contract(off)
    const int nx = p.nx, nz = p.nz, strips = (nx + SZ_COLS - 1) / SZ_COLS, pieces = (nz + SZ_OUT - 1) / SZ_OUT;
    const int piece = tile / strips, col0 = (tile - piece * strips) * SZ_COLS;
    const int lo = (int)((long)nz * piece / pieces), hi = (int)((long)nz * (piece + 1) / pieces), base = lo - SW_HALO;
    const unsigned W = (unsigned)(nx + 2 * MW_HS), plane = (unsigned)(nz + 2 * MW_HS) * W;
    const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
    auto cell = [&](int k, int i) { return (unsigned)(k + MW_HS) * W + (unsigned)(i + MW_HS); };
    {
        const int c = threadIdx.x % SZ_COLS, i = col0 + c < nx ? col0 + c : nx - 1;
#pragma unroll 8
        for (int r = threadIdx.x / SZ_COLS; r < SZ_ROWS; r += MW_TILE / SZ_COLS) {
            int k = base + r;
            k = k < 0 ? 0 : k >= nz ? nz - 1 : k;  // (a wall's halo is made of the row next to it)
            const unsigned at = cell(k, i);
#pragma unroll
            for (int ll = 0; ll < MW_VARS; ++ll) lds[(ll * SZ_COLS + c) * SZ_STRIDE + r] = p.in[ll * plane + at];
        }
    }
    const MwHydro hy(p.hydro, nz);
    const int first = base + SZ_CELLS * lane;
    float h0[SZ_CELLS], h1[SZ_CELLS], h2[SZ_CELLS];
#pragma unroll
    for (int j = 0; j < SZ_CELLS; ++j) {
        int k = first + j;
        k = k < 0 ? 0 : k > nz ? nz : k;
        h0[j] = hy.dens_int[k]; h1[j] = hy.dens_theta_int[k]; h2[j] = hy.pressure_int[k];
    }
    const float dz_inv = 1.0f / p.dz;
    const bool bottom = lo == 0, top = base + SZ_ROWS > nz;
    const int top_at = nz - 1 - base;  // where the topmost row of cells is in the stretch
    __syncthreads();
#pragma unroll 1
    for (int c = wave; c < SZ_COLS; c += MW_TILE / 64) {
        if (col0 + c >= nx) break;
        float *column = lds + c * SZ_STRIDE + SZ_CELLS * lane;
        float init[MW_VARS][SZ_CELLS], cur[MW_VARS][SZ_CELLS], f[MW_VARS][SZ_CELLS + 1];
#pragma unroll
        for (int ll = 0; ll < MW_VARS; ++ll)
#pragma unroll
            for (int j = 0; j < SZ_CELLS; ++j) cur[ll][j] = init[ll][j] = column[ll * SZ_COLS * SZ_STRIDE + j];
        // solid walls: no flow through, horizontal momentum scaled by the density ratio; written to memory as the halo
        // rows of `to` where they outlive the step
        auto walls = [&](float *to) {
            for (int side = 0; side < 2; ++side) {
                if (side ? !top : !bottom) continue;
                const int at = side ? top_at : SW_HALO, from = at / SZ_CELLS, slot = at % SZ_CELLS;
#pragma unroll
                for (int ll = 0; ll < MW_VARS; ++ll) {
                    float edge = cur[ll][0];
#pragma unroll
                    for (int j = 1; j < SZ_CELLS; ++j) edge = slot == j ? cur[ll][j] : edge;
                    edge = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, edge), from));
#pragma unroll
                    for (int j = 0; j < SZ_CELLS; ++j) {
                        const int k = first + j, beyond = side ? k - nz : k + 2;  // 0 or 1 in the halo
                        if (beyond != 0 && beyond != 1) continue;
                        const float v = ll == MW_WMOM ? 0.f : ll == MW_UMOM ? edge * hy.cell_const[2 * side + beyond] : edge;
                        cur[ll][j] = v;
                        if (to && (side ? hi == nz : lo == 0)) to[ll * plane + cell(k, col0 + c)] = v;
                    }
                }
            }
        };
#pragma unroll 1
        for (int stage = 0; stage < 3; ++stage) {
            const float dt = p.dt[stage], hv_coef = p.hv_coef[stage];
            if (bottom || top) walls(!LAST || stage == 1 ? nullptr : stage == 0 ? p.state : p.state_tmp);
            sweep_fluxes<SZ_CELLS>(cur, f, [&](int j, const float (&s)[MW_VARS][4], float (&out)[MW_VARS]) {
                mw_flux_z_point(s, h0[j], h1[j], h2[j], hv_coef, first + j == 0 || first + j == nz, out);
            });
#pragma unroll
            for (int j = 0; j < SZ_CELLS; ++j) {
                float tend[MW_VARS];
#pragma unroll
                for (int ll = 0; ll < MW_VARS; ++ll) tend[ll] = mw_div(-(f[ll][j + 1] - f[ll][j]), p.dz, dz_inv);
                // gravity acts on the density of the forcing state; in the second stage, which updates in place, on the updated one
                const float updated = init[MW_DENS][j] + dt * tend[MW_DENS];
                tend[MW_WMOM] = tend[MW_WMOM] - (stage == 1 ? updated : cur[MW_DENS][j]) * MW_GRAV;
                cur[MW_DENS][j] = updated;
#pragma unroll
                for (int ll = 1; ll < MW_VARS; ++ll) cur[ll][j] = init[ll][j] + dt * tend[ll];
            }
        }
        if constexpr (LAST) {  // the top faces of the third stage
#pragma unroll
            for (int j = 0; j < SZ_CELLS; ++j)
                if (first + j == nz && hi == nz)
                    for (int ll = 0; ll < MW_VARS; ++ll) p.flux[ll * (unsigned)(nz + 1) * (unsigned)(nx + 1) + (unsigned)nz * (unsigned)(nx + 1) + (unsigned)(col0 + c)] = f[ll][j];
        }
#pragma unroll
        for (int ll = 0; ll < MW_VARS; ++ll)
#pragma unroll
            for (int j = 0; j < SZ_CELLS; ++j) column[ll * SZ_COLS * SZ_STRIDE + j] = cur[ll][j];
    }
    __syncthreads();
    {
        const int c = threadIdx.x % SZ_COLS, i = col0 + c;
        if (i < nx) {
#pragma unroll 8
            for (int r = SW_HALO + threadIdx.x / SZ_COLS; r < SW_HALO + hi - lo; r += MW_TILE / SZ_COLS) {
                const unsigned at = cell(base + r, i);
#pragma unroll
                for (int ll = 0; ll < MW_VARS; ++ll) p.out[ll * plane + at] = lds[(ll * SZ_COLS + c) * SZ_STRIDE + r];
            }
        }
    }
    if constexpr (LAST) {  // the corners: the halo columns' own rows next to the walls, as the x sweep before left them
        if (tile == 0 && threadIdx.x < 2 * MW_VARS * 4) {
            const int side = threadIdx.x / (MW_VARS * 4), ll = threadIdx.x / 4 % MW_VARS, q = threadIdx.x % 4;
            const int i = q < 2 ? q - 2 : nx + q - 2;
            for (float *to : {p.state, p.state_tmp}) {
                const float edge = to[ll * plane + cell(side ? nz - 1 : 0, i)];
                for (int beyond = 0; beyond < 2; ++beyond)
                    to[ll * plane + cell(side ? nz + beyond : beyond - 2, i)] = ll == MW_WMOM ? 0.f : ll == MW_UMOM ? edge * hy.cell_const[2 * side + beyond] : edge;
            }
        }
    }
    __syncthreads();  // (the next tile's loads overwrite what this one's stores read)
}

template <bool Z, bool LAST, int LOOP = LOOP_ANY>
__global__ __launch_bounds__(MW_TILE) void miniweather_sweep_kernel(SweepArgs p, BlpArgs blp) {
    extern __shared__ __attribute__((aligned(16))) float sweep_lds[];
    tiles<LOOP>(blp, [&](TileIdx t) {
        if constexpr (Z) sweep_z<LAST>(p, t.x, sweep_lds);
        else sweep_x<LAST>(p, t.x * (MW_TILE / 64) + (int)(threadIdx.x / 64));
    });
}

}  // namespace gp

using namespace gp;

extern "C" int gp_launch_miniweather_sweep(const gp_mw_sweep_params *p, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    GP_REQUIRE(p && p->in && p->out && p->in != p->out && p->state && p->state_tmp && p->flux && p->hydro, "miniweather sweep: operands missing");
    GP_REQUIRE(p->nx >= 4 && p->nz >= 4 && (long)p->nx * p->nz <= (1L << 27), "miniweather grid %d x %d", p->nx, p->nz);
    GP_REQUIRE(p->dt[0] > 0 && p->dt[1] > 0 && p->dt[2] > 0 && p->dx > 0 && p->dz > 0, "miniweather steps must be positive");
    SweepArgs args;
    static_cast<gp_mw_sweep_params &>(args) = *p;
    for (int stage = 0; stage < 3; ++stage) args.hv_coef[stage] = -MW_HV_BETA * (p->dir_z ? p->dz : p->dx) / (16 * p->dt[stage]);
    if (p->dir_z) {
        const int tiles = (p->nx + SZ_COLS - 1) / SZ_COLS * ((p->nz + SZ_OUT - 1) / SZ_OUT);
        return p->last ? launch_tiles(GP_KSET(miniweather_sweep_kernel<true, true), tiles, 1, ctx, s, info, args, SZ_LDS, 1)
                       : launch_tiles(GP_KSET(miniweather_sweep_kernel<true, false), tiles, 1, ctx, s, info, args, SZ_LDS, 1);
    }
    const long waves = (long)p->nz * ((p->nx + SX_OUT - 1) / SX_OUT);
    const int tiles = (int)((waves + MW_TILE / 64 - 1) / (MW_TILE / 64));
    return p->last ? launch_tiles(GP_KSET(miniweather_sweep_kernel<false, true), tiles, 1, ctx, s, info, args, 0, 1)
                   : launch_tiles(GP_KSET(miniweather_sweep_kernel<false, false), tiles, 1, ctx, s, info, args, 0, 1);
}
