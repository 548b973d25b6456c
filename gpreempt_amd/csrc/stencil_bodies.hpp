// Tile bodies of the miniWeather workload: a 2-D stratified-flow solver (finite-volume fluxes with
// fourth-order interface values and hyperviscosity, three-stage Runge-Kutta, x and z sweeps) that
// the reference ships as its non-DNN preemptible workload (src/workloads/miniweather.tr.cu).
// Every kernel of a semi-discrete step is a list of 256-element tiles handed out by the same
// dispatcher as the DNN operators; the in-place state update of the last Runge-Kutta stage is not
// idempotent, which is exactly what "every tile exactly once" has to survive.
//
// Arithmetic follows the reference: fp32 state, x flux formed in fp64 (miniweather.tr.cu:337-348),
// z flux in fp32 (:447-466).  Contraction into fused multiply-adds is switched off in these
// bodies so that results do not depend on how the compiler pairs the operations.
//
// Element ids map to cells as in the reference (:322-324, :382-385, :430-432, :486-489, :511-513,
// :531-533); one lane owns one id, a wavefront reads and writes 256 contiguous bytes per access.
#pragma once
#include <hip/hip_runtime.h>
#include "../../include/gpreempt_hip.h"
#include "tile_loop.hpp"

namespace gp {

constexpr int MW_TILE = 256;
constexpr int MW_HS = 2, MW_VARS = 4, MW_DENS = 0, MW_UMOM = 1, MW_WMOM = 2, MW_RHOT = 3;
constexpr float MW_GRAV = 9.8f, MW_C0 = 27.5629410929725921310572974482f, MW_GAMMA = 1.40027894002789400278940027894f;
constexpr float MW_HV_BETA = 0.05f;

__host__ __device__ inline long mw_ids(int kernel, int nx, int nz) {
    switch (kernel) {
        case GP_MW_HALO_X: return (long)nz * MW_VARS;
        case GP_MW_FLUX_X: return (long)nz * (nx + 1);
        case GP_MW_UPDATE_X: return (long)nz * nx * MW_VARS;
        case GP_MW_HALO_Z: return (long)(nx + 2 * MW_HS) * MW_VARS;
        case GP_MW_FLUX_Z: return (long)nx * (nz + 1);
        case GP_MW_UPDATE_Z: return (long)nx * nz * MW_VARS;
    }
    return 0;
}

struct MwView {
    int nx, nz;
    __device__ __forceinline__ long st(int ll, int k, int i) const { return ((long)ll * (nz + 2 * MW_HS) + k) * (nx + 2 * MW_HS) + i; }
    __device__ __forceinline__ long fx(int ll, int k, int i) const { return ((long)ll * (nz + 1) + k) * (nx + 1) + i; }
};

// x / 12 with the bits of the division (checked against it on 1.5 * 10^7 random floats): the product with the rounded
// reciprocal, corrected by the exact remainder.  Three instructions for the eleven of an fp32 division, in kernels
// whose time is the number of vector instructions they issue per cell.
__device__ __forceinline__ float mw_div12(float x) {
    const float c = 1.0f / 12.0f;
    const float q = x * c;
    const float r = __builtin_fmaf(-q, 12.0f, x);
    return __builtin_fmaf(r, c, q);
}

// The (row, column) of a claim's ids in rows of w ids: one division per claim, then additions, instead of a
// division per id (twenty vector instructions).
struct MwCursor {
    unsigned w, i;
    int k;
    __device__ __forceinline__ MwCursor(unsigned id0, unsigned w_) : w(w_) { k = (int)(id0 / w); i = id0 - (unsigned)k * w; }
    __device__ __forceinline__ void next_tile() {
        i += MW_TILE;
        while (i >= w) { i -= w; ++k; }
    }
    __device__ __forceinline__ void lane(int &kl, int &il) const {
        unsigned x = i + threadIdx.x;
        int kk = k;
        while (x >= w) { x -= w; ++kk; }
        kl = kk; il = (int)x;
    }
};

// fourth-order interface value and (scaled) third difference from four cell averages
// (Here and in the fluxes a product and the sum it goes into are one fused operation, written out so that the kernels and the sweeps
// round alike: a rounding less each, and 24 of a face's 129 vector instructions, which is what these kernels' time goes by.)
__device__ __forceinline__ void mw_reconstruct(const float (&s)[4], float hv_coef, float &val, float &d3) {
#pragma clang fp contract(off)
    val = mw_div12(__builtin_fmaf(7.0f, s[1] + s[2], -s[0]) - s[3]);
    d3 = (__builtin_fmaf(3.0f, s[1] - s[2], -s[0]) + s[3]) * hv_coef;
}

// Pointers into the hydrostatic background buffer: cell density, cell density*theta (nz+4 each),
// interface density, density*theta, pressure (nz+1 each), four boundary density ratios.
struct MwHydro {
    const float *dens_cell, *dens_theta_cell, *dens_int, *dens_theta_int, *pressure_int, *cell_const;
    __device__ __forceinline__ MwHydro(const float *h, int nz) {
        dens_cell = h;
        dens_theta_cell = dens_cell + nz + 2 * MW_HS;
        dens_int = dens_theta_cell + nz + 2 * MW_HS;
        dens_theta_int = dens_int + nz + 1;
        pressure_int = dens_theta_int + nz + 1;
        cell_const = pressure_int + nz + 1;
    }
};

// What one element id reads, split from what it computes and writes so that a lane can have the
// loads of several ids in flight before the first result is needed (an id alone keeps 12-72 bytes
// in flight per lane, too few to cover HBM latency at 32 waves per CU).
template <int KIND> struct MwOperands;

template <> struct MwOperands<GP_MW_UPDATE_X> { unsigned c; float f0, f1, init; };
template <> struct MwOperands<GP_MW_UPDATE_Z> { unsigned c; int ll; float f0, f1, init, d0, d1, dinit; };
template <> struct MwOperands<GP_MW_FLUX_X> { int k, i; float s[MW_VARS][4], h0, h1; };
template <> struct MwOperands<GP_MW_FLUX_Z> { int k, i; float s[MW_VARS][4], h0, h1, h2; };

// a / b from the correctly rounded reciprocal c of b: the product, corrected by its exact remainder, which is the
// rounded quotient itself (Markstein's sequence; three instructions for the eleven of an fp32 division)
__device__ __forceinline__ float mw_div(float a, float b, float c) {
    const float q = a * c;
    const float r = __builtin_fmaf(-q, b, a);
    return __builtin_fmaf(r, c, q);
}
// an update id is (field, level, column): the cursor gives field * nz + level and the column
__device__ __forceinline__ bool mw_update_cell(const gp_miniweather_params &p, const MwCursor &cur, int &ll, int &k, int &i) {
    int row;
    cur.lane(row, i);
    const int nz = p.nz;
    if (row >= MW_VARS * nz) return false;
    ll = (row >= nz) + (row >= 2 * nz) + (row >= 3 * nz);
    k = row - ll * nz;
    return true;
}
__device__ __forceinline__ bool mw_load(const gp_miniweather_params &p, const MwCursor &cur, MwOperands<GP_MW_UPDATE_X> &o) {
    int ll, k, i;
    if (!mw_update_cell(p, cur, ll, k, i)) return false;
    o.c = (unsigned)(ll * (p.nz + 2 * MW_HS) + k + MW_HS) * (unsigned)(p.nx + 2 * MW_HS) + (unsigned)(i + MW_HS);
    const unsigned f = (unsigned)(ll * (p.nz + 1) + k) * (unsigned)(p.nx + 1) + (unsigned)i;
    o.f0 = p.flux[f];
    o.f1 = p.flux[f + 1];
    o.init = p.state_init[o.c];
    return true;
}
__device__ __forceinline__ void mw_finish(const gp_miniweather_params &p, const MwOperands<GP_MW_UPDATE_X> &o) {
#pragma clang fp contract(off)
    const float tend = mw_div(-(o.f1 - o.f0), p.dx, 1.0f / p.dx);
    p.state_out[o.c] = o.init + p.dt * tend;
}

__device__ __forceinline__ bool mw_load(const gp_miniweather_params &p, const MwCursor &cur, MwOperands<GP_MW_UPDATE_Z> &o) {
    int ll, k, i;
    if (!mw_update_cell(p, cur, ll, k, i)) return false;
    o.ll = ll;
    const unsigned srow = (unsigned)(p.nx + 2 * MW_HS), frow = (unsigned)(p.nx + 1);
    o.c = (unsigned)(ll * (p.nz + 2 * MW_HS) + k + MW_HS) * srow + (unsigned)(i + MW_HS);
    const unsigned f = (unsigned)(ll * (p.nz + 1) + k) * frow + (unsigned)i;
    o.f0 = p.flux[f];
    o.f1 = p.flux[f + frow];
    o.init = p.state_init[o.c];
    o.d0 = o.d1 = o.dinit = 0.f;
    if (ll == MW_WMOM) {
        // Gravity acts on the density of the forcing state.  When the forcing state is also the
        // output (second Runge-Kutta stage) other lanes overwrite that density in this very
        // kernel; in element order the density ids come first, so the value defined for this read
        // is the UPDATED one, which is recomputed from operands the kernel never writes instead
        // of being read while it changes.
        const unsigned cd = (unsigned)(k + MW_HS) * srow + (unsigned)(i + MW_HS), fd = (unsigned)k * frow + (unsigned)i;  // field 0
        if (p.state == p.state_out) {
            o.d0 = p.flux[fd];
            o.d1 = p.flux[fd + frow];
            o.dinit = p.state_init[cd];
        } else {
            o.dinit = p.state[cd];
        }
    }
    return true;
}
__device__ __forceinline__ void mw_finish(const gp_miniweather_params &p, const MwOperands<GP_MW_UPDATE_Z> &o) {
#pragma clang fp contract(off)
    const float dz_inv = 1.0f / p.dz;
    float tend = mw_div(-(o.f1 - o.f0), p.dz, dz_inv);
    if (o.ll == MW_WMOM) {
        float dens = o.dinit;
        if (p.state == p.state_out) {
            const float td = mw_div(-(o.d1 - o.d0), p.dz, dz_inv);
            dens = o.dinit + p.dt * td;
        }
        tend = tend - dens * MW_GRAV;
    }
    p.state_out[o.c] = o.init + p.dt * tend;
}

// 1 / a in fp64: the hardware's estimate (2^-23) and two Newton steps, which leaves an error of the last bit or two.
// (The compiler's own a / b is correctly rounded and handles zeros, infinities and denormals: 15 instructions with the
// scaling and the fix-up; the densities divided by here are ordinary numbers, and the quotient goes into a flux that is
// stored in fp32.)
__device__ __forceinline__ double mw_rcp(double a) {
    double y = __builtin_amdgcn_rcp(a);
    double e = __builtin_fma(-a, y, 1.0);
    y = __builtin_fma(y, e, y);
    e = __builtin_fma(-a, y, 1.0);
    return __builtin_fma(y, e, y);
}
// x^gamma in fp64 for a positive x of fp32's range (the flux kernels raise rho*theta, about 10^4-10^5): the library's
// pow, or its exp(g log(x)), spend two thirds of their 110 instructions on arguments that cannot occur here and on the
// last bits of a result that is rounded to fp32 when the flux is stored.  With x = 2^e m and m in [1/2, 1), m^gamma is
// a polynomial of degree 15 (interpolated at Chebyshev nodes; good to 1.4 10^-15 with the rounding of its evaluation)
// and 2^(gamma e) comes from a table: 22 instructions, where a series for the logarithm and one for the exponential
// (to 10^-14) took 45.
// (An infinity does not get here, where the polynomial would make -inf of it: reconstruction divides by 12 by a corrected
// product, which makes NaN of infinities, and leaves at most a twelfth of fp32's range.)  The table and the coefficients
// are checked against the power itself in tests/test_pow_table_cpu.py.
static_assert(MW_GAMMA == 1.40027894002789400278940027894f, "mw_pow2_gamma and the polynomial of mw_pow_gamma are for this exponent, rounded to fp32");
constexpr int MW_POW_E0 = -149;
static __constant__ double mw_pow2_gamma[278] = {
    1.5582319697246894e-63, 4.1129939375444373e-63, 1.08563548040066e-62, 2.865563174178731e-62, 7.563728759287419e-62, 1.9964659393861715e-61,
    5.269723933760706e-61, 1.390957380749932e-60, 3.671468295839132e-60, 9.690936353552659e-60, 2.5579479336657038e-59, 6.751770306432742e-59,
    1.782147387398094e-58, 4.704024524329383e-58, 1.2416395457503978e-57, 3.2773399747337373e-57, 8.650624367393457e-57, 2.2833548707994867e-56,
    6.026974753008142e-56, 1.5908357101180264e-55, 4.1990523609271646e-55, 1.1083508257744509e-54, 2.9255209209243183e-54, 7.721988796088612e-54,
    2.0382390889919953e-53, 5.379985251984877e-53, 1.420061143361207e-52, 3.7482884365535195e-52, 9.893705119165527e-52, 2.611469278362312e-51,
    6.893041292103295e-51, 1.8194362326344408e-50, 4.802449404177166e-50, 1.2676190495715775e-49, 3.345913552861392e-49, 8.831626115910146e-49,
    2.3311307545445504e-48, 6.153080444601027e-48, 1.6241216364171143e-47, 4.2869114318059937e-47, 1.1315414567526329e-46, 2.9867331964226483e-46,
    7.883560194262668e-46, 2.0808862810713542e-45, 5.4925536281212545e-45, 1.4497738599274026e-44, 3.8267159271192085e-44, 1.0100716526645825e-43,
    2.666110479448658e-43, 7.03726816793103e-43, 1.857505292789538e-42, 4.9029336816583894e-42, 1.2941421367709647e-41, 3.4159219334976304e-41,
    9.016415063081488e-41, 2.3799062792551125e-40, 6.281824714602454e-40, 1.6581040223710496e-39, 4.376608826114061e-39, 1.155217317996052e-38,
    3.049226249865475e-38, 8.048512239236048e-38, 2.1244258036933257e-37, 5.607477334005294e-37, 1.4801082719254254e-36, 3.906784398996914e-36,
    1.0312059347111532e-35, 2.721894968292933e-35, 7.184512781623596e-35, 1.8963708927271775e-34, 5.005520446676939e-34, 1.3212201810411088e-33,
    3.4873951378006714e-33, 9.205070450537838e-33, 2.429702360966243e-32, 6.41326277143268e-32, 1.6927974403863952e-31, 4.468183008098674e-31,
    1.1793885622431362e-30, 3.1130268796707586e-30, 8.216915666132117e-30, 2.1688763275782653e-29, 5.724805651490483e-29, 1.5110773874290776e-28,
    3.9885281873368107e-28, 1.0527824209087322e-27, 2.778846666530669e-27, 7.334838274962084e-27, 1.9360496988852118e-26, 5.1102536907303454e-26,
    1.3488647940525547e-25, 3.56036381507786e-25, 9.397673177925559e-25, 2.4805403533506618e-24, 6.547450978667953e-24, 1.7282167677761515e-23,
    4.5616732468156403e-23, 1.2040655546636166e-22, 3.1781624449744266e-22, 8.388842690103939e-22, 2.2142569141042306e-21, 5.8445888935815066e-21,
    1.5426944866872093e-20, 4.071982345702213e-20, 1.0748103637368091e-19, 2.836989996322872e-19, 7.488309110877631e-19, 1.9765587264224945e-18,
    5.21717832577432e-18, 1.3770878304331853e-17, 3.634859255928775e-17, 9.59430583759859e-17, 2.532442056875671e-16, 6.684446879210481e-16,
    1.7643771931394824e-15, 4.657119632968714e-15, 1.229258877303344e-14, 3.244660877362582e-14, 8.564367037301755e-14, 2.2605870234809245e-13,
    5.966878426009583e-13, 1.5749731278185865e-12, 4.1571826611013274e-12, 1.0972992092695668e-11, 2.8963498908287894e-11, 7.644991101094564e-11,
    2.0179153465153618e-10, 5.326340203482004e-10, 1.4059013928517513e-09, 3.7109134056633353e-09, 9.795052750035903e-09, 2.5854297281516823e-08,
    6.824309219964109e-08, 1.8012942228749257e-07, 4.754563096101391e-07, 1.2549793336221065e-06, 3.312550692849193e-06, 8.7435639764884e-06,
    2.30788652309467e-05, 6.091726689259241e-05, 0.0001607927152625915, 0.0004244165669333521, 0.001120258601226568, 0.002956951804897807,
    0.00780495143435194, 0.020601372938067797, 0.054377861349061966, 0.14353178372077663, 0.37885588780006657, 1.0,
    2.6395260894763486, 6.967097977026306, 18.389836878298823, 48.54045422148404, 128.1237953126395, 338.18610041043945,
    892.6510351316231, 2356.1756960279877, 6219.187221055969, 16415.706925315142, 43329.68670656689, 114369.83851081984,
    301882.1725985058, 796825.8705215581, 2103242.6740113557, 5551563.910552973, 14653497.779299915, 38678289.690545864,
    102092354.7345199, 269475433.85783947, 711287438.1407255, 1877461750.0892396, 4955609271.354472, 13080459960.991009,
    34526215329.38655, 91132846132.79404, 240547524975.74365, 634931467932.439, 1675918174637.1882, 4423629745782.438,
    11676286124176.373, 30819861852954.215, 81349829434929.53, 214724997167947.53, 566772232087532.5, 1496010093385786.2,
    3948757671611732.0, 1.0422848895239046e+16, 2.7511381585653204e+16, 7.261700945287083e+16, 1.9167449099060317e+17, 5.059298196567964e+17,
    1.3354149584281782e+18, 3.52486262304815e+18, 9.30396685535563e+18, 2.4558063250334405e+19, 6.4821648656268e+19, 1.710984327910889e+20,
    4.516187772205947e+20, 1.1920595449711666e+21, 3.146472269160699e+21, 8.305195644263514e+21, 2.1921780581238877e+22, 5.786311177195601e+22,
    1.5273119314036394e+23, 4.031379689708418e+23, 1.0640931867570435e+24, 2.808701728079245e+24, 7.413641488822473e+24, 1.9568500127771198e+25,
    5.165156661917334e+25, 1.3633565765363372e+26, 3.5986152530268204e+26, 9.498638846351824e+26, 2.507190504945917e+27, 6.617794749092128e+27,
    1.7467841895028257e+28, 4.610682440877507e+28, 1.2170016592986672e+29, 3.2123076306548386e+29, 8.478969798537402e+29, 2.238046199512149e+30,
    5.907381333065707e+30, 1.5592687149112505e+31, 4.115730453512505e+31, 1.0863577909298582e+32, 2.8674697316652534e+32, 7.568761167514181e+32,
    1.9977942566669148e+33, 5.273230061878331e+33, 1.3918828324138835e+34, 3.673911049650682e+34, 9.697384065968412e+34, 2.559649824179586e+35,
    6.756262490845566e+35, 1.7833331111937332e+36, 4.707154273222885e+36, 1.2424656511361886e+37, 3.279520501452189e+37, 8.656379924555611e+37,
    2.2848740651283844e+38, 6.030984706074252e+38, 1.5918941476915836e+39, 4.201846134516651e+39, 1.1090882496022048e+40, 2.927467370356676e+40,
    7.727126500147167e+40, 2.0395951993822517e+41, 5.383564740740168e+41, 1.421005958756865e+42, 3.7507823014400976e+42, 9.90028774059728e+42,
    2.6132067784629376e+43, 6.897627468949365e+43, 1.820646765978056e+44, 4.8056446385198195e+44, 1.26846244001252e+45, 3.348139703933874e+45,
    8.83750209974508e+45, 2.3326817358079153e+46, 6.157174300109967e+46, 1.6252022202593537e+47, 4.289763661049451e+47, 1.1322943101027603e+48,
    2.9887203724818594e+48, 7.888805397315338e+48, 2.0822707661015668e+49, 5.496208012478989e+49, 1.4507384442127241e+50, 3.8292619725058135e+50,
    1.0107436879868759e+51, 2.6678843342149016e+51, 7.04195030386547e+51, 1.8587411547848814e+52, 4.90619577163809e+52, 1.2950031739317287e+53,
    3.4181946635474753e+53, 9.02241399334239e+53};
__device__ __forceinline__ double mw_pow_gamma(double x) {
    const int e = __builtin_amdgcn_frexp_exp(x);
    const double scale = mw_pow2_gamma[(e < MW_POW_E0 ? MW_POW_E0 : e > 128 ? 128 : e) - MW_POW_E0], w = __builtin_amdgcn_frexp_mant(x) - 0.75;
    double q = -0.04456402927938865;
    q = __builtin_fma(q, w, 0.039499117535868794);
    q = __builtin_fma(q, w, -0.024319698187610598);
    q = __builtin_fma(q, w, 0.02244029704451375);
    q = __builtin_fma(q, w, -0.02224187094413812);
    q = __builtin_fma(q, w, 0.021330521217560506);
    q = __builtin_fma(q, w, -0.020983590087007748);
    q = __builtin_fma(q, w, 0.021461744764258113);
    q = __builtin_fma(q, w, -0.02299800593177916);
    q = __builtin_fma(q, w, 0.026249305914012522);
    q = __builtin_fma(q, w, -0.03281413517020012);
    q = __builtin_fma(q, w, 0.0473331575989851);
    q = __builtin_fma(q, w, -0.08876514527419548);
    q = __builtin_fma(q, w, 0.3330241098559923);
    q = __builtin_fma(q, w, 1.247970183953812);
    q = __builtin_fma(q, w, 0.6684222840579125);
    return q * scale;
}
// 1 / b of an ordinary fp32 number to the last bit or so, for mw_div, whose correction makes the quotient the rounded one
__device__ __forceinline__ float mw_rcpf(float b) {
    const float y = __builtin_amdgcn_rcpf(b);
    return __builtin_fmaf(__builtin_fmaf(-b, y, 1.0f), y, y);
}

__device__ __forceinline__ bool mw_load(const gp_miniweather_params &p, const MwCursor &cur, MwOperands<GP_MW_FLUX_X> &o) {
    const MwHydro hy(p.hydro, p.nz);
    cur.lane(o.k, o.i);
    if (o.k >= p.nz) return false;
    // (32-bit offsets from the base: the four fields together stay below 2^31 elements, gp_launch_miniweather)
    const unsigned plane = (unsigned)(p.nz + 2 * MW_HS) * (unsigned)(p.nx + 2 * MW_HS);
    const unsigned at = (unsigned)(o.k + MW_HS) * (unsigned)(p.nx + 2 * MW_HS) + (unsigned)o.i;
#pragma unroll
    for (int ll = 0; ll < MW_VARS; ++ll) {
        const float *c = p.state + (at + (unsigned)ll * plane);
#pragma unroll
        for (int s = 0; s < 4; ++s) o.s[ll][s] = c[s];
    }
    o.h0 = hy.dens_cell[o.k + MW_HS];
    o.h1 = hy.dens_theta_cell[o.k + MW_HS];
    return true;
}
// the four fluxes through one x interface from the four cell averages around it (miniweather.tr.cu:337-348)
__device__ __forceinline__ void mw_flux_x_point(const float (&s)[MW_VARS][4], float h0, float h1, float hv_coef, float (&f)[MW_VARS]) {
#pragma clang fp contract(off)
    float vals[MW_VARS], d3[MW_VARS];
#pragma unroll
    for (int ll = 0; ll < MW_VARS; ++ll) mw_reconstruct(s[ll], hv_coef, vals[ll], d3[ll]);
    const double r = vals[MW_DENS] + h0;
    // (one reciprocal for the three quotients, and a power function for arguments that occur: with the compiler's
    // divisions and exp(gamma log(.)) this kernel spent 55 us on 35 us of memory traffic; a general pow made it 80)
    const double r_inv = mw_rcp(r);
    const double u = vals[MW_UMOM] * r_inv;
    const double w = vals[MW_WMOM] * r_inv;
    const double th = (vals[MW_RHOT] + h1) * r_inv;
    const double pr = MW_C0 * mw_pow_gamma(r * th);
    const double ru = r * u;
    f[MW_DENS] = (float)(ru - d3[MW_DENS]);
    f[MW_UMOM] = (float)(__builtin_fma(ru, u, pr) - d3[MW_UMOM]);
    f[MW_WMOM] = (float)__builtin_fma(ru, w, -(double)d3[MW_WMOM]);
    f[MW_RHOT] = (float)__builtin_fma(ru, th, -(double)d3[MW_RHOT]);
}
__device__ __forceinline__ void mw_finish(const gp_miniweather_params &p, const MwOperands<GP_MW_FLUX_X> &o) {
    const MwView v{p.nx, p.nz};
    const float hv_coef = -MW_HV_BETA * p.dx / (16 * p.dt);
    float f[MW_VARS];
    mw_flux_x_point(o.s, o.h0, o.h1, hv_coef, f);
    const unsigned plane = (unsigned)(p.nz + 1) * (unsigned)(p.nx + 1), at = (unsigned)o.k * (unsigned)(p.nx + 1) + (unsigned)o.i;
#pragma unroll
    for (int ll = 0; ll < MW_VARS; ++ll) p.flux[at + (unsigned)ll * plane] = f[ll];
}

__device__ __forceinline__ bool mw_load(const gp_miniweather_params &p, const MwCursor &cur, MwOperands<GP_MW_FLUX_Z> &o) {
    const MwHydro hy(p.hydro, p.nz);
    cur.lane(o.k, o.i);
    if (o.k >= p.nz + 1) return false;
    const unsigned row = (unsigned)(p.nx + 2 * MW_HS), plane = (unsigned)(p.nz + 2 * MW_HS) * row;
    const unsigned at = (unsigned)o.k * row + (unsigned)(o.i + MW_HS);
#pragma unroll
    for (int ll = 0; ll < MW_VARS; ++ll) {
        const float *c = p.state + (at + (unsigned)ll * plane);
#pragma unroll
        for (int s = 0; s < 4; ++s) o.s[ll][s] = c[(unsigned)s * row];
    }
    o.h0 = hy.dens_int[o.k];
    o.h1 = hy.dens_theta_int[o.k];
    o.h2 = hy.pressure_int[o.k];
    return true;
}
// the four fluxes through one z interface (miniweather.tr.cu:447-466); wall: the bottom or the top face
__device__ __forceinline__ void mw_flux_z_point(const float (&s)[MW_VARS][4], float h0, float h1, float h2, float hv_coef, bool wall, float (&f)[MW_VARS]) {
#pragma clang fp contract(off)
    float vals[MW_VARS], d3[MW_VARS];
#pragma unroll
    for (int ll = 0; ll < MW_VARS; ++ll) mw_reconstruct(s[ll], hv_coef, vals[ll], d3[ll]);
    const float r = vals[MW_DENS] + h0;
    const float r_inv = mw_rcpf(r);  // one reciprocal for three quotients, each rounded as a division rounds it
    const float u = mw_div(vals[MW_UMOM], r, r_inv);
    float w = mw_div(vals[MW_WMOM], r, r_inv);
    const float th = mw_div(vals[MW_RHOT] + h1, r, r_inv);
    // (the power through the fp64 routine above, rounded to fp32 once: nearer to the exact power than powf is, and cheaper
    // than the library's powf, which carries its logarithm in two floats: 4-7 us per launch at 3200 x 1600)
    const float pr = MW_C0 * (float)mw_pow_gamma((double)(r * th)) - h2;
    if (wall) {  // no flow through the bottom and top faces, exact mass conservation
        w = 0.f;
        d3[MW_DENS] = 0.f;
    }
    const float rw = r * w;
    f[MW_DENS] = rw - d3[MW_DENS];
    f[MW_UMOM] = __builtin_fmaf(rw, u, -d3[MW_UMOM]);
    f[MW_WMOM] = __builtin_fmaf(rw, w, pr) - d3[MW_WMOM];
    f[MW_RHOT] = __builtin_fmaf(rw, th, -d3[MW_RHOT]);
}
__device__ __forceinline__ void mw_finish(const gp_miniweather_params &p, const MwOperands<GP_MW_FLUX_Z> &o) {
    float f[MW_VARS];
    mw_flux_z_point(o.s, o.h0, o.h1, o.h2, -MW_HV_BETA * p.dz / (16 * p.dt), o.k == 0 || o.k == p.nz, f);
    const unsigned plane = (unsigned)(p.nz + 1) * (unsigned)(p.nx + 1), at = (unsigned)o.k * (unsigned)(p.nx + 1) + (unsigned)o.i;
#pragma unroll
    for (int ll = 0; ll < MW_VARS; ++ll) p.flux[at + (unsigned)ll * plane] = f[ll];
}

// halo kernels: a few thousand ids, nothing to overlap
template <int KIND>
__device__ __forceinline__ void mw_halo(const gp_miniweather_params &p, long id) {
#pragma clang fp contract(off)
    const MwView v{p.nx, p.nz};
    const int nx = p.nx, nz = p.nz;
    if constexpr (KIND == GP_MW_HALO_X) {  // periodic in x
        const int ll = (int)(id / nz), k = (int)(id % nz);
        if (ll < MW_VARS) {
            float *row = p.state + v.st(ll, k + MW_HS, 0);
            const float a = row[nx + MW_HS - 2], b = row[nx + MW_HS - 1], c = row[MW_HS], d = row[MW_HS + 1];
            row[0] = a; row[1] = b; row[nx + MW_HS] = c; row[nx + MW_HS + 1] = d;
        }
    } else {  // solid walls: no flow through, horizontal momentum scaled by the density ratio
        const MwHydro hy(p.hydro, nz);
        const int i = (int)(id % (nx + 2 * MW_HS)), ll = (int)(id / (nx + 2 * MW_HS));
        if (ll < MW_VARS) {
            float *s = p.state;
            if (ll == MW_WMOM) {
                s[v.st(ll, 0, i)] = 0.f; s[v.st(ll, 1, i)] = 0.f;
                s[v.st(ll, nz + MW_HS, i)] = 0.f; s[v.st(ll, nz + MW_HS + 1, i)] = 0.f;
            } else {
                const float lo = s[v.st(ll, MW_HS, i)], hi = s[v.st(ll, nz + MW_HS - 1, i)];
                const bool um = ll == MW_UMOM;
                s[v.st(ll, 0, i)] = um ? lo * hy.cell_const[0] : lo;
                s[v.st(ll, 1, i)] = um ? lo * hy.cell_const[1] : lo;
                s[v.st(ll, nz + MW_HS, i)] = um ? hi * hy.cell_const[2] : hi;
                s[v.st(ll, nz + MW_HS + 1, i)] = um ? hi * hy.cell_const[3] : hi;
            }
        }
    }
}

// Tiles [first, last) of one claim: U tiles at a time, all loads first.  The ids of different
// tiles never touch the same output element, and an update reads the element it writes only
// through its own lane, so issuing the loads of U tiles ahead of their stores changes nothing.
template <int KIND>
__device__ __forceinline__ void mw_span(const gp_miniweather_params &p, int first, int last) {
    if constexpr (KIND == GP_MW_HALO_X || KIND == GP_MW_HALO_Z) {
        for (int t = first; t < last; ++t) mw_halo<KIND>(p, (long)t * MW_TILE + threadIdx.x);
    } else {
#ifndef GP_MW_FLUX_U
#define GP_MW_FLUX_U 1  // (measured 2 and 3: 3 and 8 % slower per execute; the flux kernels are bound by the instructions they issue)
#endif
        constexpr bool FLUX = KIND == GP_MW_FLUX_X || KIND == GP_MW_FLUX_Z;
        constexpr int U = FLUX ? GP_MW_FLUX_U : 4;
        MwCursor cur((unsigned)first * MW_TILE, KIND == GP_MW_FLUX_X ? (unsigned)p.nx + 1 : (unsigned)p.nx);
        for (int t = first; t < last; t += U) {
            MwOperands<KIND> op[U];
            bool ok[U];
#pragma unroll
            for (int j = 0; j < U; ++j) {
                ok[j] = t + j < last && mw_load(p, cur, op[j]);
                cur.next_tile();
            }
#pragma unroll
            for (int j = 0; j < U; ++j)
                if (ok[j]) mw_finish(p, op[j]);
        }
    }
}

template <int KIND, int LOOP = LOOP_ANY>
__global__ __launch_bounds__(MW_TILE) void miniweather_kernel(gp_miniweather_params p, BlpArgs blp) {
    spans<LOOP>(blp, [&](int first, int last) { mw_span<KIND>(p, first, last); });
}

}  // namespace gp
