// Drop-in device calculation entry points (fdtd_calculations.h).
//
// These replace the reference's five __global__ kernels and
// copySymbolsToDevice (fdtd_calculations.cu:7-428) one for one, with the same
// pointer lists, ranges and arithmetic (float products and sums, the double
// promotions of the Debye update, float Mur with correctly rounded sqrt and
// division).  Built with -ffp-contract=off, they are bit-identical to a
// straight C evaluation of the reference's equations.
//
// Launch geometry is the library's: lanes over the flattened planes or grid,
// 256 lanes per block, so every lane of a wave64 is busy whatever nx is
// (the reference's (128,1,1) blocks leave half the lanes idle at nx = 64).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>

#include "fdtd_calculations.h"
#include "fdtd_internal.h"

namespace {

struct LegacyParams {
    int nx, ny, nz;
    float dt, dx, dy, dz, mu0, eps0;
    int nsrc;
    int njz;
    int debye_mode;
    // from the host: dt/(mu0*d), dt/d per axis, rounded as the reference's
    // float expressions, and the multiplies that divide by nx and nx*ny
    float chx, chy, chz, cdx, cdy, cdz;
    uint32_t nx_mul, nx_shift, nxy_mul, nxy_shift;
};

__constant__ LegacyParams c_p;
__constant__ int c_sources[D_MAX_SOURCES * 3];
__constant__ float c_jz[D_MAX_JZ];

LegacyParams h_p = {0, 0, 0, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0, 0, FDTD_DEBYE_FIXED, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0, 0, 0, 0};
bool h_params_set = false;

constexpr int kBlock = 256;

// A cell number (Q: uint32_t, or size_t for grids of 2^32 cells and more) is
// divided by nx and nx*ny with a multiply each (div_by); two 64-bit divisions
// cost more instructions than the whole H update.
template <typename Q>
__device__ __forceinline__ int row_of(const LegacyParams &p, Q q)   // q / nx
{
    if constexpr (sizeof(Q) == 4) return (int)div_by(q, p.nx_mul, p.nx_shift);
    else return (int)(q / (Q)p.nx);
}

// The lane's cell of the flattened grid; false: past its end.
template <typename Q>
__device__ __forceinline__ bool flat_cell(const LegacyParams &p, Q &o, int &i, int &j, int &k)
{
    const Q nxy = (Q)p.nx * (Q)p.ny;
    o = blockIdx.x * (Q)kBlock + threadIdx.x;
    if (o >= nxy * (Q)p.nz) return false;
    if constexpr (sizeof(Q) == 4) k = (int)div_by(o, p.nxy_mul, p.nxy_shift);
    else k = (int)(o / nxy);
    const Q r = o - (Q)k * nxy;
    j = row_of(p, r);
    i = (int)(r - (Q)j * (Q)p.nx);
    return true;
}

// Plane pairs over blockIdx.y, in groups of kPairs over blockIdx.z (H and D).
constexpr int kPairs = 32768;

// A load that the compiler does not merge with its neighbour's (a wave's
// 8-byte load takes three times the address unit's cycles of a 4-byte one).
template <typename Q>
__device__ __forceinline__ float ld(const float *p, Q q)
{
    return __hip_atomic_load(p + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// Own-cell operands and results: streaming ones (ST) where the grid's arrays
// exceed the Infinity Cache.
template <bool ST, typename Q>
__device__ __forceinline__ float ld_own(const float *p, Q q)
{
    if (ST) return __builtin_nontemporal_load(p + q);
    return ld(p, q);
}
template <bool ST, typename Q>
__device__ __forceinline__ void st_own(float *p, Q q, float v)
{
    if (ST) __builtin_nontemporal_store(v, p + q);
    else p[q] = v;
}

// H and D: one lane per pair of cells one above the other, so that a plane's
// values serve as the next one's neighbours, and every load of the two ahead
// of the first use, with neighbours outside the grid clamped to the cell
// (those updates are masked).  100^3 in the Infinity Cache on MI355X (us): H
// 7.7 -> 5.8, D 8.8 -> 6.4 against one component after another's loads; with
// one cell per lane 6.8 and 9.0.

// fdtd_calculations.cu:32-77
template <typename Q, bool ST>
__global__ __launch_bounds__(kBlock) void legacy_h(float *hx, float *hy, float *hz, const float *ex, const float *ey,
                                                   const float *ez)
{
    const LegacyParams &p = c_p;
    const Q nxy = (Q)p.nx * (Q)p.ny, q = blockIdx.x * (Q)kBlock + threadIdx.x;
    const int k0 = (int)(blockIdx.z * kPairs + blockIdx.y) * 2;
    if (q >= nxy || k0 >= p.nz) return;
    const int j = row_of(p, q), i = (int)(q - (Q)j * (Q)p.nx);
    const bool ip = i < p.nx - 1, jp = j < p.ny - 1;
    const Q qi = ip ? q + 1 : q, qj = jp ? q + (Q)p.nx : q;
    float hx0[2], hy0[2], hz0[2], x[3], y[3], z[2], xj[2], yi[2], zi[2], zj[2];
#pragma unroll
    for (int h = 0; h < 3; h++) {
        const size_t o = (size_t)min(k0 + h, p.nz - 1) * nxy;
        x[h] = ld(ex + o, q); y[h] = ld(ey + o, q);
        if (h < 2) {
            z[h] = ld(ez + o, q);
            hx0[h] = ld_own<ST>(hx + o, q); hy0[h] = ld_own<ST>(hy + o, q); hz0[h] = ld_own<ST>(hz + o, q);
            xj[h] = ld(ex + o, qj); yi[h] = ld(ey + o, qi); zi[h] = ld(ez + o, qi); zj[h] = ld(ez + o, qj);
        }
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int k = k0 + h;
        if (k >= p.nz - 1) break;   // no component of the last plane is updated
        const size_t o = (size_t)k * nxy;
        if (i >= 1 && ip && jp) st_own<ST>(hx + o, q, hx0[h] - p.chy * (zj[h] - z[h]) + p.chy * (y[h + 1] - y[h]));
        if (ip && j >= 1 && jp) st_own<ST>(hy + o, q, hy0[h] - p.chz * (x[h + 1] - x[h]) + p.chx * (zi[h] - z[h]));
        if (ip && jp && k >= 1) st_own<ST>(hz + o, q, hz0[h] - p.chx * (yi[h] - y[h]) + p.chy * (xj[h] - x[h]));
    }
}

// fdtd_calculations.cu:80-122
template <typename Q, bool ST>
__global__ __launch_bounds__(kBlock) void legacy_d(float *dxT, float *dyT, float *dzT, const float *dxS,
                                                   const float *dyS, const float *dzS, const float *hx,
                                                   const float *hy, const float *hz)
{
    const LegacyParams &p = c_p;
    const Q nxy = (Q)p.nx * (Q)p.ny, q = blockIdx.x * (Q)kBlock + threadIdx.x;
    const int k0 = (int)(blockIdx.z * kPairs + blockIdx.y) * 2;
    if (q >= nxy || k0 >= p.nz) return;
    const int j = row_of(p, q), i = (int)(q - (Q)j * (Q)p.nx);
    const bool ip = i < p.nx - 1, jp = j < p.ny - 1, i1 = i >= 1, j1 = j >= 1;
    const Q qi = i1 ? q - 1 : q, qj = j1 ? q - (Q)p.nx : q;
    float dx[2], dy[2], dz[2], x[3], y[3], z[2], xj[2], yi[2], zi[2], zj[2];   // x[h], y[h]: plane k0 + h - 1
#pragma unroll
    for (int h = -1; h < 2; h++) {
        const size_t o = (size_t)max(min(k0 + h, p.nz - 1), 0) * nxy;
        x[h + 1] = ld(hx + o, q); y[h + 1] = ld(hy + o, q);
        if (h >= 0) {
            z[h] = ld(hz + o, q);
            dx[h] = ld_own<ST>(dxS + o, q); dy[h] = ld_own<ST>(dyS + o, q); dz[h] = ld_own<ST>(dzS + o, q);
            xj[h] = ld(hx + o, qj); yi[h] = ld(hy + o, qi); zi[h] = ld(hz + o, qi); zj[h] = ld(hz + o, qj);
        }
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int k = k0 + h;
        if (k >= p.nz - 1) break;   // no component of the last plane is updated
        const bool k1 = k >= 1;
        const size_t o = (size_t)k * nxy;
        if (ip && j1 && jp && k1) st_own<ST>(dxT + o, q, dx[h] + p.cdy * (z[h] - zj[h]) - p.cdz * (y[h + 1] - y[h]));
        if (i1 && ip && jp && k1) st_own<ST>(dyT + o, q, dy[h] + p.cdz * (x[h + 1] - x[h]) - p.cdx * (z[h] - zi[h]));
        if (i1 && ip && j1 && jp) st_own<ST>(dzT + o, q, dz[h] + p.cdx * (y[h + 1] - yi[h]) - p.cdy * (x[h + 1] - xj[h]));
    }
}

// H and D where pairs of planes do not pay (use_pairs): one lane per cell of the
// flattened grid, each component's loads where it is updated only.
template <typename Q>
__global__ __launch_bounds__(kBlock) void legacy_h_flat(float *hx, float *hy, float *hz, const float *ex, const float *ey,
                                                        const float *ez)
{
    const LegacyParams &p = c_p;
    Q o;
    int i, j, k;
    if (!flat_cell(p, o, i, j, k) || k >= p.nz - 1) return;
    const Q sy = (Q)p.nx, sz = sy * (Q)p.ny;
    const bool ip = i < p.nx - 1, jp = j < p.ny - 1;
    if (i >= 1 && ip && jp) hx[o] = hx[o] - p.chy * (ez[o + sy] - ez[o]) + p.chy * (ey[o + sz] - ey[o]);
    if (ip && j >= 1 && jp) hy[o] = hy[o] - p.chz * (ex[o + sz] - ex[o]) + p.chx * (ez[o + 1] - ez[o]);
    if (ip && jp && k >= 1) hz[o] = hz[o] - p.chx * (ey[o + 1] - ey[o]) + p.chy * (ex[o + sy] - ex[o]);
}

template <typename Q>
__global__ __launch_bounds__(kBlock) void legacy_d_flat(float *dxT, float *dyT, float *dzT, const float *dxS,
                                                        const float *dyS, const float *dzS, const float *hx,
                                                        const float *hy, const float *hz)
{
    const LegacyParams &p = c_p;
    Q o;
    int i, j, k;
    if (!flat_cell(p, o, i, j, k) || k >= p.nz - 1) return;
    const Q sy = (Q)p.nx, sz = sy * (Q)p.ny;
    const bool ip = i < p.nx - 1, jp = j < p.ny - 1, i1 = i >= 1, j1 = j >= 1, k1 = k >= 1;
    if (ip && j1 && jp && k1) dxT[o] = dxS[o] + p.cdy * (hz[o] - hz[o - sy]) - p.cdz * (hy[o] - hy[o - sz]);
    if (i1 && ip && jp && k1) dyT[o] = dyS[o] + p.cdz * (hx[o] - hx[o - sz]) - p.cdx * (hz[o] - hz[o - 1]);
    if (i1 && ip && j1 && jp) dzT[o] = dzS[o] + p.cdx * (hy[o] - hy[o - 1]) - p.cdy * (hx[o] - hx[o - sy]);
}

// fdtd_calculations.cu:187-213: one lane per listed source.
__global__ void legacy_sources(float *dzT, const float *dzS, const float *hx, const float *hy, int it)
{
    const LegacyParams p = c_p;
    const int s = threadIdx.x;
    if (s >= p.nsrc) return;
    const int x = c_sources[3 * s], y = c_sources[3 * s + 1], z = c_sources[3 * s + 2];
    const long long o = ((long long)z * p.ny + y) * p.nx + x;
    const float jz = (it >= 0 && it < p.njz) ? c_jz[it] : 0.0f;
    const float val = dzS[o] + p.dt / p.dx * (hy[o] - hy[o - 1]) - p.dt / p.dy * (hx[o] - hx[o - p.nx]) - jz;
    dzT[o] = val;
}

__device__ inline float e_update(float c, float d, float a, double g1, double g2, double g3, float e0, float e1,
                                 float d0, float d1, float d2)
{
    // c * (d*E^n - a*E^{n-1} + g1*D^{n+1} - g2*D^n + g3*D^{n-1}): the first
    // two products and their difference in float, the rest in double.
    const float fe = d * e0 - a * e1;
    double s = (double)fe + g1 * (double)d0;
    s = s - g2 * (double)d1;
    s = s + g3 * (double)d2;
    return (float)((double)c * s);
}

// fdtd_calculations.cu:125-184
template <typename Q, bool ST>
__global__ __launch_bounds__(kBlock) void legacy_e(float *exT, float *eyT, float *ezT, const float *ex0,
                                                   const float *ey0, const float *ez0, const float *ex1,
                                                   const float *ey1, const float *ez1, const float *dx0,
                                                   const float *dy0, const float *dz0, const float *dx1,
                                                   const float *dy1, const float *dz1, const float *dx2,
                                                   const float *dy2, const float *dz2, const float *sigma,
                                                   const float *epsI, const float *epsS, const float *tauD)
{
    // one lane per cell of the flattened grid: every wave's 19 streams move whole lines whatever nx*ny is (14.6 us
    // at 100^3 with the lanes numbered from each plane's start, 13.6 so)
    const LegacyParams &p = c_p;
    Q o;
    int i, j, k;
    if (!flat_cell(p, o, i, j, k)) return;
    const bool ux = i < p.nx - 1 && j >= 1 && j < p.ny - 1 && k >= 1 && k < p.nz - 1;
    const bool uyz = i >= 1 && k >= 1;
    if (!ux && !uyz) return;
    auto v = [&](const float *a) { return ST ? __builtin_nontemporal_load(a + o) : a[o]; };
    const float sg = v(sigma), ei = v(epsI), es = v(epsS), tau = v(tauD);
    const float dt = p.dt, e0 = p.eps0;
    const float a = 2.0 * e0 * ei * tau;
    const float b = a + 2.0 * dt * (e0 * es + sg * tau);
    const float cc = 1.0 / (b + sg * dt * dt);
    const float d = (p.debye_mode == FDTD_DEBYE_REF) ? (float)(2.0 * b - sg * dt * dt)
                                                      : (float)((double)a + (double)b - (double)(sg * dt * dt));
    const double g1 = 2.0 * (dt + tau);
    const double g2 = 2.0 * dt + 4.0 * tau;
    const double g3 = 2.0 * tau;
    if (ux) st_own<ST>(exT, o, e_update(cc, d, a, g1, g2, g3, v(ex0), v(ex1), v(dx0), v(dx1), v(dx2)));
    if (uyz) {
        st_own<ST>(eyT, o, e_update(cc, d, a, g1, g2, g3, v(ey0), v(ey1), v(dy0), v(dy1), v(dy2)));
        st_own<ST>(ezT, o, e_update(cc, d, a, g1, g2, g3, v(ez0), v(ez1), v(dz0), v(dz1), v(dz2)));
    }
}

inline int set_err(hipError_t e) { return (int)e; }

}  // namespace

// Streaming operands where the 25 arrays of the reference's FdtdField are well
// past the Infinity Cache.  us of H, D and E together, cached and streaming:
// 140^3 (274 MB) 76, 80; 145^3 (305) 91, 100; 155^3 (372) 112, 120; 16x500x500 (400)
// 114, 118; 500x16x500 (400) 108, 106; 160^3 (410) 113, 111; 400x32x400 (512) 150,
// 136; 200^3 (800) 242, 209.  256^3 H 123, 95, D 132, 99, E 276, 248.
static inline bool streaming() { return 100LL * h_p.nx * h_p.ny * h_p.nz > 400000000; }
static inline bool wide() { return (long long)h_p.nx * h_p.ny * h_p.nz >= (1LL << 32); }

extern "C" int fdtdSetDebyeMode(int mode)
{
    if (mode != FDTD_DEBYE_REF && mode != FDTD_DEBYE_FIXED) return FDTD_EINVAL;
    h_p.debye_mode = mode;
    if (h_params_set) return set_err(hipMemcpyToSymbol(HIP_SYMBOL(c_p), &h_p, sizeof(h_p)));
    return 0;
}

extern "C" int copySymbolsToDevice(FdtdParams *params)
{
    if (!params || params->nx < 2 || params->ny < 2 || params->nz < 2) return FDTD_EINVAL;
    const long long n = (long long)params->nx * params->ny * params->nz;
    if (n >= (1LL << 40)) return FDTD_ERANGE;
    h_p.nx = params->nx; h_p.ny = params->ny; h_p.nz = params->nz;
    h_p.dt = params->dt; h_p.dx = params->dx; h_p.dy = params->dy; h_p.dz = params->dz;
    h_p.mu0 = params->mu0; h_p.eps0 = params->eps0;
    h_p.chx = h_p.dt / (h_p.mu0 * h_p.dx); h_p.chy = h_p.dt / (h_p.mu0 * h_p.dy); h_p.chz = h_p.dt / (h_p.mu0 * h_p.dz);
    h_p.cdx = h_p.dt / h_p.dx; h_p.cdy = h_p.dt / h_p.dy; h_p.cdz = h_p.dt / h_p.dz;
    div_consts(h_p.nx, h_p.nx_mul, h_p.nx_shift);
    if (!wide()) div_consts((unsigned long long)h_p.nx * h_p.ny, h_p.nxy_mul, h_p.nxy_shift);
    const int ns = std::max(0, std::min(D_MAX_SOURCES, params->sourcesCount));
    const int nj = std::max(0, std::min(D_MAX_JZ, params->jzCount));
    for (int s = 0; s < ns; s++)
        for (int q = 0; q < 3; q++) {
            const int v = params->sources[3 * s + q];
            const int lim = q == 0 ? params->nx : (q == 1 ? params->ny : params->nz);
            // the source kernel reads x-1 and y-1
            if (v < (q < 2 ? 1 : 0) || v >= lim) return FDTD_ERANGE;
        }
    h_p.nsrc = ns;
    h_p.njz = params->jz ? nj : 0;
    hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_p), &h_p, sizeof(h_p));
    if (e == hipSuccess && ns > 0) e = hipMemcpyToSymbol(HIP_SYMBOL(c_sources), params->sources, sizeof(int) * 3 * ns);
    if (e == hipSuccess && h_p.njz > 0) e = hipMemcpyToSymbol(HIP_SYMBOL(c_jz), params->jz, sizeof(float) * h_p.njz);
    if (e == hipSuccess) h_params_set = true;
    return set_err(e);
}

static inline dim3 flat_grid()
{
    const long long n = (long long)h_p.nx * h_p.ny * h_p.nz;
    return dim3((unsigned)((n + kBlock - 1) / kBlock));
}

// H and D by pairs of planes, except in grids whose cells all are resident at
// once as lanes (2048 blocks on 256 CUs), where half the waves bring half the loads
// in flight, in thin grids, where most cells lie beside a face and the pairs' loads
// are for updates that are masked, and where the plane and the planes' number
// leave many lanes of the pairs' blocks idle.  us of H, D
// and E together, flat against pairs: 500x1000x2 15.3, 20.0; 500x500x4 22.3,
// 25.5; 400x400x6 25.7, 26.4; 300x400x8 27.2, 27.3; 300x350x9 29.3, 29.0; 500x3x700
// 26.0, 29.6; 400x5x500 25.7, 28.6; 400x7x350 28.8, 28.9; 2x500x1000 26.0, 28.5;
// 3x500x700 37.5, 34.7; filled to 0.10 (5x5x20000) 16.6, 23.3; 0.39 (10x10x5000)
// 17.3, 18.5; 0.63 (18x18x3000) 31.9, 33.1; 0.77 (14x14x5000) 31.4, 29.4; 66^3
// 12.8, 14.3; 732x29x16 12.6, 14.2; 80^3 (2000 blocks) 17.3, 17.8; 82^3 (2154) 22.1,
// 20.8; 100^3 31.6, 28.4.
static inline bool use_pairs()
{
    const long long n = (long long)h_p.nx * h_p.ny, blocks = (n + kBlock - 1) / kBlock, pairs = h_p.nz / 2 + h_p.nz % 2;
    return n * h_p.nz > 2048 * kBlock && h_p.nx >= 3 && h_p.ny >= 7 && h_p.nz >= 8 &&
           (double)n * h_p.nz >= 0.65 * (2.0 * kBlock) * blocks * pairs;
}

static inline dim3 pair_grid()
{
    const long long n = (long long)h_p.nx * h_p.ny;
    const int pairs = h_p.nz / 2 + h_p.nz % 2;
    return dim3((unsigned)((n + kBlock - 1) / kBlock), (unsigned)std::min(pairs, kPairs),
                (unsigned)((pairs + kPairs - 1) / kPairs));
}

extern "C" int updateHField(float *hx, float *hy, float *hz, float *exSource, float *eySource, float *ezSource,
                            hipStream_t stream)
{
    if (!h_params_set) return FDTD_ESTATE;
    if (use_pairs())
        (wide() ? legacy_h<size_t, true> : streaming() ? legacy_h<uint32_t, true> : legacy_h<uint32_t, false>)
            <<<pair_grid(), kBlock, 0, stream>>>(hx, hy, hz, exSource, eySource, ezSource);
    else
        (wide() ? legacy_h_flat<size_t> : legacy_h_flat<uint32_t>)
            <<<flat_grid(), kBlock, 0, stream>>>(hx, hy, hz, exSource, eySource, ezSource);
    return set_err(hipGetLastError());
}

extern "C" int updateDField(float *dxTarget, float *dyTarget, float *dzTarget, float *dxSource, float *dySource,
                            float *dzSource, float *hx, float *hy, float *hz, hipStream_t stream)
{
    if (!h_params_set) return FDTD_ESTATE;
    if (use_pairs())
        (wide() ? legacy_d<size_t, true> : streaming() ? legacy_d<uint32_t, true> : legacy_d<uint32_t, false>)
            <<<pair_grid(), kBlock, 0, stream>>>(dxTarget, dyTarget, dzTarget, dxSource, dySource, dzSource, hx, hy, hz);
    else
        (wide() ? legacy_d_flat<size_t> : legacy_d_flat<uint32_t>)
            <<<flat_grid(), kBlock, 0, stream>>>(dxTarget, dyTarget, dzTarget, dxSource, dySource, dzSource, hx, hy, hz);
    return set_err(hipGetLastError());
}

extern "C" int updateEField(float *exTarget, float *eyTarget, float *ezTarget, float *exSource0, float *eySource0,
                            float *ezSource0, float *exSource1, float *eySource1, float *ezSource1, float *dxSource0,
                            float *dySource0, float *dzSource0, float *dxSource1, float *dySource1, float *dzSource1,
                            float *dxSource2, float *dySource2, float *dzSource2, float *sigma, float *epsI,
                            float *epsS, float *tauD, hipStream_t stream)
{
    if (!h_params_set) return FDTD_ESTATE;
    (wide() ? legacy_e<size_t, true> : streaming() ? legacy_e<uint32_t, true> : legacy_e<uint32_t, false>)
        <<<flat_grid(), kBlock, 0, stream>>>(exTarget, eyTarget, ezTarget, exSource0, eySource0, ezSource0, exSource1,
                                             eySource1, ezSource1, dxSource0, dySource0, dzSource0, dxSource1,
                                             dySource1, dzSource1, dxSource2, dySource2, dzSource2, sigma, epsI, epsS,
                                             tauD);
    return set_err(hipGetLastError());
}

extern "C" int updateSources(float *dzTarget, float *dzSource, float *hx, float *hy, int currIteration,
                             hipStream_t stream)
{
    if (!h_params_set) return FDTD_ESTATE;
    if (h_p.nsrc == 0) return 0;
    legacy_sources<<<1, 64, 0, stream>>>(dzTarget, dzSource, hx, hy, currIteration);
    return set_err(hipGetLastError());
}

extern "C" int updateMurBoundary(float *exTarget, float *eyTarget, float *ezTarget, float *exSource,
                                 float *eySource, float *ezSource, float *rpx0, float *rpy0, float *rpz0,
                                 float *rpxEnd, float *rpyEnd, float *rpzEnd, hipStream_t stream)
{
    if (!h_params_set) return FDTD_ESTATE;
    MurArgs m;
    m.exT = exTarget; m.eyT = eyTarget; m.ezT = ezTarget;
    m.exS = exSource; m.eyS = eySource; m.ezS = ezSource;
    m.rpx0 = rpx0; m.rpy0 = rpy0; m.rpz0 = rpz0; m.rpxEnd = rpxEnd; m.rpyEnd = rpyEnd; m.rpzEnd = rpzEnd;
    m.nx = h_p.nx; m.ny = h_p.ny; m.nz = h_p.nz; m.pitch = h_p.nx; m.plane = (long long)h_p.nx * h_p.ny;
    m.dt = h_p.dt; m.hx = h_p.dx; m.hy = h_p.dy; m.hz = h_p.dz; m.mu0 = h_p.mu0; m.eps0 = h_p.eps0;
    mur_segments(h_p.nx, h_p.ny, h_p.nz, m.seg_start);
    return set_err(launch_mur(m, kStoreF32, stream));
}
