// cell_step: one time step of a grid in one launch, one cell per lane and no
// z-march.  A tiled launch (fused_step) of a grid in the 256 MB Infinity Cache
// is bound by the latency of its blocks' marches, not by bytes: at 64^3 it
// runs 256 blocks for 16 us.
//
// A lane computes its cell's H^{n+1/2}, D^{n+1} (with the source) and
// E^{n+1} from loads that depend on nothing but the cell's index: the six
// halo H values that curl H needs (at i-1, j-1, k-1) are recomputed from
// H^{n-1/2} and E^n, operation for operation as fused_tile does, so the two
// kernels give identical results.  All loads of a wave go out together;
// there is no LDS and no barrier.
//
// Forms, by the size of the state (cell_form):
//   * near, in the Infinity Cache: all loads and stores cached, as the next
//     step reads what this one wrote, and streaming stores would send it to
//     HBM (128^3 fp32: 38 us with them, 30 us without);
//   * mid: the lanes take their neighbours along x from each other.  In a near
//     grid the eleven loads of them cost nothing; here they hit lines that are
//     still on their way from HBM, and hold up the vector cache.  The values
//     past a row's ends come through the scalar cache;
//   * part (16 bits): and D streams past the Infinity Cache, which holds E and H;
//   * far: and so do E^{n-1} and the stores of E; H and E^n stay for longer.
// Every other step takes the planes from the highest down (flip): it starts
// on those that the last step left in the cache.
//
// The first-order Mur faces and the probe row are part of the same launch:
//   * a face cell's new E needs E^{n+1} of its inward neighbour, E^n of both
//     and nothing else, all of which the lane of that neighbour holds.  So
//     the lanes at i = 1, i = nx-2, j = 1, ... store the face cells beside
//     them, and a face cell's own lane does not store the components that a
//     face segment covers (the segments are disjoint per component, and no
//     segment writes a cell that another one reads at n+1);
//   * a probe is one wave that evaluates the cell again (for an E cell on a
//     face: its neighbour) and, instead of storing, writes the value asked
//     for, so it waits for no other wave.
//
// Measured on MI355X, whole steps, against fused_step and the Mur launch
// (us): fp32 32^3 4.8 (14.7), 64^3 7.2 (16.6), 100^3 18.9 (31.2), 128^3 30
// (47), 160x160x100 34 (60), 151x138x188 75 (83), 256^3 285 (304); fp16 64^3
// 6.8 (18.0), 96x121x77 13.0 (27.6), 256^3 181 (206), 320x320x300 318 (377).
// 128^3 moves 180 MB, 6.4 TB/s at the L2's far side, where a stream of the same
// arrays reaches 8.0; with 4 waves a SIMD instead of 7 it takes as long.  Past
// the cache fp32 waits for HBM (85 bytes a cell at 5.0 TB/s at 320x320x224;
// occupancy again makes no difference).  16-bit grids are held by the waves in
// flight: 8 a SIMD, the most there are, take 186 us at 256^3, 6 take 225.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "fdtd_device.h"
#include "fdtd_internal.h"

namespace {

constexpr int kCoefBlock = 256;

// The Mur segment (numbered as in mur_segments) that writes E component c at
// (i, j, k), and the step towards the cell whose lane evaluates it; -1: none.
__device__ __forceinline__ int face_of(int c, int i, int j, int k, int nx, int ny, int nz, int &di, int &dj, int &dk)
{
    const bool ii = i >= 1 && i < nx - 1, ji = j >= 1 && j < ny - 1, ki = k >= 1 && k < nz - 1;
    const bool il = i < nx - 1, jl = j < ny - 1, kl = k < nz - 1;
    di = dj = dk = 0;
    const int ex = i == 0 ? 0 : (i == nx - 1 ? 1 : -1), ey = j == 0 ? 0 : (j == ny - 1 ? 1 : -1),
              ez = k == 0 ? 0 : (k == nz - 1 ? 1 : -1);
    if (c == 0 && il) {
        if (ey >= 0 && ki) { dj = 1 - 2 * ey; return ey; }
        if (ez >= 0 && ji) { dk = 1 - 2 * ez; return 2 + ez; }
    } else if (c == 1 && jl) {
        if (ex >= 0 && ki) { di = 1 - 2 * ex; return 4 + ex; }
        if (ez >= 0 && ii) { dk = 1 - 2 * ez; return 6 + ez; }
    } else if (c == 2 && kl) {
        if (ex >= 0 && ji) { di = 1 - 2 * ex; return 8 + ex; }
        if (ey >= 0 && ii) { dj = 1 - 2 * ey; return 10 + ey; }
    }
    return -1;
}

// One load per value, never merged with its neighbours' (a wavefront-scope
// relaxed load is an ordinary cached load that the compiler does not widen):
// a dword, byte or short load of a wave takes 4.8 cycles of the CU's address
// unit, an 8- or 12-byte one 16.5, so two or three dword loads are cheaper.
template <typename T>
__device__ __forceinline__ float at(const char *p, uint32_t b, int d = 0)
{
    if constexpr (sizeof(T) == 4)
        return __hip_atomic_load((const float *)(p + b) + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    else
        return Elem<T>::cvt(__hip_atomic_load((const unsigned short *)(p + b) + d, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_WAVEFRONT));
}

template <typename V> using Const = const __attribute__((address_space(4))) V;

// The element at a wave-uniform offset, through the scalar cache: its own path
// beside the vector loads'.  Only for arrays that the launch does not write.
template <typename T>
__device__ __forceinline__ float at_uniform(const char *p, uint32_t b)
{
    if constexpr (sizeof(T) == 4) {
        return *(Const<float> *)(p + b);
    } else {
        const uintptr_t q = (uintptr_t)(p + b);
        return Elem<T>::cvt((unsigned short)(*(Const<uint32_t> *)(q & ~(uintptr_t)3) >> ((q & 2) * 8)));
    }
}

// The value of the lane below (above) in a wave's row of 1 << BXL lanes; the
// first (last) lane of the row gets `end`, in the wave's second row `end1`.
template <int BXL>
__device__ __forceinline__ float lane_below(float v, float end, float end1)
{
    const float r = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(end), __float_as_int(v), 0x138, 0xf, 0xf, false));
    return BXL < 6 && (threadIdx.x & 63) == 32 ? end1 : r;
}
template <int BXL>
__device__ __forceinline__ float lane_above(float v, float end, float end1)
{
    const float r = __int_as_float(
        __builtin_amdgcn_update_dpp(__float_as_int(BXL < 6 ? end1 : end), __float_as_int(v), 0x130, 0xf, 0xf, false));
    return BXL < 6 && (threadIdx.x & 63) == 31 ? end : r;
}

// A value that the next step does not read soon enough to find it in the
// Infinity Cache (NT): a streaming load.
template <typename T, bool NT>
__device__ __forceinline__ float at_once(const char *p, uint32_t b)
{
    if constexpr (NT) return Elem<T>::ld_nt((const T *)p, b);
    else return at<T>(p, b);
}

// A Mur face's new value q * x as storage type T holds it; `once` says which
// of the two roundings the tiled step gives this face.
template <typename T>
__device__ __forceinline__ float mur_round(float q, float x, bool once)
{
    if constexpr (std::is_same<T, __half>::value)
        if (once) return mur_once<T>(q, x);
    return Elem<T>::rnd(mur_twice<T>(q, x));
}

// The Mur coefficients of a face cell (launch_mur_coefs).
__device__ __forceinline__ float4 mur_coef(float dt, float h, float m0, float e0, float rpf, float rpn)
{
    const float sf = sqrtf(m0 * e0 * rpf), sn = sqrtf(m0 * e0 * rpn);
    float4 c;
    c.x = 1 / (dt + h * sf);
    c.y = dt - h * sn;
    c.z = dt + h * sn;
    c.w = dt - h * sf;
    return c;
}

// The operands of one grid's step from kernel arguments.
struct OneStep {
    const CellArgs &a;
    __device__ __forceinline__ int nx() const { return a.nx; }
    __device__ __forceinline__ int ny() const { return a.ny; }
    __device__ __forceinline__ int nz() const { return a.nz; }
    __device__ __forceinline__ uint32_t o0() const { return a.o0; }
    __device__ __forceinline__ uint32_t sy() const { return a.sy; }
    __device__ __forceinline__ uint32_t sz() const { return a.sz; }
    __device__ __forceinline__ int tiles_x() const { return a.tiles_x; }
    __device__ __forceinline__ int tiles() const { return a.tiles; }
    __device__ __forceinline__ int run() const { return a.run; }
    __device__ __forceinline__ int gx() const { return a.gx; }
    __device__ __forceinline__ uint32_t tx_mul() const { return a.tx_mul; }
    __device__ __forceinline__ uint32_t tx_shift() const { return a.tx_shift; }
    __device__ __forceinline__ const uint8_t * ids() const { return a.ids; }
    __device__ __forceinline__ const MatCoef * lut() const { return a.lut; }
    __device__ __forceinline__ float ch(int q) const { return a.ch[q]; }
    __device__ __forceinline__ float cd(int q) const { return a.cd[q]; }
    __device__ __forceinline__ ZeroTerms zmask() const { return a.zmask; }
    __device__ __forceinline__ int hi_once() const { return a.hi_once; }
    __device__ __forceinline__ int flip() const { return a.flip; }
    __device__ __forceinline__ const char * e0(int q) const { return a.e0[q]; }
    __device__ __forceinline__ const char * e1(int q) const { return a.e1[q]; }
    __device__ __forceinline__ const char * d0(int q) const { return a.d0[q]; }
    __device__ __forceinline__ const char * d1(int q) const { return a.d1[q]; }
    __device__ __forceinline__ const char * h0(int q) const { return a.h0[q]; }
    __device__ __forceinline__ char * eT(int q) const { return a.eT[q]; }
    __device__ __forceinline__ char * dT(int q) const { return a.dT[q]; }
    __device__ __forceinline__ char * h1(int q) const { return a.h1[q]; }
    __device__ __forceinline__ float jz() const { return a.jz; }
    __device__ __forceinline__ int nprobe() const { return a.p.nprobe; }
    __device__ __forceinline__ const int * probes() const { return a.p.probes; }
    // coefficients of the face (0, 1: x low, high; 2, 3: y; 4, 5: z) beside cell (i, j, k)
    __device__ __forceinline__ float4 coef(int f, int i, int j, int k) const
    {
        const long long c = f < 2 ? (long long)k * a.ny + j : f < 4 ? (long long)k * a.nx + i : (long long)j * a.nx + i;
        const float4 *p = f == 0 ? a.mur[0] : f == 1 ? a.mur[1] : f == 2 ? a.mur[2] : f == 3 ? a.mur[3] : f == 4 ? a.mur[4] : a.mur[5];
        return p[c];
    }
    __device__ __forceinline__ void record(int probe, int field, float v) const
    {
        a.p.out[(long long)a.p.row * a.p.nprobe + probe] = (double)v * a.p.factor[field];
    }
};

// The same of a batch's grid at its step n, from its descriptor: the ring
// slot and H buffer roles follow n as a single grid's do.  The y and z faces'
// coefficients come from the rp planes (a batch keeps no table of them).
struct BatchStep {
    Const<CellInst> *d;
    int s0, s1, sT, hb;     // slots of levels n, n-1, n+1; buffer of H^{n-1/2}
    int n;
    __device__ __forceinline__ int nx() const { return d->nx; }
    __device__ __forceinline__ int ny() const { return d->ny; }
    __device__ __forceinline__ int nz() const { return d->nz; }
    __device__ __forceinline__ uint32_t o0() const { return d->o0; }
    __device__ __forceinline__ uint32_t sy() const { return d->sy; }
    __device__ __forceinline__ uint32_t sz() const { return d->sz; }
    __device__ __forceinline__ int tiles_x() const { return d->tiles_x; }
    __device__ __forceinline__ int tiles() const { return d->tiles; }
    __device__ __forceinline__ int run() const { return d->run; }
    __device__ __forceinline__ int gx() const { return d->gx; }
    __device__ __forceinline__ uint32_t tx_mul() const { return d->tx_mul; }
    __device__ __forceinline__ uint32_t tx_shift() const { return d->tx_shift; }
    __device__ __forceinline__ const uint8_t * ids() const { return d->ids; }
    __device__ __forceinline__ const MatCoef * lut() const { return d->lut; }
    __device__ __forceinline__ float ch(int q) const { return d->ch[q]; }
    __device__ __forceinline__ float cd(int q) const { return d->cd[q]; }
    __device__ __forceinline__ ZeroTerms zmask() const { return {{d->zmask.w[0], d->zmask.w[1], d->zmask.w[2], d->zmask.w[3]}}; }
    __device__ __forceinline__ int hi_once() const { return d->hi_once; }
    __device__ __forceinline__ int flip() const { return n & 1; }
    __device__ __forceinline__ const char * e0(int q) const { return d->E[s0][q]; }
    __device__ __forceinline__ const char * e1(int q) const { return d->E[s1][q]; }
    __device__ __forceinline__ const char * d0(int q) const { return d->D[s0][q]; }
    __device__ __forceinline__ const char * d1(int q) const { return d->D[s1][q]; }
    __device__ __forceinline__ const char * h0(int q) const { return d->H[hb][q]; }
    __device__ __forceinline__ char * eT(int q) const { return d->E[sT][q]; }
    __device__ __forceinline__ char * dT(int q) const { return d->D[sT][q]; }
    __device__ __forceinline__ char * h1(int q) const { return d->H[hb ^ 1][q]; }
    __device__ __forceinline__ int nprobe() const { return d->nprobe; }
    __device__ __forceinline__ const int * probes() const { return d->probes; }
    __device__ __forceinline__ float jz() const
    {
        const int t = d->jz_hold3 ? (n / 3) * 3 : n;
        return t < d->jz_len ? ((Const<float> *)d->jz)[t] : 0.0f;
    }
    __device__ __forceinline__ float4 coef(int f, int i, int j, int k) const
    {
        if (f < 2) return (f == 0 ? d->murx0 : d->murx1)[(long long)k * d->ny + j];
        // the pair of cells in the reference's planes y (k, 2, i) and z (2, j, i); low faces: the first is the face
        const long long step = f < 4 ? d->nx : (long long)d->nx * d->ny;
        const long long at = f < 4 ? (long long)k * 2 * d->nx + i : (long long)j * d->nx + i;
        const float *rp = f == 2 ? d->rp[1] : f == 3 ? d->rp[4] : f == 4 ? d->rp[2] : d->rp[5];
        const float r0 = rp[at], r1 = rp[at + step];
        return mur_coef(d->dt, f < 4 ? d->h[1] : d->h[2], d->mu0, d->eps0, f & 1 ? r1 : r0, f & 1 ? r0 : r1);
    }
    __device__ __forceinline__ void record(int probe, int field, float v) const
    {
        if (n < d->probe_rows) d->probe_out[(long long)n * d->nprobe + probe] = (double)v * d->factor[field];
    }
};

// What a lane loads: the cell's operands and its neighbours'.  Suffixes: im,
// ip at i-1, i+1 and so on; no suffix: the cell.
struct Ops {
    float ex, ey, ez, ex_im, ey_im, ez_im, ey_ip, ez_ip, ex_jp, ez_jp, ex_jp_im, ex_jm, ey_jm, ez_jm, ey_jm_ip;
    float ex_kp, ey_kp, ex_kp_im, ey_kp_jm, ex_km, ey_km, ez_km, ez_km_ip, ez_km_jp;
    float hx, hy, hz, hy_im, hz_im, hx_jm, hz_jm, hx_km, hy_km;
    float dx, dy, dz;                        // D^n
    float exm, eym, ezm, dxm, dym, dzm;      // E^{n-1}, D^{n-1}
    float a, c, d, k1, k2, k3, k5;
    double g1, g2, g3;
    bool src;
};

// One block's cells (or, past the planes, its probes) of a grid's step.
// BXL: log2 of the lanes of a block along x (32 or 64); the other lanes of its
// cell_block_lanes are rows.  Exact form: cells whose material has a = g3 = +0 (zmask) do not
// load E^{n-1} and D^{n-1}, as fused_tile's zero-term rows, decided per lane;
// a grid that always loads them has an empty zmask.  C: where the step's operands
// are (OneStep, BatchStep); block bx of the C.gx() of plane bz.
template <typename T, bool EXACT, int BXL, int FORM, typename G>
__device__ __forceinline__ void cell_block(const G &C, int bx, int bz)
{
    using X = Elem<T>;
    constexpr uint32_t ES = sizeof(T);
    constexpr int LB = cell_block_lanes(FORM, sizeof(T), BXL);
    constexpr int BX = 1 << BXL, BY = LB / BX, WY = 64 / BX;
    constexpr bool LANES = FORM != kCellNear, ND = FORM >= kCellPart, NE = FORM == kCellFar;
    const int nx = C.nx(), ny = C.ny(), nz = C.nz();

    // Blocks (bx, k) of plane k in 8 runs of tiles, one run per XCD (workgroups
    // go to the XCDs round-robin by id, and a plane takes a multiple of 8, or in
    // grids of many small planes one block per tile: cell_tiles), so a
    // tile's neighbours in the plane and the same tiles of the planes around it
    // share its L2.  Rows past nz hold the probes.
    int i, j, k;
    int i0, jw;                              // the wave's first column and row
    bool deep = false, edge = false;
    int probe = -1, pf = -1, pseg = -1;      // probe: its index, field and face segment
    if (bz < nz) {
        const int t = cell_tile(bx, C.run());
        if (t >= C.tiles()) return;
        const int ty = cell_tile_row(t, C.tiles_x(), C.tx_mul(), C.tx_shift()), tx = t - ty * C.tiles_x();
        const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), l = (int)threadIdx.x & 63;
        jw = ty * BY + w * WY;
        if (jw >= ny) return;
        i0 = tx * BX;
        i = i0 + (l & (BX - 1));
        j = BX >= 64 ? jw : jw + (l >> BXL);
        k = C.flip() ? nz - 1 - bz : bz;
        if (i >= nx || j >= ny) return;
        deep = jw >= 2 && jw + WY <= ny - 2 && k >= 2 && k < nz - 2 && nx > 3;
        edge = tx == 0 || (nx - 2 >= tx * BX && nx - 2 < tx * BX + BX);
    } else {
        probe = __builtin_amdgcn_readfirstlane(((bz - nz) * C.gx() + bx) * (LB / 64) +
                                               ((int)threadIdx.x >> 6));
        if (probe >= C.nprobe()) return;
        const int *q = C.probes() + 4 * probe;
        pf = q[0]; i = q[1]; j = q[2]; k = q[3];
        if (pf >= 6) {
            int di, dj, dk;
            pseg = face_of(pf - 6, i, j, k, nx, ny, nz, di, dj, dk);
            i += di; j += dj; k += dk;
        }
        // lane 1 holds the cell, the lanes beside it its neighbours along x
        i0 = i - 1;
        jw = j;
        i = min(max(i0 + min((int)threadIdx.x & 63, 2), 0), nx - 1);
    }

    // deep: the wave's rows and plane are at least two cells inside the y and z faces, so that of the faces only
    // those along x are near (edge: its tile holds i = 1 or nx-2)
    // Byte offset of the cell from bases that lie `guard` elements before the arrays' origins.
    const uint32_t syb = C.sy(), szb = C.sz();
    const uint32_t o = C.o0() + (uint32_t)k * szb + (uint32_t)j * syb + (uint32_t)i * ES;
    const uint32_t ojp = o + syb, ojm = o - syb, okp = o + szb, okm = o - szb;
    const uint32_t id = C.ids()[o / ES];
    Ops v;
    const char *px = C.e0(0), *py = C.e0(1), *pz = C.e0(2), *qx = C.h0(0), *qy = C.h0(1), *qz = C.h0(2);
    v.ex = at<T>(px, o); v.ey = at<T>(py, o); v.ez = at<T>(pz, o);
    v.ex_jp = at<T>(px, ojp); v.ez_jp = at<T>(pz, ojp);
    v.ex_jm = at<T>(px, ojm); v.ey_jm = at<T>(py, ojm); v.ez_jm = at<T>(pz, ojm);
    v.ex_kp = at<T>(px, okp); v.ey_kp = at<T>(py, okp);
    v.ey_kp_jm = at<T>(py, okp - syb);
    v.ex_km = at<T>(px, okm); v.ey_km = at<T>(py, okm); v.ez_km = at<T>(pz, okm);
    v.ez_km_jp = at<T>(pz, okm + syb);
    v.hx = at<T>(qx, o); v.hy = at<T>(qy, o); v.hz = at<T>(qz, o);
    v.hx_jm = at<T>(qx, ojm); v.hz_jm = at<T>(qz, ojm);
    v.hx_km = at<T>(qx, okm); v.hy_km = at<T>(qy, okm);
    // Neighbours along x: near, loads of their own; else from the lanes beside
    // (below), and past the wave's ends from these.
    float end[2][11] = {};
    if constexpr (LANES) {
        const uint32_t first = C.o0() + (uint32_t)k * szb + (uint32_t)((i0 - 1) * (int)ES);
#pragma unroll
        for (int r = 0; r < (BXL < 6 ? 2 : 1); r++) {
            const uint32_t lo = first + (uint32_t)min(jw + r, ny - 1) * syb, hi = lo + (BX + 1) * ES;
            float *e = end[r];
            e[0] = at_uniform<T>(px, lo); e[1] = at_uniform<T>(py, lo); e[2] = at_uniform<T>(pz, lo);
            e[3] = at_uniform<T>(py, hi); e[4] = at_uniform<T>(pz, hi);
            e[5] = at_uniform<T>(px, lo + syb); e[6] = at_uniform<T>(py, hi - syb);
            e[7] = at_uniform<T>(px, lo + szb); e[8] = at_uniform<T>(pz, hi - szb);
            e[9] = at_uniform<T>(qy, lo); e[10] = at_uniform<T>(qz, lo);
        }
    }
    if constexpr (!LANES) {
        v.ex_im = at<T>(px, o, -1); v.ey_im = at<T>(py, o, -1); v.ez_im = at<T>(pz, o, -1);
        v.ey_ip = at<T>(py, o, 1); v.ez_ip = at<T>(pz, o, 1);
        v.ex_jp_im = at<T>(px, ojp, -1); v.ey_jm_ip = at<T>(py, ojm, 1);
        v.ex_kp_im = at<T>(px, okp, -1); v.ez_km_ip = at<T>(pz, okm, 1);
        v.hy_im = at<T>(qy, o, -1); v.hz_im = at<T>(qz, o, -1);
    }
    v.dx = at_once<T, ND>(C.d0(0), o); v.dy = at_once<T, ND>(C.d0(1), o); v.dz = at_once<T, ND>(C.d0(2), o);
    float4 mc = {0.0f, 0.0f, 0.0f, 0.0f};
    if (deep && edge && (i == 1 || i == nx - 2)) mc = C.coef(i == 1 ? 0 : 1, i, j, k);
    const uint32_t m = id & kMaterialMask;
    v.src = (id & kSourceBit) != 0;
    const char *lut = (const char *)C.lut() + m * (uint32_t)sizeof(MatCoef);
    if constexpr (EXACT) {
        const MatCoef *q = (const MatCoef *)lut;
        v.a = q->a; v.c = q->c; v.d = q->d;
        v.g1 = q->g1; v.g2 = q->g2; v.g3 = q->g3;
    } else {
        const MatCoef *q = (const MatCoef *)lut;
        v.k1 = q->k1; v.k2 = q->k2; v.k3 = q->k3; v.k5 = q->k5;
    }
    bool need = true;
    if constexpr (EXACT) need = !C.zmask().has(m);
    v.exm = v.eym = v.ezm = v.dxm = v.dym = v.dzm = 0.0f;
    if (need) {
        v.exm = at_once<T, NE>(C.e1(0), o); v.eym = at_once<T, NE>(C.e1(1), o); v.ezm = at_once<T, NE>(C.e1(2), o);
        v.dxm = at_once<T, ND>(C.d1(0), o); v.dym = at_once<T, ND>(C.d1(1), o); v.dzm = at_once<T, ND>(C.d1(2), o);
    }
    if constexpr (LANES) {   // (after the loads above are out: each of these waits for its operand)
        auto below = [&](float x, int q) { return lane_below<BXL>(x, end[0][q], end[1][q]); };
        auto above = [&](float x, int q) { return lane_above<BXL>(x, end[0][q], end[1][q]); };
        v.ex_im = below(v.ex, 0); v.ey_im = below(v.ey, 1); v.ez_im = below(v.ez, 2);
        v.ey_ip = above(v.ey, 3); v.ez_ip = above(v.ez, 4);
        v.ex_jp_im = below(v.ex_jp, 5); v.ey_jm_ip = above(v.ey_jm, 6);
        v.ex_kp_im = below(v.ex_kp, 7); v.ez_km_ip = above(v.ez_km, 8);
        v.hy_im = below(v.hy, 9); v.hz_im = below(v.hz, 10);
    }

    const float chx = C.ch(0), chy = C.ch(1), chz = C.ch(2);
    const float cdx = C.cd(0), cdy = C.cd(1), cdz = C.cd(2);
    auto up_x = [&](float h, float z, float zjp, float y, float ykp) { return h - chy * (zjp - z) + chy * (ykp - y); };
    auto up_y = [&](float h, float x, float xkp, float z, float zip) { return h - chz * (xkp - x) + chx * (zip - z); };
    auto up_z = [&](float h, float y, float yip, float x, float xjp) { return h - chx * (yip - y) + chy * (xjp - x); };
    auto st = [&](char *p, uint32_t b, float x) { X::st((T *)p, b, x); };
    auto st_d = [&](char *p, uint32_t b, float x) {
        if constexpr (ND) X::st_nt((T *)p, b, x);
        else X::st((T *)p, b, x);
    };
    auto st_e = [&](char *p, uint32_t b, float x) {
        if constexpr (NE) X::st_nt((T *)p, b, x);
        else X::st((T *)p, b, x);
    };
    auto ld = [&](const char *p, uint32_t b) { return X::ld((const T *)p, b); };

    const bool kh = k < nz - 1, kz = k >= 1 && kh;
    const bool jl = j < ny - 1, ji = j >= 1 && jl;
    const bool il = i < nx - 1, ii = i >= 1 && il;
    const float hx = (ii && jl && kh) ? up_x(v.hx, v.ez, v.ez_jp, v.ey, v.ey_kp) : v.hx;
    const float hy = (il && ji && kh) ? up_y(v.hy, v.ex, v.ex_kp, v.ez, v.ez_ip) : v.hy;
    const float hz = (il && jl && kz) ? up_z(v.hz, v.ey, v.ey_ip, v.ex, v.ex_jp) : v.hz;
    // H^{n+1/2} at j-1, i-1 and k-1 (used only where that cell exists)
    const float hx_jm = (ii && kh) ? up_x(v.hx_jm, v.ez_jm, v.ez, v.ey_jm, v.ey_kp_jm) : v.hx_jm;
    const float hz_jm = (il && kz) ? up_z(v.hz_jm, v.ey_jm, v.ey_jm_ip, v.ex_jm, v.ex) : v.hz_jm;
    const float hy_im = (ji && kh) ? up_y(v.hy_im, v.ex_im, v.ex_kp_im, v.ez_im, v.ez) : v.hy_im;
    const float hz_im = (jl && kz) ? up_z(v.hz_im, v.ey_im, v.ey, v.ex_im, v.ex_jp_im) : v.hz_im;
    const float hx_km = (ii && jl) ? up_x(v.hx_km, v.ez_km, v.ez_km_jp, v.ey_km, v.ey) : v.hx_km;
    const float hy_km = (il && ji) ? up_y(v.hy_km, v.ex_km, v.ex, v.ez_km, v.ez_km_ip) : v.hy_km;

    // A source cell's Dz is written even outside the Dz update range (as in fused_tile).
    const bool rdx = il && ji && kz, rdy = ii && jl && kz, rdz = (ii && ji && kh) || v.src;
    const bool reyz = i >= 1 && k >= 1;
    const float dxu = v.dx + cdy * (hz - hz_jm) - cdz * (hy - hy_km);
    const float dyu = v.dy + cdz * (hx - hx_km) - cdx * (hz - hz_im);
    float dzu = v.dz + cdx * (hy - hy_im) - cdy * (hx - hx_jm);
    dzu = v.src ? dzu - C.jz() : dzu;
    float dyp = dyu, dzp = dzu;
    // E cells whose D is not updated read the target slot's value (in deep rows those are the cells of the high x
    // face, whose E the face takes over).
    if (!deep && reyz && !(rdy && rdz)) {
        if (!rdy) dyp = ld(C.dT(1), o);
        if (!rdz) dzp = ld(C.dT(2), o);
    }

    float exn, eyn, ezn;
    if constexpr (EXACT) {
        {
            // see fused_tile: where d*E^n is -0 or E^n or D^n is not finite, the
            // dropped terms could show, and the operands are loaded after all.
            // -0 is the least integer; a sum of magnitudes is not finite if one
            // of them is not (or, harmlessly, if it overflows).
            const int z = min(min(__float_as_int(v.d * v.ex), __float_as_int(v.d * v.ey)), __float_as_int(v.d * v.ez));
            const float mag = __builtin_fabsf(v.ex) + __builtin_fabsf(v.ey) + __builtin_fabsf(v.ez) +
                              __builtin_fabsf(v.dx) + __builtin_fabsf(v.dy) + __builtin_fabsf(v.dz);
            if (!need && (z == (int)0x80000000 || !__builtin_isfinite(mag))) {
                v.exm = at_once<T, NE>(C.e1(0), o); v.eym = at_once<T, NE>(C.e1(1), o); v.ezm = at_once<T, NE>(C.e1(2), o);
                v.dxm = at_once<T, ND>(C.d1(0), o); v.dym = at_once<T, ND>(C.d1(1), o); v.dzm = at_once<T, ND>(C.d1(2), o);
            }
        }
        exn = e_update(v.c, v.d, v.a, v.g1, v.g2, v.g3, v.ex, v.exm, dxu, v.dx, v.dxm);
        eyn = e_update(v.c, v.d, v.a, v.g1, v.g2, v.g3, v.ey, v.eym, dyp, v.dy, v.dym);
        ezn = e_update(v.c, v.d, v.a, v.g1, v.g2, v.g3, v.ez, v.ezm, dzp, v.dz, v.dzm);
    } else {
        exn = e_update_scaled(v.k1, v.k2, v.k3, v.k5, v.ex, v.exm, dxu, v.dx, v.dxm);
        eyn = e_update_scaled(v.k1, v.k2, v.k3, v.k5, v.ey, v.eym, dyp, v.dy, v.dym);
        ezn = e_update_scaled(v.k1, v.k2, v.k3, v.k5, v.ez, v.ezm, dzp, v.dz, v.dzm);
    }

    // Mur faces beside this cell (fdtd_calculations.cu:237-427): c = {q, A, B, C} of
    // the face cell, tn, sn the neighbour (this cell) at n+1 and n, sf the face at n.
    auto mur = [](const float4 c, float tn, float sn, float sf, bool once) {
        return mur_round<T>(c.x, (c.y * tn + c.z * sn) - c.w * sf, once);
    };
    const bool hi = C.hi_once() != 0;
    if (deep) {   // only the x faces are near
        st(C.h1(0), o, hx); st(C.h1(1), o, hy); st(C.h1(2), o, hz);
        if (il) { st_d(C.dT(0), o, dxu); st_e(C.eT(0), o, exn); }
        if (ii) { st_d(C.dT(1), o, dyu); st_e(C.eT(1), o, eyn); st_e(C.eT(2), o, ezn); }
        if (rdz) st_d(C.dT(2), o, dzu);
        if (i == 1) {
            st_e(C.eT(1), o - ES, mur(mc, X::rnd(eyn), v.ey, v.ey_im, false));
            st_e(C.eT(2), o - ES, mur(mc, X::rnd(ezn), v.ez, v.ez_im, false));
        }
        if (i == nx - 2) {
            // the x-high Ey face reads the source neighbour twice (fdtd_calculations.cu:323-325)
            st_e(C.eT(1), o + ES, mur(mc, v.ey, v.ey, v.ey_ip, hi));
            st_e(C.eT(2), o + ES, mur(mc, X::rnd(ezn), v.ez, v.ez_ip, hi));
        }
        return;
    }
    float pv = 0.0f;
    auto face = [&](int seg, char *dst, uint32_t b, int side, float tn, float sn, float sf, bool once) {
        const float x = mur(C.coef(side, i, j, k), tn, sn, sf, once);
        if (probe < 0) st(dst, b, x);
        else if (seg == pseg) pv = x;
    };
    const bool fx0 = i == 1, fx1 = i == nx - 2, fy0 = j == 1, fy1 = j == ny - 2, fz0 = k == 1, fz1 = k == nz - 2;
    if (fx0 || fx1 || fy0 || fy1 || fz0 || fz1) {
        const float rx = X::rnd(exn), ry = X::rnd(eyn);
        // Ez at k = 0 is outside the E update: a face there reads the target slot (not written in this step)
        float rz = X::rnd(ezn);
        if (k == 0) rz = ld(C.eT(2), o);
        if (fx0) {
            if (jl && kz) face(4, C.eT(1), o - ES, 0, ry, v.ey, v.ey_im, false);
            if (ji && kh) face(8, C.eT(2), o - ES, 0, rz, v.ez, v.ez_im, false);
        }
        if (fx1) {
            if (jl && kz) face(5, C.eT(1), o + ES, 1, v.ey, v.ey, v.ey_ip, hi);
            if (ji && kh) face(9, C.eT(2), o + ES, 1, rz, v.ez, v.ez_ip, hi);
        }
        if (fy0) {
            if (il && kz) face(0, C.eT(0), o - syb, 2, rx, v.ex, v.ex_jm, true);
            if (ii && kh) face(10, C.eT(2), o - syb, 2, rz, v.ez, v.ez_jm, true);
        }
        if (fy1) {
            if (il && kz) face(1, C.eT(0), o + syb, 3, rx, v.ex, v.ex_jp, true);
            if (ii && kh) face(11, C.eT(2), o + syb, 3, rz, v.ez, v.ez_jp, true);
        }
        if (fz0) {
            if (il && ji) face(2, C.eT(0), o - szb, 4, rx, v.ex, v.ex_km, true);
            if (ii && jl) face(6, C.eT(1), o - szb, 4, ry, v.ey, v.ey_km, true);
        }
        if (fz1) {
            if (il && ji) face(3, C.eT(0), o + szb, 5, rx, v.ex, v.ex_kp, true);
            if (ii && jl) face(7, C.eT(1), o + szb, 5, ry, v.ey, v.ey_kp, true);
        }
    }
    if (probe < 0) {
        st(C.h1(0), o, hx); st(C.h1(1), o, hy); st(C.h1(2), o, hz);
        if (rdx) { st_d(C.dT(0), o, dxu); st_e(C.eT(0), o, exn); }
        if (rdy) st_d(C.dT(1), o, dyu);
        if (rdz) st_d(C.dT(2), o, dzu);
        // face cells that a segment covers are stored by their neighbour's lane
        const bool fy = (i == nx - 1 && jl && kz) || (k == nz - 1 && ii && jl);
        const bool fz = (i == nx - 1 && ji && kh) || ((j == 0 || j == ny - 1) && ii && kh);
        if (reyz && !fy) st_e(C.eT(1), o, eyn);
        if (reyz && !fz) st_e(C.eT(2), o, ezn);
        return;
    }
    // the value probe pf records: what this step stores, or what the target slot keeps
    switch (pf) {
    case 0: pv = rdx ? X::rnd(dxu) : ld(C.dT(0), o); break;
    case 1: pv = rdy ? X::rnd(dyu) : ld(C.dT(1), o); break;
    case 2: pv = rdz ? X::rnd(dzu) : ld(C.dT(2), o); break;
    case 3: pv = X::rnd(hx); break;
    case 4: pv = X::rnd(hy); break;
    case 5: pv = X::rnd(hz); break;
    default:
        if (pseg < 0) {
            if (pf == 6) pv = rdx ? X::rnd(exn) : ld(C.eT(0), o);
            else if (pf == 7) pv = reyz ? X::rnd(eyn) : ld(C.eT(1), o);
            else pv = reyz ? X::rnd(ezn) : ld(C.eT(2), o);
        }
        break;
    }
    if ((threadIdx.x & 63) == 1) C.record(probe, pf, pv);
}

template <typename T, bool EXACT, int BXL, int FORM>
__global__ __launch_bounds__(cell_block_lanes(FORM, sizeof(T), BXL)) void cell_step(const CellArgs C)
{
    // What the lanes need of the arguments before their loads can go out, and
    // something of the other cache lines, in one go: left alone, each first use
    // of a line, and each of these, waits in turn (24^3: 5.9 -> 5.2 us a step, 64^3
    // 8.2 -> 8.0).  Never taken: the launch has checked the same.
    if (!cell_args_ok(C)) return;
    cell_block<T, EXACT, BXL, FORM>(OneStep{C}, (int)blockIdx.x, (int)blockIdx.y);
}

// One step of a group of a batch's grids: blocks [start[q], start[q + 1]) of
// the launch are grid q's, a multiple of 8 but for grids of many small planes, so
// that cell_block's mapping of tiles to XCDs holds.  Grids outside their step window are skipped.
template <typename T, bool EXACT, int FORM>
__global__ __launch_bounds__(cell_block_lanes(FORM, sizeof(T), 6)) void cell_batch(const CellInst *inst, const CellGroups *groups, int first,
                                                         int count, int step)
{
    Const<CellGroups> *S = (Const<CellGroups> *)groups;
    const int b = (int)blockIdx.x + S->start[first];
    int lo = first, hi = first + count - 1;
    while (lo < hi) {   // the last grid whose blocks start at or before b
        const int mid = (lo + hi + 1) / 2;
        if (S->start[mid] <= b) lo = mid;
        else hi = mid - 1;
    }
    Const<CellInst> *d = (Const<CellInst> *)inst + S->idx[lo];
    const int n = step - d->start;
    if (n < 0 || n >= d->nsteps) return;
    const int local = b - S->start[lo], gx = d->gx;
    const int bz = local / gx, bx = local - bz * gx;
    const BatchStep C{d, (n + 2) % 3, (n + 1) % 3, n % 3, n & 1, n};
    if constexpr (sizeof(T) == 4 || FORM <= kCellMid) {   // cell_lanes_log2; near groups may take a step in mid
        if (d->bxl == 5) {
            cell_block<T, EXACT, 5, FORM>(C, bx, bz);
            return;
        }
    }
    cell_block<T, EXACT, 6, FORM>(C, bx, bz);
}

template <typename T, bool EXACT>
hipError_t launch_cell_t(const CellArgs &c, hipStream_t s, hipEvent_t t0, hipEvent_t t1)
{
    if (!cell_args_ok(c)) return hipErrorInvalidValue;
    constexpr int kPart = sizeof(T) == 2 ? kCellPart : kCellFar;   // 16 bits only
    const void *wide[] = {(const void *)cell_step<T, EXACT, 6, kCellNear>, (const void *)cell_step<T, EXACT, 6, kCellMid>,
                          (const void *)cell_step<T, EXACT, 6, kPart>, (const void *)cell_step<T, EXACT, 6, kCellFar>};
    const void *k = wide[c.form];
    if (c.bxl == 5) {   // cell_lanes_log2, cell_form: fp32 near, mid and far, 16 bits near
        k = (const void *)cell_step<T, EXACT, 5, kCellNear>;
        if constexpr (sizeof(T) == 4) {
            if (c.form == kCellMid) k = (const void *)cell_step<T, EXACT, 5, kCellMid>;
            if (c.form == kCellFar) k = (const void *)cell_step<T, EXACT, 5, kCellFar>;
        }
    }
    const unsigned gx = (unsigned)c.gx;
    const unsigned waves = (unsigned)c.lanes / 64, pb = ((unsigned)c.p.nprobe + waves - 1) / waves;
    const dim3 grid(gx, (unsigned)c.nz + (pb + gx - 1) / gx);
    CellArgs arg = c;
    void *args[] = {&arg};
    return hipExtLaunchKernel(k, grid, dim3((unsigned)c.lanes), args, 0, s, t0, t1, 0);
}

// One coefficient per thread; blockIdx.y: the face.
__global__ __launch_bounds__(kCoefBlock) void mur_coefs(const MurCoefArgs a)
{
    const int f = (int)blockIdx.y, axis = f >> 1, end = f & 1;
    const long long n = axis == 0 ? (long long)a.ny * a.nz : axis == 1 ? (long long)a.nx * a.nz : (long long)a.nx * a.ny;
    const long long q = (long long)blockIdx.x * kCoefBlock + threadIdx.x;
    if (q >= n) return;
    // the two cells of the pair in the reference's plane: x (k, j, 2), y (k, 2, i), z (2, j, i)
    const long long k = q / a.nx, at = axis == 0 ? 2 * q : axis == 1 ? 2 * k * a.nx + (q - k * a.nx) : q;
    const long long step = axis == 0 ? 1 : axis == 1 ? a.nx : n;
    const float *rp = axis == 0 ? a.rp[end ? 3 : 0] : axis == 1 ? a.rp[end ? 4 : 1] : a.rp[end ? 5 : 2];
    const float rpf = rp[at + (end ? step : 0)], rpn = rp[at + (end ? 0 : step)];
    const float h = axis == 0 ? a.h[0] : axis == 1 ? a.h[1] : a.h[2];
    const long long nyz = (long long)a.ny * a.nz, nxz = (long long)a.nx * a.nz;
    const long long base = axis == 0 ? 0 : axis == 1 ? 2 * nyz : 2 * (nyz + nxz);
    a.out[base + end * n + q] = mur_coef(a.dt, h, a.mu0, a.eps0, rpf, rpn);
}

}  // namespace

hipError_t launch_mur_coefs(const MurCoefArgs &a, int faces, hipStream_t s)
{
    const long long m = std::max({(long long)a.ny * a.nz, (long long)a.nx * a.nz, (long long)a.nx * a.ny});
    mur_coefs<<<dim3((unsigned)((m + kCoefBlock - 1) / kCoefBlock), (unsigned)faces), kCoefBlock, 0, s>>>(a);
    return hipGetLastError();
}

hipError_t launch_cell_step(const CellArgs &c, int storage, hipStream_t s, hipEvent_t t0, hipEvent_t t1)
{
    switch (storage) {
    case kStoreF32: return launch_cell_t<float, true>(c, s, t0, t1);
    case kStoreF32Fast: return launch_cell_t<float, false>(c, s, t0, t1);
    case kStoreF16: return launch_cell_t<__half, false>(c, s, t0, t1);
    case kStoreBF16: return launch_cell_t<__hip_bfloat16, false>(c, s, t0, t1);
    default: return hipErrorInvalidValue;
    }
}

template <typename T, bool EXACT>
static hipError_t launch_cell_batch_t(const CellInst *inst, const CellGroups *groups, int first, int count, int blocks,
                                      int step, int form, int lanes, hipStream_t s)
{
    const dim3 grid((unsigned)blocks), block((unsigned)lanes);
    constexpr int kPart = sizeof(T) == 2 ? kCellPart : kCellFar;   // 16 bits only
    switch (form) {
    case kCellNear: cell_batch<T, EXACT, kCellNear><<<grid, block, 0, s>>>(inst, groups, first, count, step); break;
    case kCellMid: cell_batch<T, EXACT, kCellMid><<<grid, block, 0, s>>>(inst, groups, first, count, step); break;
    case kCellPart: cell_batch<T, EXACT, kPart><<<grid, block, 0, s>>>(inst, groups, first, count, step); break;
    default: cell_batch<T, EXACT, kCellFar><<<grid, block, 0, s>>>(inst, groups, first, count, step); break;
    }
    return hipGetLastError();
}

hipError_t launch_cell_batch(const CellInst *inst, const CellGroups *groups, int first, int count, int blocks, int step,
                             int form, int lanes, int storage, hipStream_t s)
{
    switch (storage) {
    case kStoreF32: return launch_cell_batch_t<float, true>(inst, groups, first, count, blocks, step, form, lanes, s);
    case kStoreF32Fast: return launch_cell_batch_t<float, false>(inst, groups, first, count, blocks, step, form, lanes, s);
    case kStoreF16: return launch_cell_batch_t<__half, false>(inst, groups, first, count, blocks, step, form, lanes, s);
    case kStoreBF16: return launch_cell_batch_t<__hip_bfloat16, false>(inst, groups, first, count, blocks, step, form, lanes, s);
    default: return hipErrorInvalidValue;
    }
}
