// Internal declarations shared by the HIP translation units of libfdtd_amd.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <string.h>
#include <algorithm>
#include <initializer_list>
#include <stdint.h>

#include "fdtd_amd.h"

// q / d for every 32-bit q by a multiply (Granlund and Montgomery, Division by
// invariant integers using multiplication, 1994): with s = ceil(log2 d) and
// mul = floor(2^32 (2^s - d) / d) + 1.  div_consts: 2 <= d < 2^32.
inline void div_consts(unsigned long long d, uint32_t &mul, uint32_t &shift)
{
    uint32_t s = 0;
    while ((1ull << s) < d) s++;
    mul = (uint32_t)((((1ull << s) - d) << 32) / d + 1);
    shift = s - 1;
}
__host__ __device__ inline uint32_t div_by(uint32_t q, uint32_t mul, uint32_t shift)
{
    const uint32_t t = (uint32_t)(((uint64_t)mul * q) >> 32);
    return (t + ((q - t) >> 1)) >> shift;
}

// Per-material Debye coefficients in the precision the reference evaluates
// them (fdtd_calculations.cu:141-155): a, c, d are double expressions rounded
// to float; the three D weights are double.  With these, an E update
// c*(d*E^n - a*E^{n-1} + g1*D^{n+1} - g2*D^n + g3*D^{n-1}) evaluated as
// float products, then double sums, reproduces the reference's rounding.
struct MatCoef {
    float a, c, d, pad;
    double g1, g2, g3;
    // Scaled-unit form for 16-bit storage (fields stored as E/sE, (D/eps0)/sD,
    // (eta0 H)/sH; all arithmetic fp32):
    // E' = k1 E - k2 E_prev + k3 (D' - D) + k5 ((D' - D) - (D - D_prev)).
    float k1, k2, k3, k5;
};

// Material id byte: low 7 bits index the coefficient table, the top bit marks
// a soft Jz source cell (fdtd_calculations.cu:187-213 semantics).
constexpr int kMaxMaterials = 128;
constexpr uint8_t kSourceBit = 0x80;
constexpr uint8_t kMaterialMask = 0x7f;

// Host-side coefficient builder shared by the legacy and fused paths.
MatCoef fdtd_mat_coef(float dt, float eps0, float sigma, float epsS, float epsI, float tau, int debye_mode);

// Field storage of a context.
enum Storage { kStoreF32 = 0, kStoreF16 = 1, kStoreBF16 = 2, kStoreF32Fast = 3 };

// Arguments of the fused H -> D (+source) -> E kernel for one time step.
// Field pointers point at element type float, __half or __hip_bfloat16
// according to the launch's storage.
struct StepArgs {
    const void *hxo, *hyo, *hzo;    // H^{n-1/2}
    void *hxn, *hyn, *hzn;          // H^{n+1/2}
    const void *ex0, *ey0, *ez0;    // E^n
    const void *ex1, *ey1, *ez1;    // E^{n-1}
    void *exT, *eyT, *ezT;          // E^{n+1} (ring target slot)
    const void *dx0, *dy0, *dz0;    // D^n
    const void *dx1, *dy1, *dz1;    // D^{n-1}
    void *dxT, *dyT, *dzT;          // D^{n+1} (ring target slot)
    const uint8_t *ids;
    const MatCoef *lut;
    int nmat;
    float jz;
    int nx, ny, nz;
    int pitch;                      // elements between rows (>= nx)
    long long plane;                // elements between z planes (>= pitch*ny)
    float chx, chy, chz;            // dt/(mu0*dx), dt/(mu0*dy), dt/(mu0*dz)
    float cdx, cdy, cdz;            // dt/dx, dt/dy, dt/dz
    int kchunk;                     // z planes per block
    int tiles_x, tiles_y, tiles_z;  // logical tile grid
    int xcd_remap;                  // block -> tile order (FdtdExt.xcd_remap; xcd_logical)
    unsigned guard;                 // addressable elements before and after every field array (and ids)
    // Mur x faces updated inside the fused kernel (fused_mur_x): 0 none, 1
    // all four (Ey, Ez at i = 0 and nx-1), 2 the two at i = 0 only.
    int mur_x;
    const float4 *murx0, *murx1;    // per (k, j) coefficients of the x-low / x-high faces (launch_mur_coefs)
    int cpl;                        // cells per lane: 1, or 2 for 16-bit storage (128-cell tiles)
    int txw;                        // threads per tile row with one cell per lane: 64 or 128
    // Exact fp32 form: a half wave (32 cells of a tile row) whose cells all
    // have materials whose Debye update multiplies E^{n-1} and D^{n-1} by +0
    // (a = +0 and g3 = +0, i.e. tau = +0) does not load those six operands
    // (see fused_tile).
    int zskip;
};

// Coefficients {q, A, B, C} of the first-order Mur update of one face
// cell, E' = q*((A*tn + B*sn) - C*sf), evaluated in float exactly as the
// reference's expression (fdtd_calculations.cu:216-428) rounds
// them: q = 1/(dt + h sqrt(mu0 eps0 rp_face)), A = dt - h sqrt(mu0 eps0
// rp_nb), B = dt + h sqrt(mu0 eps0 rp_nb), C = dt - h sqrt(mu0 eps0
// rp_face).  launch_mur_coefs: of the first `faces` of a grid's six, from its rp
// planes in fdtd_ctx_set_rp's order: out holds x low, x high in (k, j) order,
// y low, y high in (k, i) order, z low, z high in (j, i) order, one after the
// other.
struct MurCoefArgs {
    const float *rp[6];
    float4 *out;
    int nx, ny, nz;
    float dt, h[3], mu0, eps0;
};
inline size_t mur_coef_count(int nx, int ny, int nz)
{
    return 2 * ((size_t)ny * nz + (size_t)nx * nz + (size_t)nx * ny);
}
hipError_t launch_mur_coefs(const MurCoefArgs &a, int faces, hipStream_t s);

// Which Mur x faces the fused kernel takes over.  The x-high faces need the
// cell at i = nx-2 from the face's wave: E^{n+1}_z from the previous lane
// through a wave shuffle, and E^n_y, E^n_z from the LDS column that lane
// staged, read after the plane's last barrier (only the staging wave's own
// program order keeps the next plane from overwriting it).  When nx-1 is a
// multiple of the cells one wave covers (tile_cells: 64, or 128 with two
// cells per lane; a 128-wide tile of one cell per lane is two waves of 64)
// the face is the first cell of a wave, that neighbour belongs to another
// wave or tile, and both x-high faces stay in the Mur kernel.
// The fused kernel stages the coefficients of its z-chunk in LDS, so chunks
// longer than kFusedMurMaxChunk planes leave the x faces to the Mur kernel.
constexpr int kFusedMurMaxChunk = 16;
inline int fused_mur_x(int nx, int kchunk, int tile_cells)
{
    if (kchunk > kFusedMurMaxChunk) return 0;
    return (nx - 1) % tile_cells == 0 ? 2 : 1;
}
// Mur segments (in mur_segments order) left to the Mur kernel.
inline unsigned mur_skip_mask(int mur_x)
{
    // segments 4, 5: Ey at i = 0, nx-1; 8, 9: Ez at i = 0, nx-1
    return mur_x == 1 ? (1u << 4 | 1u << 5 | 1u << 8 | 1u << 9) : mur_x == 2 ? (1u << 4 | 1u << 8) : 0u;
}

// Row pitch (elements) of the fused layout: rows start on 128-byte lines, so
// the 256-byte row segment a wave64 of fp32 lanes reads (or a 128-byte one
// of 16-bit lanes) never straddles an extra line.  Measured on MI355X: a
// 100x100x130 grid streams at 2.5 TB/s with rows packed (pitch = nx) and a
// 128^3 one at 4.4 TB/s.  Rows of 4 KiB or more whose length is a multiple
// of 2 KiB get one more line: such strides map the rows of a tile, and the
// planes of a z-march, onto the same DRAM channels.  Fused kernel, box
// phantom, best z-chunk each way (Gcell-updates/s): 2048x512x300 55.9 ->
// 63.1, 1536x1024x200 55.6 -> 62.7, 2048x1024x150 52.1 -> 60.8,
// 1000x1000x300 (pitch 1024) 56.4 -> 59.9, 1024x1024x200 60.2 -> 61.7; 2 KiB
// rows (512 fp32) gain nothing (512^3 61.5 -> 61.7), 1 KiB rows lose.
inline int fused_pitch(int nx, size_t esz)
{
    const int q = (int)(128 / esz);
    const int p = (nx + q - 1) / q * q;
    const size_t bytes = (size_t)p * esz;
    return bytes >= 4096 && bytes % 2048 == 0 ? p + q : p;
}

// Guard (in elements) the fused kernel needs around every field array and
// the id array so that its halo loads need no bounds checks: one plane, ten
// rows and 256 elements (tiles are at most 8 rows high and 128 cells wide).
// Extra elements between consecutive field arrays: staggers the arrays' starts
// across HBM channels, also where a plane is a power of two (256^3 fp32 by cells,
// us a step: 327 with 0, 1024 or 65536, 280 to 285 with 64, 4160 or 1088).  Tiles,
// 1088 against 65536 and 66624: 128^3 48.6, 46.3, 45.9; 223x190x170 141, 139, 138;
// 300x250x220 304, 295, 295; 290x310x300 511, 506, 503; 320x320x880 1512, 1530,
// 1509; but 192^3 127, 130, 130 and 256^3 287, 295, 293.
constexpr size_t kCellSkew = 1088, kTileSkew = 66624;
inline long long fused_guard(int pitch, long long plane) { return plane + 10LL * pitch + 256; }

// Arguments of the 6-face first-order Mur kernel (fdtd_calculations.cu:216-428).
struct MurArgs {
    void *exT, *eyT, *ezT;               // E^{n+1}
    const void *exS, *eyS, *ezS;         // E^n
    const float *rpx0, *rpy0, *rpz0, *rpxEnd, *rpyEnd, *rpzEnd;
    int nx, ny, nz, pitch;
    long long plane;
    float dt, hx, hy, hz, mu0, eps0;
    int seg_start[13];                   // prefix sums of the 12 face segments
};

struct ProbeArgs {
    const void *field[9];                // Dx Dy Dz Hx Hy Hz Ex Ey Ez of the newest level
    double factor[9];                    // stored value -> SI (1 for fp32 storage)
    const int *probes;                   // nprobe x (field, i, j, k)
    int nprobe;
    int pitch;
    long long plane;
    double *out;                         // [step][probe]
    int row;
};

// Electromagnetic energy sum_cells (E.D / 2 + mu0 |H|^2 / 2) of the newest
// levels, accumulated in fp64: per-block partial sums, then one block adds
// them in a fixed order (the result does not depend on scheduling).
struct EnergyArgs {
    const void *E[3], *D[3], *H[3];
    int nx, ny, nz, pitch;
    long long plane;
    double ed_factor, hh_factor;         // stored products -> SI: E.D and mu0 H^2
    double *partial;                     // kEnergyBlocks doubles
    double *out;                         // the sum is written here
};
constexpr int kEnergyBlocks = 1024;
hipError_t launch_energy(const EnergyArgs &a, int storage, hipStream_t s);

// One bit per material: set where a = g3 = +0.  All ids have one, as in the
// tiles' zero-term rows: with a single word, a grid whose vacuum had an id of 40
// took 30.7 us a step at 128^3 and 307 at 256^3, with four 28.0 and 287; ids
// below 32 take as long as with one.
struct ZeroTerms {
    uint32_t w[kMaxMaterials / 32];
    __host__ __device__ bool has(uint32_t m) const
    {
        static_assert(kMaxMaterials == 128, "four words");
        const uint32_t lo = m & 32 ? w[1] : w[0], hi = m & 32 ? w[3] : w[2];   // selects: w may lie in scalar registers
        return (m & 64 ? hi : lo) >> (m & 31) & 1u;
    }
};

// One step of a grid in one launch, one cell per lane, with its Mur faces and
// probe row (fdtd_cell.hip).  The field and id pointers lie fused_guard
// elements before the arrays' origins; o0 = the guard in bytes.
// Forms of cell_step: its state in the Infinity Cache; x neighbours from the
// lanes beside instead of loads; the same with D past the cache (16 bits only);
// with D and all but the loads of E^n past it.
enum { kCellNear, kCellMid, kCellPart, kCellFar };
struct CellArgs {
    const char *e0[3], *e1[3], *d0[3], *d1[3], *h0[3];   // E, D at levels n and n-1, H^{n-1/2}
    char *eT[3], *dT[3], *h1[3];                         // E, D at level n+1, H^{n+1/2}
    const uint8_t *ids;
    const MatCoef *lut;
    int nx, ny, nz;
    uint32_t o0, sy, sz;           // bytes: guard, row, plane
    int tiles_x, tiles, run, gx;   // tiles per row and per plane; tiles in a row on one XCD, or 0; blocks per plane (cell_tiles)
    uint32_t tx_mul, tx_shift;     // div_consts(tiles_x)
    float ch[3], cd[3], jz;
    ZeroTerms zmask;               // materials whose cells do not load levels n-1
    int bxl, lanes;                // 5 or 6: 32 or 64 lanes of a tile along x; lanes of a tile and block
    int hi_once;                   // the tiled step leaves the x-high faces to the Mur kernel (fused_mur_x 2)
    int form;                      // kCellNear, ...
    int flip;                      // planes from the highest down: every other step, so that a step starts where
                                   // the last one ended
    const float4 *mur[6];          // launch_mur_coefs: x low, x high, y low, ...
    ProbeArgs p;                   // p.nprobe = 0: no probe row; p.field is not read
};
// Even addresses and pitches, counts that are not negative.
__host__ __device__ inline bool cell_args_ok(const CellArgs &c)
{
    uintptr_t odd = (uintptr_t)c.ids | (uintptr_t)c.mur[0] | (uintptr_t)c.dT[0] | (uintptr_t)c.d1[0] | (uintptr_t)c.lut;
    for (int q = 0; q < 3; q++) odd |= (uintptr_t)c.e0[q] | (uintptr_t)c.h0[q] | (uintptr_t)c.d0[q];
    odd |= c.o0 | c.sy | c.sz;
    const int neg = c.nx | c.ny | c.nz | c.tiles_x | c.tiles | c.run | c.flip;
    return !(((uint32_t)odd & 1u) | ((uint32_t)neg >> 31));
}
// Padded state (bytes of the 24 field arrays) up to which a context steps
// with cell_step.  Far past the Infinity Cache both launches wait for HBM, and
// the tiled one keeps more of it in flight; what cell_step gains there is the
// part of the state that the last step left in the cache.  fp32, tiles' time
// over cell_step's, each with its own stagger of the arrays, means over two to
// four placements that differ by less than 1 %:
//   an odd number of half waves a row (cell_lanes_log2: two rows a wave): 96x450x450 1.00, 151x300x420 1.01, 160x400x300
//     1.01, 223x300x300 1.03, 280x280x255 1.03, 350x330x178 1.02 (1.8 to 2.0 GB); 350x330x260 0.99, 410x300x240 1.00 (2.9);
//   up to four half waves: 0.6 GB 1.04 to 1.06, 0.8 GB 1.00 to 1.06, 1.0 GB 0.95 to 1.00, 2.0 GB 0.92 to 0.95;
//   six: 0.85 GB 1.06 to 1.08, 1.1 to 1.3 GB 0.99 to 1.02, 1.5 GB 0.95 to 0.97;
//   more, whole waves: 1.6 GB 0.98 to 1.04, 320x320x224 1.03, 256x256x384 (2.4) 1.03, 2.5 to 2.6 GB 0.98 to 1.00;
//   more, others: 1.2 GB 1.01 to 1.05, 300x250x220 (1.7) 0.97, 300^3 0.98, 500x300x250 (3.7) 0.97.
// 16 bits: 1.03 to 1.3 for rows of 20 to 512 cells at 4.5 to 6.4 GB.
constexpr int kCellMaxPlanes = 60000;   // planes and, in rows of at least 8 blocks, probes are blockIdx.y
constexpr int kCellMaxProbes = 40000;
inline size_t cell_state_limit(int nx, size_t esz)
{
    if (esz == 2) return 6000000000;
    const int half = (nx + 31) / 32;
    if (half % 2) return 2000000000;
    if (half <= 4) return 850000000;
    return half == 6 || nx % 64 ? 1200000000 : 2450000000;
}
// The same of a batch's grids, whose tiles (fused_batch) take 0 to 10 % longer
// than a context's.  fp32, their time over cell_batch's: two half waves 0.7 GB
// 1.01, 1.0 to 1.1 GB 0.95 to 0.97; four 1.0 to 1.6 GB 1.00 to 1.04, 2.0 GB 0.99;
// six 1.7 to 2.0 GB 1.02, 2.3 GB 1.00, 2.5 GB 0.98; 256 to 448 cells 2.2 to 2.6 GB
// 1.01 to 1.09; an odd number 1.9 to 2.4 GB 1.04 to 1.06.
inline size_t cell_batch_limit(int nx, size_t esz)
{
    if (esz == 2) return 6000000000;
    const int half = (nx + 31) / 32;
    if (half % 2) return 2000000000;
    if (half == 2) return 850000000;
    if (nx % 64) return 1200000000;
    return half == 4 ? 1600000000 : half == 6 ? 2300000000 : 2600000000;
}
// Its form.  us of near, mid and far, or of near, mid and part, over rows of 64
// to 320 cells, means over three or four placements, which differ by up to 2 %.
// fp32: 220 MB 30 to 35, 30 to 35, 41 to 49; 270 MB 47 to 52, 44 to 50, 47 to 58;
// 320 MB 65 to 70, 57 to 64, 57 to 71; 360 MB 75 to 83, 66 to 75, 60 to 76; 500 MB
// 100 to 109, 93 to 102, 82 to 101.  16 bits: 222 MB 38 to 44, 39 to 41, 49 to 54;
// 248 MB 44 to 51, 43 to 49, 53 to 58; 268 MB 54 to 61, 53 to 57, 58 to 63; 280 MB
// 63 to 71, 59 to 67, 60 to 65; 360 MB 92 to 101, 83 to 92, 77 to 83.  From there
// part over mid: rows that are no whole waves 0.93 to 1.00 at every size, most
// 0.96 to 0.98; whole waves 0.94 to 0.99 to 450 MB, 0.99 to 1.03 at 550 to 800 MB
// (256^3 184 mid, 188 part), 0.98 to 1.00 at 900 MB, 0.95 to 0.98 past 1 GB.  far
// over part from 1.1 to 5.8 GB: rows of 64 and 100 cells 1.02 to 1.04, 160 to 256
// 0.99 to 1.03, 300 to 384 0.98 to 1.01 (most below 1), 417 to 777 0.97 to 0.99.
inline int cell_form(int nx, size_t state, size_t esz)
{
    if (state <= 220000000) return kCellNear;
    if (esz == 2) {
        if (state <= 275000000) return kCellMid;
        if (state > 1000000000 && nx > 256) return kCellFar;
        return nx % 64 == 0 && state > 500000000 && state <= 850000000 ? kCellMid : kCellPart;
    }
    return state <= 360000000 ? kCellMid : kCellFar;
}
// log2 of the lanes of its tiles along x: 64, or 32.  Near: 32 where 64 leave
// clearly more lanes idle (96 wide: 16.1 against 16.8 us in fp32, 13.0 against
// 13.8 in fp16; 160 wide, where 32 lanes would fill 20 % more: 35.2 against
// 37.5).  Else in fp32 wherever they take fewer lanes (90x150x300 88 against 101
// us, 151x138x188 77.8 against 81.1, 210x150x150 84.2 against 87.1; as many:
// 256^3 299 against 291); not for 16-bit fields, whose second row's ends cost
// more (71x79x1000 140 against 119).
inline int cell_lanes_log2(int nx, int form, size_t esz)
{
    if (form != kCellNear) return esz == 4 && ((nx + 31) / 32) % 2 ? 5 : 6;
    const double e6 = (double)nx / (64 * ((nx + 63) / 64)), e5 = (double)nx / (32 * ((nx + 31) / 32));
    return e6 < 0.8 * e5 ? 5 : 6;
}
// Lanes of a block: one wave, or four where fp32 streams past the cache in
// 64-lane tiles and the rows of a block share their halo rows' lines (us, 64
// against 256: 256^3 298, 289; 192^3 126, 122).  Elsewhere a block of one wave
// leaves and makes room at once: 32^3 4.8, 5.4; 100^3 18.9, 20.5; 151x138x188
// 74.6, 78.7; fp16 96x121x77 13.1, 13.4, 320x320x300 320, 323; twelve batched
// grids 28.2, 29.7 ms (128 lanes in between).
constexpr int cell_block_lanes(int form, size_t esz, int bxl)
{
    return form == kCellFar && esz == 4 && bxl == 6 ? 256 : 64;
}
// The tile geometry of a grid (CellArgs, CellInst) and the materials whose
// cells skip levels n-1.
// A plane takes 8 runs of blocks, one per XCD (cell_tile), the last ones part
// empty.  Where that leaves a launch of many planes mostly of empty blocks it is
// their dispatch, about one a nanosecond, that takes the time; such a plane takes
// as many blocks as it has tiles, as they come (run = 0): us a step, 3x3x10000
// fp32 77 -> 29, 10x10x10000 fp16 143 -> 76, 130x3x10000 fp32 187 -> 109 (in tiles
// 38, 120, 122).
template <typename A>
inline void cell_tiles(int nx, int ny, int nz, int nprobe, int form, size_t esz, A &a)
{
    a.bxl = cell_lanes_log2(nx, form, esz);
    a.lanes = cell_block_lanes(form, esz, a.bxl);
    const int bx = 1 << a.bxl, by = a.lanes / bx;
    a.tiles_x = (nx + bx - 1) / bx;
    if (a.tiles_x > 1) div_consts(a.tiles_x, a.tx_mul, a.tx_shift);
    else a.tx_mul = a.tx_shift = 0;
    a.tiles = a.tiles_x * ((ny + by - 1) / by);
    a.run = (a.tiles + 7) / 8;
    const long long rows = nz + ((long long)nprobe + a.tiles - 1) / a.tiles;   // blockIdx.y, without the runs
    if (10LL * a.tiles < 64LL * a.run && 8LL * a.run * nz > 16384 && rows < 65536) a.run = 0;
    a.gx = a.run ? 8 * a.run : a.tiles;
}
// The tile of block bx of a plane.
__host__ __device__ inline int cell_tile(int bx, int run) { return run ? (bx & 7) * run + (bx >> 3) : bx; }
// The row of tiles that tile t of a plane lies in.
__host__ __device__ inline int cell_tile_row(int t, int tiles_x, uint32_t tx_mul, uint32_t tx_shift)
{
    return tiles_x == 1 ? t : (int)div_by((uint32_t)t, tx_mul, tx_shift);
}
inline ZeroTerms cell_zmask(const MatCoef *lut, int nmat)
{
    ZeroTerms z = {};
    for (int m = 0; m < nmat; m++) {
        uint32_t a, g[2];
        memcpy(&a, &lut[m].a, 4);
        memcpy(g, &lut[m].g3, 8);
        if (a == 0 && g[0] == 0 && g[1] == 0) z.w[m >> 5] |= 1u << (m & 31);
    }
    return z;
}
hipError_t launch_cell_step(const CellArgs &c, int storage, hipStream_t s, hipEvent_t t0 = nullptr,
                            hipEvent_t t1 = nullptr);

// Streaming probe (fdtd_stream_probe): 15 read and 9 written arrays of n floats.
struct StreamMix {
    const float *r[15];
    float *w[9];
    long long n;
    // row > 0: the 24 arrays interleaved by rows of `row` elements (row
    // records: the 24 rows of cells [q*row, (q+1)*row) contiguous, 15 read
    // then 9 written) from r[0]; r and w unused otherwise
    int row;
};
hipError_t launch_stream_mix(const StreamMix &p, int blocks, hipStream_t s);
// Blocks of the streaming probe resident on the whole device at once.
int stream_mix_resident_blocks();

// t0, t1 (optional): events that take the launch's start and end times.
hipError_t launch_fused_step(const StepArgs &a, int ty, int storage, hipStream_t s, hipEvent_t t0 = nullptr,
                             hipEvent_t t1 = nullptr);

// Two time steps in one launch (fp32 storage, the exact form).  A holds the
// roles of step n -> n+1 (level n+1 goes to A.exT.., A.dxT..); step n+1 ->
// n+2 writes level n+2 into the spare slot exS.., dxS.. and H^{n+3/2} into
// A.hxn..  A.tiles_* and A.kchunk describe the two-step tile grid
// (two_step_tiles); A.mur_x is not read (all six faces of step n+1 are
// applied in the kernel, those of step n+2 are left to the Mur kernel).
struct Step2Args {
    StepArgs A;
    void *exS, *eyS, *ezS;                   // E^{n+2}
    void *dxS, *dyS, *dzS;                   // D^{n+2}
    float jz2;                               // the source value of step n+1 -> n+2
    const float *rpy0, *rpyEnd, *rpz0, *rpzEnd;   // Mur planes of the y and z faces (MurArgs layout)
    float dt, hy, hz, mu0, eps0;
};
// Rows of the two-step kernel's 64-lane tiles; each tile stores the inner
// 62 x (rows - 2) cells.
constexpr int kTwoStepRows = 8;
constexpr int kTwoStepCols = 62;
inline void two_step_tiles(int nx, int ny, int nz, int kchunk, int rows, int *tx, int *ty, int *tz)
{
    *tx = (nx + kTwoStepCols - 1) / kTwoStepCols;
    *ty = (ny + rows - 3) / (rows - 2);
    *tz = (nz + kchunk - 1) / kchunk;
}
hipError_t launch_fused_step2(const Step2Args &a, int rows, hipStream_t s, hipEvent_t t0 = nullptr,
                              hipEvent_t t1 = nullptr);
hipError_t launch_mur(const MurArgs &a, int storage, hipStream_t s);
hipError_t launch_probes(const ProbeArgs &a, int storage, hipStream_t s);
// Halo planes of a z-slab: n runs of `words` 16-byte words each.
constexpr int kHaloFields = 5;
struct PlaneCopy {
    const uint4 *src[kHaloFields];
    uint4 *dst[kHaloFields];
    int n;
    long long words;
};
hipError_t launch_plane_copy(const PlaneCopy &p, hipStream_t s);
// The nine newest fields of a context as packed fp32 volumes in the
// reference's layout (field f at out + f*nx*ny*nz, OFFSET order), stored
// values times factor[f] in double (scales undone), as get_field computes
// them on the host; fp32 storage copies the bits.
struct SnapArgs {
    const void *field[9];
    double factor[9];
    float *out;
    int nx, ny, nz, pitch;
    long long plane;
    uint32_t nx_mul, nx_shift;     // div_consts(nx), set at launch
};
hipError_t launch_snapshot(const SnapArgs &a, int storage, hipStream_t s);
// Mur faces and one probe row in one launch (p.nprobe = 0: faces only).  The
// probe fields must be the newest levels, with E the Mur target a.exT..ezT.
hipError_t launch_mur_probes(const MurArgs &a, const ProbeArgs &p, int storage, hipStream_t s);
// Prefix sums of the 12 Mur face segments; segments whose bit is set in
// `skip` get no cells.
void mur_segments(int nx, int ny, int nz, int *seg_start, unsigned skip = 0);

// ---- batches of independent grids -------------------------------------
//
// A batch advances many grids with one persistent fused launch per storage
// class and step, one Mur launch and one probe launch.  The launches read
// everything that changes from device memory (the instance descriptors, the
// per-class work tables and a batch step counter), so a captured sequence of
// steps replays unchanged while grids join and leave between replays.

constexpr int kBatchMaxInst = 512;        // descriptors per batch
constexpr int kBatchMaxProbes = 64;       // probes per instance
// Kernel classes of a batch: the four storage forms with one cell per lane
// (class = Storage value), then fp16 and bf16 with two cells per lane.
constexpr int kBatchClasses = 6;
inline int batch_class(int storage, int cpl)
{
    return cpl == 2 ? (storage == kStoreF16 ? 4 : 5) : storage;
}
inline int class_storage(int cls) { return cls < 4 ? cls : (cls == 4 ? kStoreF16 : kStoreBF16); }

// Cells per lane of the fused kernel for a grid nx wide: 16-bit storage runs
// two per lane (128-cell tiles) unless that leaves clearly more lanes idle
// than 64-cell tiles (a pair tile costs ~0.82 of a single one per cell, as
// measured at 256^3); `requested` 1 or 2 overrides.
inline int auto_lane_cells(int nx, size_t esz, int requested)
{
    if (esz != 2) return 1;
    if (requested == 1 || requested == 2) return requested;
    const double e1 = (double)nx / (64.0 * ((nx + 63) / 64)), e2 = (double)nx / (128.0 * ((nx + 127) / 128));
    return e2 >= 0.85 * e1 ? 2 : 1;
}

// Default launch shape of a grid launched alone (tile rows ty given), from
// sweeps on MI355X of 9 grid sizes (64^3 to 320x320x880) x tile rows {2, 4,
// 8} x z-chunks {4, 8, 16}, fp32, and of 8 sizes x {1, 2} cells per lane,
// fp16 and bf16:
//  * pairs (128-cell tiles, one 32-bit access per stream) beat single cells
//    where 128-cell rows are nearly full and the launch fills the GPU (fp16
//    256^3: 203 against 267 us; 128^3: 35 against 45), and lose elsewhere
//    (320 wide: 1115 against 1101; 200 wide: 53 against 48), also where
//    64-cell tiles would waste as many lanes;
//  * the z-chunk trades prologues (each block reloads and recomputes the
//    plane below its chunk) against the partial last round of blocks.  A
//    launch of B blocks on R resident ones costs about ceil(B / R) rounds
//    of kchunk + 2 planes; the chunk of least cost among 4, 8 and 16 is the
//    measured best, or within 2%, at every size but 200x100x100 (within 6%):
//    fp32 320x320x880 16 planes, 1544 against 1620 us at 4; 192^3 8 planes,
//    138 against 148 (16: 153); fp16 320x320x880 16 planes, 1101 against 1251.
// Resident blocks per CU: 4 waves per SIMD for pairs (their VGPR budget), 5
// for single cells, over ty waves a block.
inline long long alone_blocks(int nx, int ny, int nz, int width, int ty, int kchunk)
{
    return (long long)((nx + width - 1) / width) * ((ny + ty - 1) / ty) * ((nz + kchunk - 1) / kchunk);
}
inline long long alone_resident(int cus, int ty, int cpl)
{
    return (long long)cus * std::max(1, 4 * (cpl == 2 ? 4 : 5) / ty);
}
inline int auto_lane_cells_alone(int nx, int ny, int nz, int ty, int kchunk, size_t esz, int requested, int cus)
{
    if (esz != 2) return 1;
    if (requested == 1 || requested == 2) return requested;
    if ((double)nx / (128.0 * ((nx + 127) / 128)) < 0.9) return 1;
    return alone_blocks(nx, ny, nz, 128, ty, kchunk > 0 ? kchunk : 4) >= alone_resident(cus, ty, 2) ? 2 : 1;
}
inline int auto_kchunk_alone(int nx, int ny, int nz, int ty, int cpl, int cus)
{
    const long long R = alone_resident(cus, ty, cpl);
    int best = 4;
    long long best_cost = -1;
    for (int kc : {4, 8, 16}) {
        const long long rounds = (alone_blocks(nx, ny, nz, 64 * cpl, ty, kc) + R - 1) / R;
        const long long cost = rounds * (kc + 2);
        if (best_cost < 0 || cost <= best_cost) { best = kc; best_cost = cost; }
    }
    return std::min(best, nz);
}
constexpr int kMurBlock = 256;            // Mur face cells per block

// Device descriptor of one grid of a batch.  Instance step n (0-based) runs
// at batch step start + n for n < nsteps; outside that window the instance
// is left untouched.
struct BatchInst {
    void *E[3][3];                 // [ring slot][component]
    void *D[3][3];
    void *H[2][3];                 // [buffer][component]; buffer n % 2 holds H^{n-1/2}
    const uint8_t *ids;            // with fused_guard() bytes before and after
    const MatCoef *lut;
    const float *jz;               // per-step source values in storage units
    const float *rp[6];            // rpx0 rpy0 rpz0 rpxEnd rpyEnd rpzEnd
    const int *probes;             // nprobe x (field, i, j, k)
    double *probe_out;             // [step][probe], nsteps rows
    double factor[9];              // stored value -> SI, per field
    long long plane;
    int nmat, jz_len, jz_hold3, start, nsteps, storage;
    int nx, ny, nz, pitch;
    unsigned guard;
    float ch[3], cd[3];
    int kchunk, tiles_x, tiles_y, tiles_z;
    int mur_x;                     // see StepArgs
    const float4 *murx0, *murx1;   // see StepArgs
    int cpl;                       // cells per lane (kernel class)
    int zskip;                     // see StepArgs
    int nprobe, probe_rows;        // probe_out holds probe_rows rows
    float dt, hx, hy, hz, mu0, eps0;
    int mur_seg[13];
};

// Work list of one storage class: instance indices and prefix sums of their
// fused tiles.
struct BatchClass {
    int n, total;
    int idx[kBatchMaxInst];
    int start[kBatchMaxInst + 1];
};

// Work lists shared by all classes: Mur blocks per instance (prefix sums in
// units of kMurBlock face cells) and the flattened probe records.
struct BatchShared {
    int step;                      // batch step counter (advanced on the device)
    int nmur, mur_total;
    int mur_idx[kBatchMaxInst];
    int mur_start[kBatchMaxInst + 1];
    int nrec;
    int rec[kBatchMaxInst * kBatchMaxProbes][2];   // (instance, probe)
};

// A batch's grid as cell_batch steps it.  Field and id pointers as in
// CellArgs, by ring slot and H buffer.
struct CellInst {
    char *E[3][3], *D[3][3], *H[2][3];
    const uint8_t *ids;
    const MatCoef *lut;
    const float *jz;
    const float *rp[6];
    const float4 *murx0, *murx1;
    const int *probes;
    double *probe_out;
    double factor[9];
    int nx, ny, nz;
    uint32_t o0, sy, sz;
    int tiles_x, tiles, run, gx;
    uint32_t tx_mul, tx_shift;
    float ch[3], cd[3];
    ZeroTerms zmask;
    int hi_once, bxl, lanes;
    int nprobe, probe_rows, jz_len, jz_hold3, start, nsteps;
    float dt, h[3], mu0, eps0;
};

// The groups' grids one after another, and prefix sums of their blocks.
struct CellGroups {
    int idx[kBatchMaxInst];
    int start[kBatchMaxInst + 1];
};
// Blocks of a grid's step: its planes' and its probes' (one a wave).
inline int cell_blocks(const CellInst &d)
{
    const int gx = d.gx, w = d.lanes / 64, pb = (d.nprobe + w - 1) / w;
    return gx * (d.nz + (pb + gx - 1) / gx);
}
hipError_t launch_cell_batch(const CellInst *inst, const CellGroups *groups, int first, int count, int blocks, int step,
                             int form, int lanes, int storage, hipStream_t s);

struct BatchLaunch {
    const BatchInst *inst;
    const BatchClass *cls;         // the launch's class
    BatchShared *sh;
    int off;                       // step offset from sh->step
    int xcd_runs;                  // tiles per XCD run (kBatchXcdRun), 0 = identity order
};
// Tile order of the batch's persistent kernel: each group of 8 runs of this
// many tiles gives one run to each XCD, so consecutive tiles (rows along x
// and their neighbouring rows, which read the same halo lines) share an L2.
// Batched set on MI355X (64 grids, fp32): 43.06 against 42.75 Gcell-updates/s
// for the identity order; runs of 4 and 16 tiles gain less, an eighth of each
// round of resident blocks per XCD loses 2 %.
constexpr int kBatchXcdRun = 8;

// LDS bytes of the batch's fused kernel (coefficient table of kMaxMaterials).
size_t batch_fused_lds();
hipError_t launch_fused_batch(const BatchLaunch &l, int ty, int cls, int grid, hipStream_t s);
hipError_t launch_mur_batch(const BatchLaunch &l, int grid, hipStream_t s);
hipError_t launch_batch_advance(BatchShared *sh, int steps, hipStream_t s);
// Resident blocks of the fused batch kernel of a class per CU.
int batch_fused_occupancy(int ty, int cls);

// ---- shared host helpers (fdtd_common.cpp) ------------------------------

struct GridGeom {
    float dt, dx, dy, dz, mu0, eps0;
};

int fdtd_fail(int code, const char *fmt, ...);
int fdtd_hip_fail(hipError_t e, const char *what);
uint16_t f32_to_f16(float f);
float f16_to_f32(uint16_t h);
uint16_t f32_to_bf16(float f);
float bf16_to_f32(uint16_t h);
void fdtd_scaled_coef(MatCoef &m, double dt, double eps0, double sg, double es, double ei, double tau, int debye_mode,
                      double ratio);
void fdtd_build_lut(const float *table, int nmat, float dt, float eps0, int debye_mode, int storage, double sE,
                    double sD, MatCoef *lut);
void fdtd_curl_coefs(const GridGeom &g, int storage, double sE, double sD, double sH, float ch[3], float cd[3]);
float fdtd_jz_stored(float jz, int storage, float eps0, double sD);
float fdtd_jz_at(const float *jz, int jz_len, int jz_limit, int jz_mode, int n);
void fdtd_auto_scales(const float *jz, int jz_len, float eps0, const FdtdExt &e, double *sE, double *sD, double *sH);
double fdtd_field_factor(int storage, float mu0, float eps0, double sE, double sD, double sH, int field);
size_t fdtd_storage_bytes(int storage);
void fdtd_to_storage(int storage, const float *in, size_t n, double factor, void *out);
void fdtd_from_storage(int storage, const void *in, size_t n, double factor, float *out);
// Row-pitched host images of a field (rows of nx values `pitch` apart,
// padding zeroed) and of an id array, for one contiguous device copy.
void fdtd_to_storage_pitched(int storage, const float *in, int nx, size_t rows, int pitch, double factor, void *out);
void fdtd_from_storage_pitched(int storage, const void *in, int nx, size_t rows, int pitch, double factor, float *out);
void fdtd_pitch_bytes(const unsigned char *in, int nx, size_t rows, int pitch, unsigned char *out);
// First cell whose material id is not below nmat; n: none.
size_t fdtd_first_bad_id(const unsigned char *ids, size_t n, int nmat);
int fdtd_check_ext(const FdtdExt &e);

// Phantom input (fdtd_phantom.cpp).  phantom_read_table fills a 95-row
// {sigma, eps_s, eps_inf, tau} table and returns the rows read;
// phantom_read_slice fills nx*ny ids of one PGM slice and returns the
// largest code; both return a negative FDTD_E* code with a message in err.
#include <string>
#include <vector>
int phantom_read_table(const char *path, float *specs, std::string &err);
int phantom_read_slice(const char *path, int nx, int ny, int mode, unsigned char *ids, std::vector<char> &buf,
                       std::string &err);
int fdtd_check_sources(int nx, int ny, int nz, int nsrc, const int *xyz);

// Device state of one grid on the drop-in path (the reference's FdtdField
// arrays, fdtd.h:37-54) and its probe buffers; shared by fdtd_dropin_solve
// (which allocates it) and fdtd_dropin_solve_noalloc (which carves it from a
// static device array).
struct DropinState {
    float *E[3][3], *D[3][3], *H[3];
    float *mat[4];                 // sigma, eps_s, eps_inf, tau per cell
    float *rp[6];
    int *probes = nullptr;         // nprobe x (field, i, j, k)
    double *probe_out = nullptr;   // steps x nprobe
};
// Argument checks of the drop-in solve; fills the effective FdtdExt.
int dropin_check(const FdtdParams *p, const FdtdExt *ext, const FdtdInstance *in, const double *probes_host,
                 FdtdExt *out);
// Uploads the symbols, runs inst->steps steps of the five entry points on
// `stream` over state whose fields start at zero, copies the probe rows to
// probes_host and waits for the stream.
int dropin_run(const FdtdParams *p, const FdtdExt &e, const FdtdInstance *in, const DropinState &st,
               double *probes_host, hipStream_t stream);
int fdtd_check_probes(int nx, int ny, int nz, int nprobe, const int *probes);
// Largest |value| of each probe over `rows` rows of a series (SI units, row
// major, nprobe per row), in stored units (divided by its field's storage
// factor).  Returns how many probes saw a signal (peak > 0) that peaked
// below fp16's smallest normal number under fp16 storage (0 for the other
// storages).
int fdtd_probe_peaks(int storage, const double *series, int rows, int nprobe, const int *fields, const double *factor,
                     double *peak);

#define HIP_TRY(call)                                              \
    do {                                                           \
        hipError_t e_ = (call);                                    \
        if (e_ != hipSuccess) return fdtd_hip_fail(e_, #call);     \
    } while (0)
