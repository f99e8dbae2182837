"""Index arithmetic of the one-lane-per-cell step, on the CPU: the header that
the kernels share is compiled for the host and every tile of a plane mapped
to its row and column, for rows of one tile up to millions of cells."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include <cstdio>
#include <cstring>
#include "fdtd_internal.h"
int main()
{
    CellArgs c;
    memset((void *)&c, 0, sizeof c);
    c.nx = c.ny = c.nz = 3;
    if (!cell_args_ok(c)) return 1;
    CellArgs d = c; d.e0[2] = (const char *)0x1001;
    if (cell_args_ok(d)) return 2;
    d = c; d.sy = 129;
    if (cell_args_ok(d)) return 3;
    d = c; d.ids = (const uint8_t *)0x77;
    if (cell_args_ok(d)) return 4;
    d = c; d.run = -1;
    return cell_args_ok(d) ? 5 : 0;
}
"""

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "fdtd_internal.h"
struct Tiles { int bxl, lanes, tiles_x, tiles, run, gx; uint32_t tx_mul, tx_shift; };
int main(int argc, char **argv)
{
    for (int q = 1; q + 3 < argc; q += 4) {   // nx ny form esz
        Tiles a;
        const int nx = atoi(argv[q]), ny = atoi(argv[q + 1]);
        cell_tiles(nx, ny, 3, 0, atoi(argv[q + 2]), (size_t)atoi(argv[q + 3]), a);
        long long bad = 0;
        for (int t = 0; t < a.tiles; t++) bad += cell_tile_row(t, a.tiles_x, a.tx_mul, a.tx_shift) != t / a.tiles_x;
        printf("%d %d %lld\n", a.tiles_x, a.tiles, bad);
    }
    for (unsigned long long d : {2ull, 3ull, 5ull, 7ull, 64ull, 65ull, 641ull, 65535ull, 65537ull, 1ull << 31, (1ull << 31) + 1,
                                 (1ull << 32) - 1}) {
        uint32_t m, s;
        div_consts(d, m, s);
        for (unsigned long long k = 0; k < 4000; k++)
            for (int e = -1; e <= 1; e++) {   // around multiples of d over the whole range
                const uint32_t v = (uint32_t)((0xffffffffull / 3999 * k) / d * d + e);
                if (div_by(v, m, s) != v / d) { printf("%u / %llu\n", v, d); return 1; }
            }
    }
    return 0;
}
"""

# rows of one tile, of a few, and so long that a rounded reciprocal's error adds up to a tile
SHAPES = [(3, 3), (64, 5), (65, 130), (96, 37), (150, 150), (1024, 1024), (85016, 2495), (106023, 1995), (550190, 65),
          (950358, 33), (1900757, 3)]


def _build(tmp_path, text):
    src, exe = tmp_path / "cells.cpp", tmp_path / "cells"
    src.write_text(text)
    subprocess.run(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{ROOT}/include",
                    f"-I{ROOT}/fdtd_amd/csrc", str(src), "-o", str(exe)], check=True)
    return exe


LIMIT = r"""
#include <cstdio>
#include <cstdlib>
#include "fdtd_internal.h"
int main(int argc, char **argv)
{
    for (int q = 1; q + 3 < argc; q += 4) {   // nx ny nz esz
        const int nx = atoi(argv[q]), ny = atoi(argv[q + 1]), nz = atoi(argv[q + 2]), esz = atoi(argv[q + 3]);
        const size_t state = 24 * (size_t)fused_pitch(nx, esz) * ny * nz * esz;
        printf("%d%d ", state <= cell_state_limit(nx, esz) ? 1 : 0, state <= cell_batch_limit(nx, esz) ? 1 : 0);
    }
    return 0;
}
"""

# fp32 grids on either side of where a context's and a batch's tiles are measured to be faster (times in the comments of
# cell_state_limit and cell_batch_limit): whether a context and a batch step them by cells
LIMITS = [((64, 64, 1300), "11"), ((64, 450, 720), "00"), ((128, 300, 230), "11"), ((128, 300, 310), "01"), ((128, 450, 360), "00"),
          ((100, 300, 310), "01"), ((100, 300, 360), "00"), ((192, 192, 192), "11"), ((192, 270, 230), "11"), ((192, 300, 300), "01"),
          ((192, 400, 345), "00"), ((180, 300, 300), "00"), ((256, 256, 256), "11"), ((320, 320, 224), "11"), ((256, 256, 384), "11"),
          ((384, 300, 225), "01"), ((300, 200, 190), "11"), ((300, 250, 220), "00"), ((160, 400, 300), "11"), ((350, 330, 178), "11"),
          ((350, 330, 260), "00"), ((320, 320, 880), "00"), ((24, 24, 24), "11")]


def test_state_limits(tmp_path):
    exe = _build(tmp_path, LIMIT)
    args = [str(v) for shape, _ in LIMITS for v in (*shape, 4)]
    out = subprocess.run([str(exe), *args], capture_output=True, text=True, check=True).stdout.split()
    assert out == [want for _, want in LIMITS]


FORM = r"""
#include <cstdio>
#include <cstdlib>
#include "fdtd_internal.h"
int main(int argc, char **argv)
{
    for (int q = 1; q + 3 < argc; q += 4) {   // nx ny nz esz
        const int nx = atoi(argv[q]), ny = atoi(argv[q + 1]), nz = atoi(argv[q + 2]), esz = atoi(argv[q + 3]);
        const size_t state = 24 * (size_t)fused_pitch(nx, esz) * ny * nz * esz;
        const int form = cell_form(nx, state, esz), l = cell_lanes_log2(nx, form, esz);
        printf("%d %d %d %d\n", state <= cell_state_limit(nx, esz) ? 1 : 0, form, l, cell_block_lanes(form, esz, l));
    }
    return 0;
}
"""

PLANES = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "fdtd_internal.h"
struct Tiles { int bxl, lanes, tiles_x, tiles, run, gx; uint32_t tx_mul, tx_shift; };
int main(int argc, char **argv)
{
    for (int q = 1; q + 4 < argc; q += 5) {   // nx ny nz nprobe esz
        Tiles a;
        const int nx = atoi(argv[q]), ny = atoi(argv[q + 1]), nz = atoi(argv[q + 2]), np = atoi(argv[q + 3]), esz = atoi(argv[q + 4]);
        cell_tiles(nx, ny, nz, np, cell_form(nx, 24 * (size_t)fused_pitch(nx, esz) * ny * nz * esz, esz), esz, a);
        const int gx = a.gx, waves = a.lanes / 64;
        std::vector<int> seen(a.tiles, 0);
        for (int b = 0; b < gx; b++)
            if (const int t = cell_tile(b, a.run); t < a.tiles) seen[t]++;
        for (int t = 0; t < a.tiles; t++)
            if (seen[t] != 1) return 1;
        const int pb = (np + waves - 1) / waves;
        if (nz + (pb + gx - 1) / gx > 65535) return 2;
        printf("%d ", a.run == 0 ? 1 : 0);
    }
    return 0;
}
"""

# (shape, probes, bytes of a value) -> whether a plane takes only as many blocks as it has tiles
PLANE_CASES = [((3, 3, 300), 0, 4, 0), ((3, 3, 10000), 0, 4, 1), ((3, 3, 10000), 40000, 4, 1), ((3, 3, 60000), 40000, 4, 0),
               ((64, 4, 10000), 9, 4, 1), ((130, 3, 10000), 5, 4, 1), ((16, 16, 10000), 0, 4, 0), ((10, 10, 10000), 0, 2, 1),
               ((3, 30, 10000), 0, 4, 0), ((24, 24, 24), 0, 4, 0), ((256, 256, 256), 3, 4, 0)]


def test_every_tile_of_a_plane_has_one_block(tmp_path):
    exe = _build(tmp_path, PLANES)
    args = [str(v) for shape, np_, esz, _ in PLANE_CASES for v in (*shape, np_, esz)]
    r = subprocess.run([str(exe), *args], capture_output=True, text=True)
    assert r.returncode == 0 and [int(v) for v in r.stdout.split()] == [want for *_, want in PLANE_CASES]


# (shape, bytes of a value) -> form (0 near, 1 mid, 2 part, 3 far), log2 of a tile's lanes along x, lanes of a block.
# Every combination that the dispatch has; tests/test_gpu_cell_forms.py steps these grids.
FORMS = [((100, 30, 20), 4, (0, 6, 64)), ((90, 30, 20), 4, (0, 5, 64)), ((65, 90, 420), 4, (1, 5, 64)), ((64, 90, 530), 4, (1, 6, 64)),
         ((70, 91, 620), 4, (3, 5, 64)), ((64, 64, 1300), 4, (3, 6, 256)), ((120, 65, 600), 4, (3, 6, 256)),
         ((100, 30, 20), 2, (0, 6, 64)), ((90, 30, 20), 2, (0, 5, 64)), ((64, 90, 900), 2, (1, 6, 64)), ((100, 121, 330), 2, (1, 6, 64)),
         ((64, 128, 1300), 2, (1, 6, 64)), ((100, 121, 900), 2, (2, 6, 64)), ((64, 91, 1100), 2, (2, 6, 64)),
         ((300, 121, 560), 2, (3, 6, 64))]


def test_forms_and_lanes(tmp_path):
    exe = _build(tmp_path, FORM)
    args = [str(v) for shape, esz, _ in FORMS for v in (*shape, esz)]
    out = subprocess.run([str(exe), *args], capture_output=True, text=True, check=True).stdout.split()
    got = np.asarray([int(v) for v in out]).reshape(-1, 4)
    for (shape, esz, want), (cells, *form) in zip(FORMS, got):
        assert cells == 1 and tuple(form) == want, (shape, esz, form)


MASK = r"""
#include <cstring>
#include "fdtd_internal.h"
int main()
{
    MatCoef lut[kMaxMaterials];
    memset((void *)lut, 0, sizeof lut);
    auto zero = [](int m) { return m * 7 % 11 < 4; };
    for (int m = 0; m < kMaxMaterials; m++) {
        if (zero(m)) continue;
        if (m % 3 == 0) lut[m].a = -0.0f;          // only +0 counts
        else if (m % 3 == 1) lut[m].g3 = 1e-300;
        else lut[m].a = 1e-38f;
    }
    for (int nmat : {1, 31, 32, 33, 64, 95, 97, 128}) {
        const ZeroTerms z = cell_zmask(lut, nmat);
        for (int m = 0; m < kMaxMaterials; m++)
            if (z.has(m) != (m < nmat && zero(m))) return 1 + m;
    }
    return 0;
}
"""


def test_zero_terms_of_every_material(tmp_path):
    assert subprocess.run([str(_build(tmp_path, MASK))]).returncode == 0


def test_launch_refuses_what_the_kernel_would_skip(tmp_path):
    assert subprocess.run([str(_build(tmp_path, CHECK))]).returncode == 0


@pytest.mark.parametrize("esz", [4, 2])
def test_tiles_map_to_rows(tmp_path, esz):
    exe = _build(tmp_path, PROGRAM)
    cases = [(nx, ny, form) for nx, ny in SHAPES for form in (0, 1, 3)]
    args = [str(v) for nx, ny, form in cases for v in (nx, ny, form, esz)]
    out = subprocess.run([str(exe), *args], capture_output=True, text=True, check=True).stdout.split()
    got = np.asarray([int(v) for v in out]).reshape(-1, 3)
    assert len(got) == len(cases)
    for (nx, ny, form), (tiles_x, tiles, bad) in zip(cases, got):
        assert tiles_x * 64 >= nx and tiles >= tiles_x * ((ny + 7) // 8)
        assert bad == 0, f"{nx}x{ny} form {form}: {bad} of {tiles} tiles in a wrong row"
