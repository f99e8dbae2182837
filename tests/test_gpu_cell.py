"""The one-lane-per-cell step (small grids) against the tiled step and the
oracle: widths at and around the tile edges, the smallest grids, faces seen
by probes, sources on the upper faces, every storage form."""
import numpy as np
import pytest

import fdtd_amd as F
from tests.helpers import bits_equal, first_diff

pytestmark = pytest.mark.gpu

DT, DX = 3.8105118e-12, 2.0e-3
MU0, EPS0 = 1.2566371e-06, 8.841941e-12

SHAPES = [(3, 3, 3), (4, 9, 5), (33, 5, 4), (64, 6, 5), (65, 9, 6), (97, 12, 7), (31, 66, 12), (130, 17, 9)]


def _probes(shape):
    """Every field inside, at the corners of the box and on each face."""
    nx, ny, nz = shape
    at = [(nx // 2, ny // 2, nz // 2), (0, 0, 0), (nx - 1, ny - 1, nz - 1), (0, ny // 2, nz // 2),
          (nx - 1, ny // 2, nz // 2), (nx // 2, 0, nz // 2), (nx // 2, ny - 1, nz // 2), (nx // 2, ny // 2, 0),
          (nx // 2, ny // 2, nz - 1), (1, 1, 1), (nx - 2, ny - 2, nz - 2), (0, 1, 0)]
    return np.asarray([(f, *c) for c in at for f in range(9)], np.int32)


def _run(shape, storage, steps, tiled):
    rng = np.random.default_rng([*shape, storage])
    nx, ny, nz = shape
    table = np.asarray([(0.0, 1.0, 1.0, 0.0), (0.8, 55.0, 40.0, 8e-12), (0.1, 4.0, 3.0, 0.0)], np.float32)
    ids = rng.integers(0, 3, (nz, ny, nx)).astype(np.uint8)
    rps = [rng.uniform(1.0, 3.0, n).astype(np.float32) for n in (2 * ny * nz, nx * 2 * nz, nx * ny * 2) * 2]
    src = np.asarray([(nx - 1, 1, nz // 2), (1, ny - 1, nz - 1), (nx // 2 or 1, ny // 2 or 1, nz // 2)], np.int32)
    jz = rng.uniform(-1.0, 1.0, steps).astype(np.float32)
    probes = _probes(shape)
    with F.Context(F.make_params(shape, DT, DX, 1.1 * DX, 0.9 * DX, MU0, EPS0), storage=storage,
                   tile_y=4 if tiled else 0) as ctx:
        ctx.set_materials(ids, table)
        ctx.set_rp(rps)
        ctx.set_sources(src, jz)
        ctx.set_probes(probes, steps)
        ctx.step()
        ctx.run(steps - 1)
        fields = {(f, lv): ctx.get(f, lv) for f in range(9) for lv in ([0] if 3 <= f < 6 else [0, 1, 2])}
        series = ctx.probes()
    for p, (f, i, j, k) in enumerate(probes):   # a probe's last row is the field's value
        assert np.float32(series[-1, p]) == fields[(f, 0)][k, j, i], f"probe {F.FIELDS[f]} at {(i, j, k)}"
    return fields, series


@pytest.mark.filterwarnings("ignore::fdtd_amd.PrecisionWarning")
@pytest.mark.parametrize("storage", [F.STORE_F32, F.STORE_F16, F.STORE_BF16, F.STORE_F32_FAST])
@pytest.mark.parametrize("shape", SHAPES)
def test_cells_equal_tiles(shape, storage):
    a, pa = _run(shape, storage, 7, False)
    b, pb = _run(shape, storage, 7, True)
    for key in a:
        assert bits_equal(a[key], b[key]), f"{F.FIELDS[key[0]]} level {key[1]}: {first_diff(a[key], b[key])}"
    assert np.array_equal(pa.view(np.uint64), pb.view(np.uint64))
    assert np.isfinite(pa).all() and np.abs(pa).max() > 0


@pytest.mark.filterwarnings("ignore::fdtd_amd.PrecisionWarning")
@pytest.mark.parametrize("shape", [(96, 37, 30), (65, 40, 33)])   # x-high faces in the tile, and left to the Mur kernel
def test_cells_equal_tiles_f16_faces(shape):
    """fp16 faces round once or twice as the tiled step does; it takes many
    face updates to tell."""
    a, pa = _run(shape, F.STORE_F16, 90, False)
    b, pb = _run(shape, F.STORE_F16, 90, True)
    for key in a:
        assert bits_equal(a[key], b[key]), f"{F.FIELDS[key[0]]} level {key[1]}: {first_diff(a[key], b[key])}"


@pytest.mark.filterwarnings("ignore::fdtd_amd.PrecisionWarning")
@pytest.mark.parametrize("shape,storage", [((65, 90, 420), F.STORE_F32), ((3, 300, 600), F.STORE_F32),
                                           ((64, 64, 1300), F.STORE_F32), ((130, 127, 260), F.STORE_F32_FAST),
                                           ((65, 90, 620), F.STORE_F16), ((130, 160, 1000), F.STORE_BF16),
                                           ((70, 91, 420), F.STORE_F32), ((64, 64, 800), F.STORE_F32),
                                           ((100, 121, 900), F.STORE_F16)])
def test_cells_equal_tiles_past_the_cache(shape, storage):
    """States larger than the Infinity Cache, whose lanes take their x
    neighbours from each other: one and more waves a row, a few lanes of one,
    two rows a wave, a single last row, with cached and with streaming accesses."""
    a, pa = _run(shape, storage, 4, False)
    b, pb = _run(shape, storage, 4, True)
    for key in a:
        assert bits_equal(a[key], b[key]), f"{F.FIELDS[key[0]]} level {key[1]}: {first_diff(a[key], b[key])}"
    assert np.array_equal(pa.view(np.uint64), pb.view(np.uint64))
    assert np.isfinite(pa).all() and np.abs(pa).max() > 0


@pytest.mark.parametrize("shape", [(3, 9, 5), (33, 20, 11), (64, 24, 9)])
def test_cells_equal_the_oracle(shape):
    from oracle import oracle as O
    rng = np.random.default_rng(list(shape))
    nx, ny, nz = shape
    table = np.asarray([(0.0, 1.0, 1.0, 0.0), (0.8, 55.0, 40.0, 8e-12)], np.float32)
    ids = rng.integers(0, 2, (nz, ny, nx)).astype(np.uint8)
    src, jz = np.asarray([(1, 2, 1), (nx - 1, ny - 1, nz - 1)], np.int32), rng.uniform(-1, 1, 9).astype(np.float32)
    probes = _probes(shape)
    ctx = F.Context(F.make_params(shape, DT, DX, mu0=MU0, eps0=EPS0))
    ctx.set_materials(ids, table)
    ctx.set_sources(src, jz)
    ctx.set_probes(probes, 9)
    sim = O.Sim(shape, DT, DX, DX, DX, MU0, EPS0, prec=32)
    t = table[ids.astype(np.int64)]
    sim.set_materials(t[..., 0], t[..., 1], t[..., 2], t[..., 3])
    sim.set_sources(src, jz, jz_mode=1)
    for f in range(9):                          # random start: every operand non-zero
        for lv in ([0] if 3 <= f < 6 else [0, 1, 2]):
            v = rng.uniform(-1, 1, (nz, ny, nx)).astype(np.float32)
            ctx.set(f, lv, v)
            sim.set(f, lv, v)
    ctx.run(9)
    ref = sim.run(9, probes)
    for f in range(9):
        for lv in ([0] if 3 <= f < 6 else [0, 1, 2]):
            a, b = ctx.get(f, lv), sim.get(f, lv)
            assert bits_equal(a, b), f"{F.FIELDS[f]} level {lv}: {first_diff(a, b)}"
    assert np.array_equal(ctx.probes().astype(np.float32).view(np.uint32), ref.astype(np.float32).view(np.uint32))


@pytest.mark.filterwarnings("ignore::fdtd_amd.PrecisionWarning")
def test_batch_groups_equal_single_grids():
    """Grids of a batch stepped in groups: several grids of one storage form
    in a launch, forms in groups of their own, probes past the planes' blocks,
    grids that join and finish inside a run, 32- and 64-lane tiles."""
    from tests.test_gpu_batch import assert_same, make_case, single
    cases = [((20, 24, 28), 4, 17, F.STORE_F32, F.JZ_STEP, False, 6), ((33, 17, 40), 12, 70, F.STORE_F32, F.JZ_HOLD3, True, 64),
             ((66, 9, 12), 6, 45, F.STORE_F16, F.JZ_STEP, True, 6), ((96, 16, 16), 5, 33, F.STORE_F16, F.JZ_STEP, False, 0),
             ((16, 16, 16), 5, 9, F.STORE_F32_FAST, F.JZ_STEP, False, 6), ((48, 40, 20), 8, 40, F.STORE_BF16, F.JZ_STEP, True, 6),
             ((65, 5, 7), 4, 33, F.STORE_F32, F.JZ_STEP, False, 9), ((3, 3, 3), 2, 50, F.STORE_F32, F.JZ_STEP, False, 64)]
    insts = [make_case(300 + q, *c[:6], nprobe=c[6]) for q, c in enumerate(cases)]
    refs = [single(x) for x in insts]
    with F.Batch(1 << 30) as b:
        ids = [b.add(x) for x in insts[:5]]
        b.run(11)
        ids += [b.add(x) for x in insts[5:]]
        b.run(1)
        b.run(90)
        for q, (i, x) in enumerate(zip(ids, insts)):
            assert_same(b, i, x, refs[q], f"grid {q} {x.shape}")


@pytest.mark.parametrize("count,edge", [(3, 100), (2, 148)])   # two groups of fp32 grids; one group and one grid in tiles
def test_batch_groups_and_tiles(count, edge):
    from tests.test_gpu_batch import assert_same, make_case, single
    insts = [make_case(400 + q, (edge + q, edge, edge - 3 * q), 5, 40 + q) for q in range(count)]
    refs = [single(x) for x in insts]
    with F.Batch(4 << 30) as b:
        ids = [b.add(x) for x in insts]
        b.run(45)
        for q, (i, x) in enumerate(zip(ids, insts)):
            assert_same(b, i, x, refs[q], f"grid {q} {x.shape}")


@pytest.mark.filterwarnings("ignore::fdtd_amd.PrecisionWarning")
@pytest.mark.parametrize("shape,storage", [((96, 130, 300), F.STORE_F32), ((64, 128, 420), F.STORE_F32), ((130, 127, 260), F.STORE_F32),
                                           ((100, 121, 500), F.STORE_F16), ((100, 121, 900), F.STORE_BF16)])
def test_batch_grids_past_the_cache(shape, storage):
    """Grids that make a group of their own, in the forms past the cache, with
    a small one that ends first and joins again."""
    from tests.test_gpu_batch import assert_same, make_case, single
    insts = [make_case(500, shape, 5, 9, storage), make_case(501, (30, 20, 25), 5, 4, storage)]
    refs = [single(x) for x in insts]
    with F.Batch(4 << 30) as b:
        ids = [b.add(x) for x in insts]
        b.run(5)
        ids.append(b.add(insts[1]))
        b.run(6)
        for i, q in zip(ids, (0, 1, 1)):
            assert_same(b, i, insts[q], refs[q], f"grid {q} {insts[q].shape}")


def test_more_probes_than_blocks_take_tiles():
    """A context with more probes than the launch has room for steps in tiles;
    up to there by cells, with the same series."""
    shape, out = (20, 18, 16), {}
    for n in (40000, 40001):
        probes = np.tile(_probes(shape), (n // 108 + 1, 1))[:n]
        with F.Context(F.make_params(shape, DT, DX, mu0=MU0, eps0=EPS0)) as ctx:
            ctx.set_sources(np.asarray([(9, 8, 7)], np.int32), np.linspace(1.0, 2.0, 9).astype(np.float32))
            ctx.set_probes(probes, 9)
            assert ctx.by_cells() == (n == 40000)
            ctx.run(9)
            out[n] = ctx.probes()[:, :108]
            assert np.array_equal(ctx.probes()[:, 108:216], out[n])
    assert np.array_equal(out[40000], out[40001]) and np.abs(out[40000]).max() > 0
