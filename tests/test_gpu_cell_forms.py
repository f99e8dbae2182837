"""Which kernel steps a grid, and the two kernels against each other where the
choice or its index arithmetic is at a limit."""
import numpy as np
import pytest
import torch

import fdtd_amd as F

pytestmark = pytest.mark.gpu

DT, DX = 3.8105118e-12, 2.0e-3
MU0, EPS0 = 1.2566371e-06, 8.841941e-12


def _long_row(shape, tiled):
    """Steps a grid of few, very long rows from random fields; its nine fields."""
    nx, ny, nz = shape
    rng = np.random.default_rng(list(shape))
    with F.Context(F.make_params(shape, DT, DX, mu0=MU0, eps0=EPS0), tile_y=4 if tiled else 0) as ctx:
        assert ctx.by_cells() == (not tiled)
        table = np.asarray([(0.0, 1.0, 1.0, 0.0), (0.8, 55.0, 40.0, 8e-12)], np.float32)
        ctx.set_materials(rng.integers(0, 2, (nz, ny, nx), np.uint8), table)
        ctx.set_sources(np.asarray([(nx - 1, 1, 1), (nx // 2, ny - 1, 1)], np.int32), np.ones(4, np.float32))
        for f in range(3, 9):
            ctx.set(f, 0, rng.random((nz, ny, nx), np.float32) - 0.5)
        ctx.run(3)
        out = torch.empty((9, nz, ny, nx), device="cuda")
        ctx.snapshot(out.data_ptr())
        torch.cuda.synchronize()
    return out


def test_very_long_rows():
    """Rows of tens of thousands of tiles: a tile's row is its number divided
    by that count."""
    shape = (1900757, 3, 3)
    print(f"\nlong rows {shape}", flush=True)
    a, b = _long_row(shape, False), _long_row(shape, True)
    for f in range(9):
        assert torch.equal(a[f].view(torch.int32), b[f].view(torch.int32)), F.FIELDS[f]
    assert a.isfinite().all() and (a.abs().amax(dim=(1, 2, 3)) > 0).all()


@pytest.mark.filterwarnings("ignore::fdtd_amd.PrecisionWarning")
@pytest.mark.parametrize("graph_steps", [0, 7])
def test_batch_cells_and_tiles_together(graph_steps):
    """A batch whose grids step partly in tiles (graphs that count the steps on
    the device) and partly in groups (step numbers from the host): runs that
    are no multiple of a graph's steps, and grids of both kinds that join late
    and end inside a run."""
    from tests.test_gpu_batch import assert_same, make_case, single
    deep = 60001   # more planes than cell_step takes
    insts = [make_case(600, (3, 4, deep), 4, 41), make_case(601, (30, 20, 25), 5, 77),
             make_case(602, (3, 3, deep), 3, 23, F.STORE_F16), make_case(603, (66, 9, 12), 6, 19, F.STORE_F16),
             make_case(604, (3, 4, deep), 4, 66), make_case(605, (33, 17, 20), 4, 90)]
    print(f"\ncells and tiles, {graph_steps} steps a graph", flush=True)
    refs = [single(x) for x in insts]
    with F.Batch(8 << 30) as b:
        b.set_shape(graph_steps=graph_steps)
        ids = [b.add(x) for x in insts[:4]]
        assert [b.by_cells(i) for i in ids] == [False, True, False, True]
        b.run(13)
        ids += [b.add(x) for x in insts[4:]]
        b.run(1)
        b.run(45)                      # both early tiled grids end inside
        assert b.info()["running"] == 3
        b.run(75)
        assert b.info()["running"] == 0
        for q, (i, x) in enumerate(zip(ids, insts)):
            assert_same(b, i, x, refs[q], f"grid {q} {x.shape}")
        b.remove(ids[1])               # only tiles, then none running
        last = b.add(insts[0])
        b.run(50)
        assert_same(b, last, insts[0], refs[0], "tiles alone")


@pytest.mark.parametrize("fixed", [False, True])
def test_batch_autotune_without_cell_grids_keeps_the_choice(fixed):
    """Where no grid may step by cells there is nothing to choose: grids that
    are added later step as they would without the autotuner."""
    from tests.test_gpu_batch import make_case
    with F.Batch(2 << 30) as b:
        if fixed:
            b.set_shape(tile_y=4, kchunk=8)
        for _ in range(3):
            deep = b.add(make_case(610, (3, 3, 60001), 3, 9))
            print(f"\nautotune in tiles, fixed={fixed}", flush=True)
            b.autotune(trial_steps=1)
            assert not b.by_cells(deep)
            small = b.add(make_case(611, (20, 20, 20), 3, 9))
            assert b.by_cells(small) == (not fixed)
            b.run(9)
            b.remove(small)
            b.remove(deep)


def test_step_that_cannot_be_launched_is_not_counted():
    """A step whose launch the runtime refuses (here: on a stream whose capture
    is no longer valid) leaves the context as it was."""
    import ctypes as C

    from fdtd_amd import hip
    rt = hip.rt()
    rt.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    rt.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    out = []
    for refuse in (False, True):
        with F.Context(F.make_params((20, 18, 16), DT, DX, mu0=MU0, eps0=EPS0)) as ctx:
            ctx.set_sources(np.asarray([(9, 8, 7)], np.int32), np.linspace(1.0, 2.0, 9).astype(np.float32))
            ctx.set_probes(np.asarray([(8, 9, 8, 7), (3, 8, 8, 7)], np.int32), 9)
            assert ctx.by_cells()
            ctx.run(4)
            hip.sync()
            if refuse:
                s, graph = hip.Stream(), C.c_void_p()
                hip.ok(rt.hipStreamBeginCapture(s.handle, 1), "begin capture")   # thread-local
                assert rt.hipStreamSynchronize(s.handle) != 0                    # ends its validity
                with pytest.raises(F.FdtdError):
                    ctx.step(s.handle)
                rt.hipStreamEndCapture(s.handle, C.byref(graph))
                s.destroy()
                rt.hipGetLastError()
                assert F.lib().fdtd_ctx_steps_done(ctx._h) == 4 and len(ctx.probes()) == 4
            ctx.run(5)
            out.append((ctx.probes(), ctx.get(8)))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert np.abs(out[0][0]).max() > 0


def _mur(h, dt, rpf, rpn, tn, sn, sf):
    """q and x of a face's new value q * x, in fp32 (fdtd_calculations.cu:216-428)."""
    f = np.float32
    k = f(MU0) * f(EPS0)
    rf, rn = np.sqrt(k * rpf), np.sqrt(k * rpn)
    h, dt = f(h), f(dt)
    return f(1) / (dt + h * rf), ((dt - h * rn) * tn + (dt + h * rn) * sn) - (dt - h * rf) * sf


@pytest.mark.parametrize("nx", [96, 65])
@pytest.mark.parametrize("tile_y", [0, 4])
def test_fp16_faces_round_as_stated(nx, tile_y):
    """Faces of the Mur kernel round their fp16 product once; x faces that a
    tile updates (all but the high ones of a row that starts a tile) by way of
    fp32; and the one-lane-per-cell step as the tiles do."""
    ny, nz = 260, 250
    rng = np.random.default_rng([nx, tile_y])
    rps = [rng.uniform(1.0, 3.0, n).astype(np.float32) for n in (2 * ny * nz, nx * 2 * nz, nx * ny * 2) * 2]
    with F.Context(F.make_params((nx, ny, nz), DT, DX, mu0=MU0, eps0=EPS0), storage=F.STORE_F16, scales=(1.0, 1.0, 1.0),
                   tile_y=tile_y) as ctx:
        assert ctx.by_cells() == (tile_y == 0)
        ctx.set_rp(rps)
        for f in range(6, 9):
            ctx.set(f, 0, rng.uniform(-1, 1, (nz, ny, nx)).astype(np.float32))
        old = [ctx.get(f) for f in range(6, 9)]
        ctx.step()
        new = [ctx.get(f) for f in range(6, 9)]
    inner = slice(1, -1)
    rpy, rpye = rps[1].reshape(nz, 2, nx), rps[4].reshape(nz, 2, nx)
    rpx, rpxe = rps[0].reshape(nz, ny, 2), rps[3].reshape(nz, ny, 2)
    faces = []   # name, stored, (q, x), rounds once
    for name, j, jn, rf, rn in (("Ex y0", 0, 1, rpy[:, 0], rpy[:, 1]), ("Ex y1", -1, -2, rpye[:, 1], rpye[:, 0])):
        s = (inner, slice(0, -1))
        e = [a[:, j][s] for a in (new[0], old[0])] + [a[:, jn][s] for a in (new[0], old[0])]
        faces.append((name, e[0], _mur(DX, DT, rf[s], rn[s], e[2], e[3], e[1]), True))
    for name, i, im, rf, rn in (("Ez x0", 0, 1, rpx[..., 0], rpx[..., 1]), ("Ez x1", -1, -2, rpxe[..., 1], rpxe[..., 0])):
        s = (inner, inner)
        e = [a[:, :, i][s] for a in (new[2], old[2])] + [a[:, :, im][s] for a in (new[2], old[2])]
        faces.append((name, e[0], _mur(DX, DT, rf[s], rn[s], e[2], e[3], e[1]), i == -1 and nx == 65))
    for name, got, (q, x), once in faces:
        one = (q.astype(np.float64) * x.astype(np.float64)).astype(np.float16).astype(np.float32)
        two = (q * x).astype(np.float16).astype(np.float32)
        want = one if once else two
        assert np.array_equal(got, want), f"{name}: {np.count_nonzero(got != want)} cells"
        if nx == 96 and name == "Ez x0":
            assert (one != two).any()   # the two differ somewhere in these inputs


@pytest.mark.parametrize("first", [31, 32, 64, 95, 127])
def test_zero_terms_of_high_material_ids(first):
    """Materials of every id skip their zero terms, and no other does: the same
    bits as with every operand loaded, in a grid that holds them all."""
    shape = (70, 40, 30)
    nx, ny, nz = shape
    rng = np.random.default_rng(first)
    table = np.asarray([(0.8, 55.0, 40.0, 8e-12)] * 128, np.float32)
    table[first] = (0.0, 1.0, 1.0, 0.0)
    ids = np.full((nz, ny, nx), first, np.uint8)
    ids[8:20, 10:30, 20:60] = rng.integers(0, 128, (12, 20, 40))
    jz = rng.uniform(-1, 1, 60).astype(np.float32)
    out = []
    for load in (0, 1):
        with F.Context(F.make_params(shape, DT, DX, mu0=MU0, eps0=EPS0), load_zero_terms=load) as ctx:
            assert ctx.by_cells()
            ctx.set_materials(ids, table)
            ctx.set_sources(np.asarray([(30, 20, 15), (5, 5, 5)], np.int32), jz)
            ctx.run(60)
            out.append([ctx.get(f) for f in range(9)])
    for f, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), F.FIELDS[f]


def _forms():
    from tests.test_cell_tiles import FORMS
    for q, (shape, esz, _) in enumerate(FORMS):
        yield shape, (F.STORE_F32, F.STORE_F32, F.STORE_F32_FAST)[q % 3] if esz == 4 else (F.STORE_F16, F.STORE_BF16)[q % 2]


@pytest.mark.filterwarnings("ignore::fdtd_amd.PrecisionWarning")
@pytest.mark.parametrize("shape,storage", list(_forms()))
def test_every_form_equals_tiles(shape, storage):
    """Each form and tile width of the one-lane-per-cell step (which of them a
    grid takes is pinned in test_cell_tiles.py) against the tiled step."""
    from tests.test_gpu_cell import _run
    from tests.helpers import bits_equal, first_diff
    for tile_y in (0, 4):
        with F.Context(F.make_params(shape, DT, DX, mu0=MU0, eps0=EPS0), storage=storage, tile_y=tile_y) as ctx:
            assert ctx.by_cells() == (tile_y == 0)
    print(f"\n{shape} storage {storage}", flush=True)
    a, pa = _run(shape, storage, 4, False)
    b, pb = _run(shape, storage, 4, True)
    for key in a:
        assert bits_equal(a[key], b[key]), f"{F.FIELDS[key[0]]} level {key[1]}: {first_diff(a[key], b[key])}"
    assert np.array_equal(pa.view(np.uint64), pb.view(np.uint64))
    assert np.isfinite(pa).all() and np.abs(pa).max() > 0


@pytest.mark.parametrize("when", ["never", "before", "after", "late", "autotune"])
@pytest.mark.filterwarnings("ignore::fdtd_amd.PrecisionWarning")
def test_batch_shape_fixed_at_any_time(when):
    """A batch staggers a grid's arrays for the kernel that steps it; a grid that
    has not stepped follows a later choice, one that has keeps its place."""
    from tests.test_gpu_batch import assert_same, make_case, single
    insts = [make_case(620, (96, 110, 110), 5, 21), make_case(621, (100, 128, 90), 4, 18, F.STORE_F16), make_case(622, (30, 20, 25), 4, 25)]
    refs = [single(x) for x in insts]
    print(f"\nshape fixed {when}", flush=True)
    with F.Batch(1 << 30) as b:
        if when == "before":
            b.set_shape(tile_y=4, kchunk=8)
        ids = [b.add(x) for x in insts[:2]]
        if when == "after":
            b.set_shape(tile_y=2, kchunk=6)
        if when == "autotune":
            b.autotune(trial_steps=1)
        b.run(7)
        ids.append(b.add(insts[2]))
        if when == "late":
            b.set_shape(tile_y=8, kchunk=4)
        if when != "autotune":
            assert [b.by_cells(i) for i in ids] == [when == "never"] * 3
        b.run(30)
        for q, (i, x) in enumerate(zip(ids, insts)):
            assert_same(b, i, x, refs[q], f"grid {q} {x.shape}")


def test_comparisons_with_tiles_have_two_kernels_to_compare():
    """The grids of test_gpu_cell.py step by cells by default and in tiles with
    tile_y fixed, in every storage form."""
    from tests import test_gpu_cell as T
    past = [m.args[1] for m in T.test_cells_equal_tiles_past_the_cache.pytestmark if m.name == "parametrize"][0]
    both = [(s, st) for s in T.SHAPES for st in (F.STORE_F32, F.STORE_F16, F.STORE_BF16, F.STORE_F32_FAST)] + past
    for shape, storage in both:
        for tile_y in (0, 4):
            with F.Context(F.make_params(shape, DT, DX, mu0=MU0, eps0=EPS0), storage=storage, tile_y=tile_y) as ctx:
                assert ctx.by_cells() == (tile_y == 0), (shape, storage)


@pytest.mark.parametrize("tile_y", [0, 4])
def test_autotune_that_cannot_time_cells_keeps_the_choice(tile_y):
    """With more probes than the step by cells takes there is only one kernel to
    time; the choice is the context's own again once it has fewer."""
    with F.Context(F.make_params((20, 18, 16), DT, DX, mu0=MU0, eps0=EPS0), tile_y=tile_y) as ctx:
        for _ in range(3):
            ctx.set_probes(np.zeros((40001, 4), np.int32), 1)
            assert not ctx.by_cells()
            print(f"\nautotune with 40001 probes, tile_y {tile_y}", flush=True)
            ctx.autotune(trial_steps=1)
            ctx.set_probes(np.zeros((1, 4), np.int32), 1)
            assert ctx.by_cells() == (tile_y == 0)


@pytest.mark.parametrize("args,cells", [(("--shape", "64x4x8"), False), ((), True)])
def test_bench_lines_name_the_kernels_that_ran(args, cells):
    from tests.test_gpu_bench import _bench
    d = _bench("--workload", "plain_small", "--steps", "8", "--warmup", "2", "--advance", "8", "--no-cpu-baseline",
               "--timing-launches", "8", *args)
    launch = d["config"]["launch"]
    assert launch["by_cells"] == cells and ("tile_y" in launch) == (not cells)
    assert d["roofline"]["kernel"] == ("cell_step" if cells else "fused_step")
    d = _bench("--workload", "batched", "--no-sequential", *args)
    c, kernel = d["config"], d["roofline"]["kernel"]
    assert ("cell_batch" in kernel) == (c["grids_by_cells"] > 0) and ("fused_batch" in kernel) == (c["grids_by_cells"] < 64)
    assert (c["tile_y"] is None) == (c["grids_by_cells"] == 64)
    if not cells:
        assert c["grids_by_cells"] == 0 and (c["tile_y"], c["kchunk"]) == (4, 8)


def test_batch_bytes_of_a_grid():
    """Grids by cells lie close together in the arena (their groups have to fit
    the Infinity Cache); instance_bytes holds for either way of stepping."""
    from tests.test_gpu_batch import make_case
    x = make_case(630, (96, 110, 110), 5, 3)
    for fixed in (False, True):
        with F.Batch(x.nbytes() * 2) as b:
            if fixed:
                b.set_shape(tile_y=4, kchunk=8)
            b.add(x)
            used = b.info()["used_bytes"]
            assert used == x.nbytes() if fixed else used + 23 * 65000 * 4 < x.nbytes()
            b.add(x)
            b.run(3)


@pytest.mark.filterwarnings("ignore::fdtd_amd.PrecisionWarning")
@pytest.mark.parametrize("shape,storage", [((3, 3, 4000), F.STORE_F32), ((64, 4, 5000), F.STORE_F32), ((10, 10, 5000), F.STORE_F16),
                                           ((130, 3, 4000), F.STORE_BF16), ((130, 3, 10000), F.STORE_F32)])
def test_many_small_planes_equal_tiles(shape, storage):
    """Planes that take only as many blocks as they have tiles (pinned in
    test_cell_tiles.py), with their faces and probes."""
    from tests.test_gpu_cell import _run
    from tests.helpers import bits_equal, first_diff
    print(f"\nmany small planes {shape} storage {storage}", flush=True)
    a, pa = _run(shape, storage, 4, False)
    b, pb = _run(shape, storage, 4, True)
    for key in a:
        assert bits_equal(a[key], b[key]), f"{F.FIELDS[key[0]]} level {key[1]}: {first_diff(a[key], b[key])}"
    assert np.array_equal(pa.view(np.uint64), pb.view(np.uint64))


def test_batch_with_many_small_planes():
    from tests.test_gpu_batch import assert_same, make_case, single
    insts = [make_case(640, (3, 3, 5000), 4, 12), make_case(641, (30, 20, 25), 5, 12), make_case(642, (64, 4, 4000), 4, 9),
             make_case(643, (24, 24, 24), 5, 12)]
    refs = [single(x) for x in insts]
    print("\nbatch with many small planes", flush=True)
    with F.Batch(2 << 30) as b:
        ids = [b.add(x) for x in insts]
        assert all(b.by_cells(i) for i in ids)
        b.run(12)
        for q, (i, x) in enumerate(zip(ids, insts)):
            assert_same(b, i, x, refs[q], f"grid {q} {x.shape}")


@pytest.mark.filterwarnings("ignore::fdtd_amd.PrecisionWarning")
def test_batch_a_step_at_a_time_past_the_cache():
    """Several groups, whose state is past the Infinity Cache, a step at a time:
    one launch for the small grids of a storage form, in the form for states
    past the cache; with two steps at a time in groups; and a larger grid."""
    from tests.test_gpu_batch import assert_same, make_case, single
    insts = [make_case(650, (100, 98, 96), 4, 9), make_case(651, (96, 90, 100), 5, 6), make_case(652, (90, 100, 104), 4, 9),
             make_case(653, (96, 110, 90), 4, 9, F.STORE_F16), make_case(654, (70, 90, 130), 4, 7, F.STORE_F16),
             make_case(655, (130, 100, 110), 4, 8), make_case(656, (60, 100, 90), 4, 9, F.STORE_F32_FAST), make_case(657, (20, 20, 20), 4, 3, F.STORE_F16)]
    print("\nbatch a step at a time", flush=True)
    refs = [single(x) for x in insts]
    with F.Batch(4 << 30) as b:
        ids = [b.add(x) for x in insts]
        for n in (1, 1, 2, 1, 1, 1, 2):
            b.run(n)
        for q, (i, x) in enumerate(zip(ids, insts)):
            assert_same(b, i, x, refs[q], f"grid {q} {x.shape}")
