"""The tiled kernels at sizes that step by cells unless a launch shape is
fixed: zero-term rows through infinities and NaN in a context and in a batch,
the reference's Debye mode in a batch, and z-slabs that exchange halos between
tiled steps; and the infinities in the forms of the step by cells past the
cache."""
import numpy as np
import pytest

import fdtd_amd as F
from fdtd_amd import hip
from fdtd_amd import workloads as W
from tests.helpers import EPS0, MU0, random_materials, random_rp, random_sources, random_state
from tests.test_gpu_batch import assert_same, make_case, single
from tests.test_gpu_zero_terms import _run, _same

pytestmark = [pytest.mark.gpu, pytest.mark.filterwarnings("ignore::fdtd_amd.PrecisionWarning")]

DT, DX = 3.8105118e-12, 2.0e-3


@pytest.mark.parametrize("shape_kw", [{"tile_y": 4}, {"tile_x": 128, "tile_y": 2, "kchunk": 6}, {"tile_y": 8, "kchunk": 16}])
def test_zero_term_rows_through_overflow_in_tiles(shape_kw):
    w = W.plain_small(steps=220)
    print(f"\noverflow in tiles, {shape_kw}", flush=True)
    a, sa = _run(w, 220, 0, debye=F.DEBYE_REF, shape_kw=shape_kw)
    b, sb = _run(w, 220, 1, debye=F.DEBYE_REF, shape_kw=shape_kw)
    c, sc = _run(w, 220, 0, debye=F.DEBYE_REF)
    assert not np.isfinite(a[(8, 0)]).all()
    _same(a, b, "loading")
    assert np.array_equal(sa.view(np.uint64), sb.view(np.uint64))
    for key in a:   # by cells: the same but for which NaN it is
        assert np.array_equal(a[key], c[key], equal_nan=True), key
    assert np.array_equal(sa, sc, equal_nan=True)


def test_zero_term_rows_change_no_bit_in_default_tiles():
    w = W.plain_small(steps=300)
    print("\nzero-term rows, 4 tile rows", flush=True)
    a, sa = _run(w, 300, 0, shape_kw={"tile_y": 4})
    b, sb = _run(w, 300, 1, shape_kw={"tile_y": 4})
    _same(a, b, "fixed")
    assert np.array_equal(sa.view(np.uint64), sb.view(np.uint64))


@pytest.mark.parametrize("debye,steps", [(F.DEBYE_FIXED, 60), (F.DEBYE_REF, 220)])
def test_zero_term_rows_in_a_tiled_batch(debye, steps):
    ws = W.batched_set(count=4, seed=778) if debye == F.DEBYE_FIXED else [W.plain_small(steps=steps)]
    out = []
    for load in (0, 1):
        insts = [F.Instance(w.params, F.make_ext(debye=debye, load_zero_terms=load), w.ids, w.table, w.sources, w.jz,
                            min(w.steps, steps), w.probes) for w in ws]
        print(f"\ntiled batch, load {load}", flush=True)
        with F.Batch(int(sum(x.nbytes() for x in insts) * 1.05) + (32 << 20)) as b:
            b.set_shape(tile_y=4, kchunk=8)
            ids = [b.add(x) for x in insts]
            assert not any(b.by_cells(i) for i in ids)
            b.run(steps)
            out.append([(b.probes(i), b.get(i, 8), b.get(i, 2, 1)) for i in ids])
    assert debye == F.DEBYE_FIXED or not np.isfinite(out[0][0][1]).all()
    for q, (x, y) in enumerate(zip(*out)):
        for u, v in zip(x, y):
            assert np.array_equal(np.ascontiguousarray(u).view(np.uint8), np.ascontiguousarray(v).view(np.uint8)), q


def test_tiled_batch_in_the_reference_debye_mode():
    insts = [make_case(700, (24, 20, 22), 5, 12, debye=F.DEBYE_REF), make_case(701, (70, 12, 9), 4, 15, debye=F.DEBYE_REF)]
    refs = [single(x) for x in insts]
    print("\ntiled batch, reference Debye mode", flush=True)
    with F.Batch(256 << 20) as b:
        b.set_shape(tile_y=4, kchunk=8)
        ids = [b.add(x) for x in insts]
        b.run(15)
        for q, (i, x) in enumerate(zip(ids, insts)):
            assert_same(b, i, x, refs[q], f"grid {q}")


@pytest.mark.parametrize("shape", [(64, 90, 530), (70, 91, 420), (64, 64, 1300), (70, 91, 620)])
def test_zero_terms_through_overflow_past_the_cache(shape):
    """mid and far, 64 and 32 lanes along x: fields that become infinite and NaN
    where cells skip their zero terms."""
    nx, ny, nz = shape
    ids = np.zeros((nz, ny, nx), np.uint8)
    ids[nz // 3:nz // 2, ny // 3:ny // 2, nx // 3:nx // 2] = 1
    table = np.asarray([(0.0, 1.0, 1.0, 0.0), (0.8, 55.0, 40.0, 8e-12)], np.float32)
    print(f"\noverflow past the cache {shape}", flush=True)
    out = []
    for load in (0, 1):
        with F.Context(F.make_params(shape, DT, DX, mu0=MU0, eps0=EPS0), debye=F.DEBYE_REF, load_zero_terms=load) as ctx:
            assert ctx.by_cells()
            ctx.set_materials(ids, table)
            ctx.set_sources(np.asarray([(nx // 2, ny // 2, nz // 4)], np.int32), np.sin(np.arange(64) * 0.3).astype(np.float32))
            ctx.run(170)
            out.append([ctx.get(f) for f in range(9)])
    assert not np.isfinite(out[0][8]).all() and np.isfinite(out[0][8]).any()
    for f, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), F.FIELDS[f]


@pytest.mark.parametrize("storage,tile_y", [(F.STORE_F32, 4), (F.STORE_F32, 8), (F.STORE_F16, 4)])
def test_tiled_slabs_equal_whole_grid(storage, tile_y):
    """Slabs whose steps are tiled, with a halo exchange before each, against
    the whole grid in tiles: every real plane, field and ring level."""
    shape, cuts = (37, 29, 40), (0, 13, 27, 40)
    nx, ny, nz = shape
    rng = np.random.default_rng(31)
    ids, table = random_materials(rng, shape)
    rps = random_rp(rng, shape)
    src = random_sources(rng, shape, 6)
    src[0, 2], src[1, 2] = cuts[1] - 1, cuts[1]
    jz = rng.uniform(-2, 2, 30).astype(np.float32)
    st = random_state(rng, shape) if storage == F.STORE_F32 else {}
    planes = [r.reshape(s) for r, s in zip(rps, [(nz, ny, 2), (nz, 2, nx), (2, ny, nx)] * 2)]

    def ctx_for(g0, g1, r0, r1):
        c = F.Context(F.make_params((nx, ny, g1 - g0), DT, DX, mu0=MU0, eps0=EPS0), storage=storage, tile_y=tile_y)
        assert not c.by_cells()
        c.set_materials(ids[g0:g1], table)
        c.set_rp([(p if q % 3 == 2 else p[g0:g1]).ravel() for q, p in enumerate(planes)])
        own = src[(src[:, 2] >= r0) & (src[:, 2] < r1)].copy()
        own[:, 2] -= g0
        c.set_sources(own, jz)
        for (f, lv), a in st.items():
            c.set(f, lv, a[g0:g1])
        return c

    print(f"\ntiled slabs, storage {storage}, {tile_y} rows", flush=True)
    whole = ctx_for(0, nz, 0, nz)
    slabs = []
    for r0, r1 in zip(cuts, cuts[1:]):
        g0, g1 = r0 - (r0 > 0), r1 + (r1 < nz)
        slabs.append((ctx_for(g0, g1, r0, r1), g0, r0, r1))
    up = hip.DeviceArray(slabs[0][0].halo_bytes(F.HALO_UP) // 4)
    down = hip.DeviceArray(slabs[0][0].halo_bytes(F.HALO_DOWN) // 4)
    for _ in range(9):
        for (lo, *_), (hi, *_) in zip(slabs, slabs[1:]):
            lo.halo_pack(F.HALO_UP, up.ptr)
            hi.halo_unpack(F.HALO_UP, up.ptr)
            hi.halo_pack(F.HALO_DOWN, down.ptr)
            lo.halo_unpack(F.HALO_DOWN, down.ptr)
        for c, *_ in slabs:
            c.step()
        whole.step()
    for f in range(9):
        for lv in ([0] if 3 <= f < 6 else [0, 1, 2]):
            ref = whole.get(f, lv)
            for c, g0, r0, r1 in slabs:
                got = c.get(f, lv)[r0 - g0:r1 - g0]
                assert np.array_equal(got.view(np.uint32), ref[r0:r1].view(np.uint32)), f"{F.FIELDS[f]} level {lv} [{r0},{r1})"
    assert np.abs(whole.get(8)).max() > 0
    up.free()
    down.free()
