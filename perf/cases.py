"""The timed work of a user of fdtd_amd, through its public entry points.

A case is one of four kinds of program:
  ctx     one grid in a Context: `steps` time steps (Context.run, or
          Context.step where `steps` is 1), then the nine newest fields of
          the whole grid as fp32 volumes in device memory (Context.snapshot):
          a run that dumps its fields every `steps` steps.
  slabs   the grid cut into z-slabs that exchange their halo planes before
          every step (Context.halo_pack / halo_unpack), as a multi-GPU run
          does on each of its devices, then the fields of every slab.
  dropin  the five entry points of the reference (updateHField ...
          updateMurBoundary) called step by step on the caller's own packed
          device arrays, the way the reference's main loop drives them.
  batch   `grids` uneven grids solved together: added to a Batch that the
          program keeps, run to their step counts, probe series read back,
          removed.

The sizes are those of the framework's own workloads: 24^3 (the smoke run),
32^3 to 192^3 edges (served requests and batched sets), 64^3 and 256^3 (the
plain grids), 100^3 (the reference's input_params), 320x320x880 (the large
phantom), with ragged edges among them; fp32 storage first (the reference's
arithmetic), fp16 and bf16 beside it.

Grids are vacuum with a seeded phantom of Debye tissues kept inside the
faces, point sources that carry a continuous wave, and the Mur planes of a
vacuum background.
"""
import ctypes as C
import math

import numpy as np
import torch

import fdtd_amd as F

C0 = 3.0e8
MU0 = 1.2566371e-06
EPS0 = 8.841941e-12
CELL = 2.0e-3
DT = 0.99 * CELL / (C0 * math.sqrt(3.0))
FREQ = 2.45e9
WAVE = 8192                    # entries of a source waveform
DROPIN_WAVE = 512              # the reference's device table
STORE = {"f32": F.STORE_F32, "f16": F.STORE_F16, "bf16": F.STORE_BF16, "f32_fast": F.STORE_F32_FAST}
BATCH_BYTES = 4 << 30


def listed():
    return [
        # one step at a time with a look at the fields after it, the smallest grid: launches and latency
        dict(name="step_24", kind="ctx", storage="f32", nx=24, ny=24, nz=24, steps=1),
        # the smallest served request, a short burst of steps
        dict(name="run_32", kind="ctx", storage="f32", nx=32, ny=32, nz=32, steps=50),
        # plain_small's grid
        dict(name="run_64", kind="ctx", storage="f32", nx=64, ny=64, nz=64, steps=50),
        # a ragged served request in fp16
        dict(name="run_f16_96x121x77", kind="ctx", storage="f16", nx=96, ny=121, nz=77, steps=40),
        # the largest grid of the batched set, ragged in x and y
        dict(name="run_151x138x188", kind="ctx", storage="f32", nx=151, ny=138, nz=188, steps=30),
        # a ragged request in bf16
        dict(name="run_bf16_130x156x150", kind="ctx", storage="bf16", nx=130, ny=156, nz=150, steps=30),
        # plain_256's grid
        dict(name="run_256", kind="ctx", storage="f32", nx=256, ny=256, nz=256, steps=20),
        # the same in fp16
        dict(name="run_f16_256", kind="ctx", storage="f16", nx=256, ny=256, nz=256, steps=20),
        # the large phantom's grid, the size the headline figure is quoted on
        dict(name="run_320x320x880", kind="ctx", storage="f32", nx=320, ny=320, nz=880, steps=24),
        # a large grid as four slabs, halos exchanged every step
        dict(name="slabs_320x320x224", kind="slabs", storage="f32", nx=320, ny=320, nz=224, steps=8, slabs=4),
        # the reference's own grid through its own entry points
        dict(name="dropin_100", kind="dropin", storage="f32", nx=100, ny=100, nz=100, steps=30),
        # a sweep of uneven grids solved together
        dict(name="batch_12", kind="batch", storage="f32", grids=12, edge=96, steps=200),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["ctx"] * 8 + ["slabs", "dropin", "batch"])
    if kind == "batch":
        return dict(kind=kind, storage=rng.choice(["f32", "f32", "f16"]), grids=rng.randint(3, 24),
                    edge=int(_log(rng, 48, 128)), steps=rng.randint(50, 250))
    storage = "f32" if kind != "ctx" else rng.choice(["f32"] * 5 + ["f16", "bf16", "f32_fast"])
    base = {"ctx": _log(rng, 26, 380), "slabs": _log(rng, 64, 256), "dropin": _log(rng, 32, 160)}[kind]
    nx, ny, nz = (max(24, int(base * rng.uniform(0.75, 1.4))) for _ in range(3))
    cells = nx * ny * nz
    c = dict(kind=kind, storage=storage, nx=nx, ny=ny, nz=nz)
    if kind == "ctx":
        c["steps"] = 1 if rng.random() < 0.1 else max(1, min(rng.randint(8, 100), int(1.5e9 / cells)))
    elif kind == "slabs":
        c["slabs"] = rng.randint(2, 4)
        c["steps"] = rng.randint(2, 10)
    else:
        c["steps"] = rng.randint(6, 40)
    return c


# ---- inputs -----------------------------------------------------------------

def _phantom(g, nx, ny, nz):
    """Vacuum, a body of elliptical cross-section in seeded tissue layers, and
    seeded boxes of further tissues, all inside the faces."""
    n = 12
    ei = g.uniform(4.0, 45.0, n)
    es = np.maximum(ei + 1.0, g.uniform(5.0, 80.0, n))
    rows = np.stack([g.uniform(0.02, 2.5, n), es, ei, g.uniform(5e-12, 50e-12, n)], 1)
    table = np.concatenate([[(0.0, 1.0, 1.0, 0.0)], rows]).astype(np.float32)
    m = [min(10, e // 3) for e in (nx, ny, nz)]
    ids = np.zeros((nz, ny, nx), np.uint8)
    cx, cy = nx / 2 + g.uniform(-1, 1), ny / 2 + g.uniform(-1, 1)
    ax, ay = g.uniform(0.3, 0.4) * (nx - 2 * m[0]), g.uniform(0.3, 0.4) * (ny - 2 * m[1])
    y, x = np.mgrid[0:ny, 0:nx]
    body = ((x - cx) / ax) ** 2 + ((y - cy) / ay) ** 2 <= 1.0
    body &= (x >= m[0]) & (x < nx - m[0]) & (y >= m[1]) & (y < ny - m[1])
    z0, z1 = m[2], nz - m[2]
    layer = max(1, (z1 - z0) // 8)
    for q, z in enumerate(range(z0, z1, layer)):
        ids[z:min(z + layer, z1)] = body * np.uint8(1 + (q + int(g.integers(0, 3))) % n)
    for b in range(8):
        lo = [m[d] + int(g.uniform(0.1, 0.6) * (e - 2 * m[d])) for d, e in enumerate((nx, ny, nz))]
        hi = [min(e - m[d], lo[d] + max(1, int(g.uniform(0.08, 0.3) * (e - 2 * m[d]))))
              for d, e in enumerate((nx, ny, nz))]
        ids[lo[2]:hi[2], lo[1]:hi[1], lo[0]:hi[0]] = 1 + (b + 4) % n
    return ids, table


def _sources(g, nx, ny, nz, count=6):
    """Distinct seeded cells inside the faces."""
    seen = []
    while len(seen) < count:
        c = tuple(int(g.integers(3, e - 3)) for e in (nx, ny, nz))
        if c not in seen:
            seen.append(c)
    return np.asarray(seen, np.int32)


def _wave(g, n):
    """A carrier that swells over its first period and then goes on."""
    t = (np.arange(n) + 1) * DT
    return (g.uniform(0.5, 2.0) * np.sin(2 * np.pi * FREQ * t) * np.minimum(1.0, t * FREQ)).astype(np.float32)


def _inputs(case, seed):
    g = np.random.default_rng([int(seed), case["nx"], case["ny"], case["nz"]])
    shape = (case["nx"], case["ny"], case["nz"])
    ids, table = _phantom(g, *shape)
    jz = _wave(g, DROPIN_WAVE if case["kind"] == "dropin" else WAVE)
    return shape, ids, table, _sources(g, *shape), jz


def _batch_grids(case):
    """(shape, steps) of the grids of a batch."""
    g = np.random.default_rng([case["grids"], case["edge"], case["steps"]])
    return [(tuple(int(case["edge"] * v) for v in g.uniform(0.6, 1.4, 3)),
             int(case["steps"] * g.uniform(0.5, 1.0)) + 1) for _ in range(case["grids"])]


def _batch_inputs(case, seed):
    g = np.random.default_rng([int(seed), case["grids"], case["edge"]])
    out = []
    for shape, steps in _batch_grids(case):
        nx, ny, nz = shape
        ids, table = _phantom(g, *shape)
        src = _sources(g, *shape, count=1)
        x, y, z = (int(v) for v in src[0])
        probes = [(8, nx // 2, ny // 2, nz // 2), (8, min(x + 3, nx - 2), y, z), (3, x, y, z), (1, x, y, z)]
        out.append((shape, ids, table, src, _wave(g, steps), steps, np.asarray(probes, np.int32)))
    return out


def _begun(case):
    """Steps taken before the pass: a program that steps one by one has begun
    its run."""
    return 40 if case["kind"] == "ctx" and case["steps"] == 1 else 0


def _params(shape):
    return F.make_params(shape, DT, CELL, mu0=MU0, eps0=EPS0)


def _bounds(case):
    n = case["slabs"]
    return [case["nz"] * s // n for s in range(n + 1)]


def prepare(case, seed):
    if case["kind"] == "batch":
        ext = F.make_ext(storage=STORE[case["storage"]])
        insts = [F.Instance(_params(shape), ext, ids, table, src, jz, steps, probes=probes)
                 for shape, ids, table, src, jz, steps, probes in _batch_inputs(case, seed)]
        return dict(kind="batch", batch=F.Batch(BATCH_BYTES), insts=insts)
    shape, ids, table, src, jz = _inputs(case, seed)
    nx, ny, nz = shape
    if case["kind"] == "ctx":
        ctx = F.Context(_params(shape), storage=STORE[case["storage"]])
        ctx.set_materials(ids, table)
        ctx.set_sources(src, jz)
        ctx.run(_begun(case))
        out = torch.zeros((9, nz, ny, nx), device="cuda")
        return dict(kind="ctx", ctx=ctx, steps=case["steps"], out=out)
    if case["kind"] == "slabs":
        b = _bounds(case)
        slabs, outs = [], []
        for s in range(case["slabs"]):
            g0, g1 = b[s] - (s > 0), b[s + 1] + (s < case["slabs"] - 1)
            ctx = F.Context(_params((nx, ny, g1 - g0)), storage=STORE[case["storage"]])
            ctx.set_materials(ids[g0:g1], table)
            own = src[(src[:, 2] >= b[s]) & (src[:, 2] < b[s + 1])].copy()
            own[:, 2] -= g0
            ctx.set_sources(own, jz)
            slabs.append(ctx)
            outs.append(torch.zeros((9, g1 - g0, ny, nx), device="cuda"))
        up, down = slabs[0].halo_bytes(F.HALO_UP), slabs[0].halo_bytes(F.HALO_DOWN)
        ups = [torch.empty(up, dtype=torch.uint8, device="cuda") for _ in slabs[1:]]
        downs = [torch.empty(down, dtype=torch.uint8, device="cuda") for _ in slabs[1:]]
        return dict(kind="slabs", slabs=slabs, outs=outs, ups=ups, downs=downs, steps=case["steps"])
    # dropin: the reference's FdtdField arrays, on the device
    E = torch.zeros((3, 3, nz, ny, nx), device="cuda")   # [ring slot][component]
    D = torch.zeros((3, 3, nz, ny, nx), device="cuda")
    H = torch.zeros((3, nz, ny, nx), device="cuda")
    mats = torch.from_numpy(table).cuda()[torch.from_numpy(ids).cuda().long()]
    mats = [mats[..., q].contiguous() for q in range(4)]   # sigma, epsS, epsI, tauD
    rp = [torch.ones(n, device="cuda") for n in (2 * ny * nz, nx * 2 * nz, nx * ny * 2) * 2]
    params = _params(shape)
    src = np.ascontiguousarray(src)
    params.sourcesCount = len(src)
    params.sources = src.ctypes.data_as(C.POINTER(C.c_int))
    params.jzCount = len(jz)
    params.jz = jz.ctypes.data_as(C.POINTER(C.c_float))
    p = lambda t: t.data_ptr()  # noqa: E731
    calls = []
    for t in range(3):
        s1, s2 = (t + 2) % 3, (t + 1) % 3
        e, d, h = [[p(x) for x in a] for a in E], [[p(x) for x in a] for a in D], [p(x) for x in H]
        calls.append(dict(h=(*h, *e[s1], None), d=(*d[t], *d[s1], *h, None), src=(d[t][2], d[s1][2], h[0], h[1]),
                          e=(*e[t], *e[s1], *e[s2], *d[t], *d[s1], *d[s2], p(mats[0]), p(mats[2]), p(mats[1]),
                             p(mats[3]), None),
                          mur=(*e[t], *e[s1], *[p(x) for x in rp], None)))
    return dict(kind="dropin", E=E, D=D, H=H, mats=mats, rp=rp, params=params, keep=(src, jz), calls=calls, n=0,
                steps=case["steps"])


# ---- one pass ---------------------------------------------------------------

def _fields(v):
    return {name: v[q] for q, name in enumerate(F.FIELDS)}


def run(state):
    return {"ctx": _run_ctx, "slabs": _run_slabs, "dropin": _run_dropin, "batch": _run_batch}[state["kind"]](state)


def _run_ctx(s):
    if s["steps"] == 1:
        s["ctx"].step()
    else:
        s["ctx"].run(s["steps"])
    s["ctx"].snapshot(s["out"].data_ptr())
    return _fields(s["out"])


def _run_slabs(s):
    slabs, last = s["slabs"], len(s["slabs"]) - 1
    for _ in range(s["steps"]):
        for q in range(last):
            lo, hi, up, down = slabs[q], slabs[q + 1], s["ups"][q].data_ptr(), s["downs"][q].data_ptr()
            lo.halo_pack(F.HALO_UP, up)
            hi.halo_unpack(F.HALO_UP, up)
            hi.halo_pack(F.HALO_DOWN, down)
            lo.halo_unpack(F.HALO_DOWN, down)
        for c in slabs:
            c.step()
    res = {}
    for q, (c, out) in enumerate(zip(slabs, s["outs"])):
        c.snapshot(out.data_ptr())
        # a slab's own planes: its ghost planes belong to its neighbours
        res[f"slab{q}"] = _fields(out[:, (q > 0):out.shape[1] - (q < last)])
    return res


def _run_dropin(s):
    L = F.lib()
    F.check(L.copySymbolsToDevice(C.byref(s["params"])), "copySymbolsToDevice")
    for n in range(s["n"], s["n"] + s["steps"]):
        c = s["calls"][n % 3]
        F.check(L.updateHField(*c["h"]), "updateHField")
        F.check(L.updateDField(*c["d"]), "updateDField")
        F.check(L.updateSources(*c["src"], n, None), "updateSources")
        F.check(L.updateEField(*c["e"]), "updateEField")
        F.check(L.updateMurBoundary(*c["mur"]), "updateMurBoundary")
    s["n"] += s["steps"]
    t = (s["n"] - 1) % 3
    return _fields([*s["D"][t], *s["H"], *s["E"][t]])


def _run_batch(s):
    b = s["batch"]
    ids = [b.add(i) for i in s["insts"]]
    b.run(max(i.steps for i in s["insts"]))
    out = [b.probes(i) for i in ids]
    for i in ids:
        b.remove(i)
    return out


# ---- what a pass cannot do without ------------------------------------------

def work(case):
    """Per cell and step the state is read once (E and D at two levels, H, the
    material id) and written once (E, D, H): 24 values and a byte, with about
    110 operations of the update; a snapshot reads nine values and writes nine
    floats."""
    if case["kind"] == "batch":
        cells, steps = sum(nx * ny * nz * n for (nx, ny, nz), n in _batch_grids(case)), 1
    else:
        cells, steps = case["nx"] * case["ny"] * case["nz"], case["steps"]
    size = 2 if case["storage"] in ("f16", "bf16") else 4
    nbytes = cells * steps * (24 * size + 1)
    if case["kind"] == "dropin":
        nbytes += cells * steps * 15   # four floats of material instead of an id byte
    elif case["kind"] != "batch":
        nbytes += cells * 9 * (size + 4)
    return {"bytes": nbytes, "flops": 110.0 * cells * steps}


# ---- the same in 64 bits ----------------------------------------------------

def _solve64(shape, ids, table, src, jz, steps, probes=None):
    """Yee H, D, soft Jz, Debye E (d = a + b - sigma dt^2) and first-order Mur
    in float64; returns the nine fields, or the probe rows."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    nx, ny, nz = shape
    f = lambda v: float(np.float32(v))  # noqa: E731   the scalars as the framework takes them
    dt, dx, mu0, eps0 = f(DT), f(CELL), f(MU0), f(EPS0)
    ch, cd = dt / (mu0 * dx), dt / dx
    t64 = torch.from_numpy(table).to(dev).double()
    sg, es, ei, tau = t64.unbind(1)
    a = 2 * eps0 * ei * tau
    b = a + 2 * dt * (eps0 * es + sg * tau)
    coef = [1 / (b + sg * dt * dt), a + b - sg * dt * dt, a, 2 * (dt + tau), 2 * dt + 4 * tau, 2 * tau]
    idx = torch.from_numpy(ids).to(dev).long()
    cc, dd, aa, g1, g2, g3 = [v[idx] for v in coef]
    del idx
    zeros = lambda: [torch.zeros((nz, ny, nx), dtype=torch.float64, device=dev) for _ in range(3)]  # noqa: E731
    E0, E1, D0, D1, H = zeros(), zeros(), zeros(), zeros(), zeros()
    s = slice
    L, I, A = s(0, -1), s(1, -1), s(None)  # [0, n-1), [1, n-1), all
    up = s(1, None)
    root = math.sqrt(mu0 * eps0) * dx
    q, p, m = 1 / (dt + root), dt + root, dt - root
    sz, sy, sx = (torch.from_numpy(np.ascontiguousarray(src[:, d])).to(dev).long() for d in (2, 1, 0))
    rows = []
    for n in range(steps):
        (ex, ey, ez), (hx, hy, hz) = E0, H
        hx[L, L, I] += ch * ((ey[up, L, I] - ey[L, L, I]) - (ez[L, up, I] - ez[L, L, I]))
        hy[L, I, L] += ch * ((ez[L, I, up] - ez[L, I, L]) - (ex[up, I, L] - ex[L, I, L]))
        hz[I, L, L] += ch * ((ex[I, up, L] - ex[I, L, L]) - (ey[I, L, up] - ey[I, L, L]))
        D2 = [v.clone() for v in D0]
        D2[0][I, I, L] += cd * ((hz[I, I, L] - hz[I, s(0, -2), L]) - (hy[I, I, L] - hy[s(0, -2), I, L]))
        D2[1][I, L, I] += cd * ((hx[I, L, I] - hx[s(0, -2), L, I]) - (hz[I, L, I] - hz[I, L, s(0, -2)]))
        D2[2][L, I, I] += cd * ((hy[L, I, I] - hy[L, I, s(0, -2)]) - (hx[L, I, I] - hx[L, s(0, -2), I]))
        D2[2][sz, sy, sx] -= float(jz[n]) if n < len(jz) else 0.0
        E2 = zeros()
        for k, r in ((0, (I, I, L)), (1, (up, A, up)), (2, (up, A, up))):
            E2[k][r] = cc[r] * (dd[r] * E0[k][r] - aa[r] * E1[k][r] + g1[r] * D2[k][r] - g2[r] * D0[k][r]
                                + g3[r] * D1[k][r])
        for k, rng in ((0, (I, I, L)), (1, (I, L, I)), (2, (L, I, I))):
            for axis in range(3):
                if 2 - axis == k:       # E_x has no x face, and so on
                    continue
                for face, nb in ((0, 1), (-1, -2)):
                    at, to = list(rng), list(rng)
                    at[axis], to[axis] = face, nb
                    at, to = tuple(at), tuple(to)
                    # the framework's E_y face at the high x end takes the neighbour at n for n+1 (as the
                    # reference does)
                    tn = E0[k][to] if (k == 1 and axis == 2 and face == -1) else E2[k][to]
                    E2[k][at] = q * (m * tn + p * E0[k][to] - m * E0[k][at])
        E1, E0, D1, D0 = E0, E2, D0, D2
        if probes is not None:
            now = [*D0, *H, *E0]
            rows.append(torch.stack([now[w][k, j, i] for w, i, j, k in probes.tolist()]))
    return torch.stack(rows) if probes is not None else [*D0, *H, *E0]


def exact(case, seed):
    if case["kind"] == "batch":
        return [_solve64(shape, ids, table, src, jz, steps, probes)
                for shape, ids, table, src, jz, steps, probes in _batch_inputs(case, seed)]
    shape, ids, table, src, jz = _inputs(case, seed)
    v = _solve64(shape, ids, table, src, jz, _begun(case) + case["steps"])
    # z-directed sources drive no H_z in vacuum: what there is comes from the tissues, late, and is rounding
    # until then in any precision
    v[F.FIELDS.index("Hz")] = None
    if case["kind"] != "slabs":
        return _fields(v)
    b = _bounds(case)
    return {f"slab{q}": _fields([x if x is None else x[b[q]:b[q + 1]] for x in v]) for q in range(case["slabs"])}
