"""fdtd_ctx_snapshot against the host copies of the fields: cell counts around
a block's 1024, rows with and without padding, scaled and unscaled storage."""
import numpy as np
import pytest

import fdtd_amd as F
from fdtd_amd import hip
from tests.helpers import bits_equal, first_diff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [F.STORE_F32, F.STORE_F16, F.STORE_BF16, F.STORE_F32_FAST])
@pytest.mark.parametrize("shape", [(3, 3, 3), (16, 16, 4), (32, 8, 4), (5, 41, 5), (65, 7, 9), (128, 3, 11)])
def test_snapshot_equals_fields(shape, storage):
    rng = np.random.default_rng([*shape, storage])
    nx, ny, nz = shape
    n = nx * ny * nz
    with F.Context(F.make_params(shape, 3.8e-12, 2e-3, mu0=1.2566371e-06, eps0=8.841941e-12), storage=storage,
                   scales=(1.0, 1.0, 1.0) if storage in (F.STORE_F16, F.STORE_BF16) else (0.0, 0.0, 0.0)) as ctx:
        for f in range(9):
            ctx.set(f, 0, rng.uniform(-1, 1, (nz, ny, nx)).astype(np.float32))
        out = hip.DeviceArray(9 * n + 64)          # and what lies behind the copy stays as it is
        ctx.snapshot(out.ptr)
        hip.sync()
        got = out.download()
        for f in range(9):
            want = ctx.get(f)
            have = got[f * n:(f + 1) * n].reshape(nz, ny, nx)
            assert bits_equal(have, want), f"{F.FIELDS[f]}: {first_diff(have, want)}"
        assert not got[9 * n:].any()
        out.free()
