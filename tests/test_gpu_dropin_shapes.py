"""The drop-in H, D and E kernels where their lanes' mapping can go wrong:
odd and even plane counts (lanes take plane pairs), the smallest edges, rows
that are no divisor of a block, and a grid large enough for the streaming
form (more than 256 MB in the reference's 25 arrays)."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import oracle_sim, random_materials, random_rp, random_sources, random_state
from tests.test_gpu_parity import DT, DX, Legacy, _compare_all

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,steps", [((3, 3, 3), 4), ((3, 4, 4), 4), ((5, 3, 7), 4), ((257, 3, 6), 4),
                                         ((16, 16, 5), 4), ((100, 51, 8), 3), ((139, 140, 139), 1)])
def test_dropin_shapes_bit_exact(shape, steps):
    print(f"drop-in {shape}", flush=True)
    rng = np.random.default_rng(list(shape))
    ids, table = random_materials(rng, shape)
    rps, src = random_rp(rng, shape), random_sources(rng, shape, 3)
    jz = rng.uniform(-2, 2, 40).astype(np.float32)
    st = random_state(rng, shape)
    leg = Legacy(shape, table, ids, rps, src, jz, O.DEBYE_FIXED)
    leg.set_state(st)
    sim = oracle_sim(shape, DT, DX, debye=O.DEBYE_FIXED)
    t = table[ids.astype(np.int64)]
    sim.set_materials(t[..., 0], t[..., 1], t[..., 2], t[..., 3])
    sim.set_rp(rps)
    sim.set_sources(src, jz, jz_mode=0)
    for (f, lv), a in st.items():
        sim.set(f, lv, a)
    for n in range(steps):
        leg.step((n // 3) * 3)
        sim.step()
    _compare_all(leg.get, sim.get, f"drop-in {shape}")
