"""The drop-in H and D kernels on either side of the rule that sends small
and thin grids past the pairs of planes: few planes, few rows or columns, planes that fill
little of a block; and odd and even plane counts on both sides."""
import pytest

from tests import test_gpu_dropin_shapes as S

pytestmark = pytest.mark.gpu

FLAT = [(60, 40, 3), (60, 40, 7), (60, 3, 40), (60, 6, 21), (5, 5, 40), (18, 18, 31), (3, 80, 12), (300, 200, 4)]
PAIRS = [(300, 230, 8), (300, 230, 9), (733, 7, 110), (3, 510, 351), (80, 82, 81), (257, 101, 23)]
SMALL = [(60, 47, 8), (60, 47, 9), (16, 16, 9), (80, 80, 80), (64, 64, 128)]   # all cells resident at once: one lane per cell


@pytest.mark.parametrize("shape", FLAT + PAIRS + SMALL)
def test_dropin_thin_and_pairs_bit_exact(shape):
    S.test_dropin_shapes_bit_exact(shape, 4 if shape[0] * shape[1] * shape[2] < 100000 else 1)


@pytest.mark.parametrize("shape", [(159, 160, 159), (1010, 1000, 4)])
def test_dropin_streaming_forms_bit_exact(shape):
    """More than 400 MB in the reference's 25 arrays: streaming H, D and E, and
    a thin grid with streaming E."""
    assert 100 * shape[0] * shape[1] * shape[2] > 400_000_000
    S.test_dropin_shapes_bit_exact(shape, 1)
