"""Rays to lamps over the block tree against the binary tree (the counting kernels)."""
import numpy as np
import pytest

from tests.helpers import small_canopy
from tests.test_gpu_sources import POS, ROTS, TYPES, WIDTHS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("predicates", ["reference", "watertight"])
@pytest.mark.parametrize("d", [1, 8, 9])
@pytest.mark.parametrize("height", [0.7, 4.0])
def test_same_bits_as_binary_tree(ctx, periodic, predicates, d, height):
    """Lamps above the canopy and inside it (rays of a few centimetres): every ray has the same strength and
    occlusion in both, added in the same order, so the sums have the same bits."""
    s = small_canopy(17, 900, periodic=periodic)
    g = ctx.scene(s.transforms, s.types, s.twosided, periodic=s.periodic)
    pos = POS[1:].copy()
    pos[[0, 2, 3], 2] = height
    try:
        ctx.set_predicates(predicates)
        a = g.direct_sums_src(d, 5, pos, TYPES[1:], WIDTHS[1:], ROTS[1:])
        ctx.set_counting(True)
        b = g.direct_sums_src(d, 5, pos, TYPES[1:], WIDTHS[1:], ROTS[1:])
    finally:
        ctx.set_counting(False)
        ctx.set_predicates("reference")
    assert np.array_equal(a, b)
    assert a.max() > 0
