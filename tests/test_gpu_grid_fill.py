"""Occlusion grid lists built from rectangles of very different sizes in one workgroup of 256 leaves."""
import numpy as np
import pytest

from helios_amd import native
from tests.helpers import small_canopy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [1, 2, 64, 255, 256, 257, 700])
def test_mixed_rectangles(ctx, P):
    """A patch under the whole scene, long strips and small patches: the grid's decisions are the BVH's, and
    both kernels write count x strength, so the sums have the same bits."""
    rng = np.random.default_rng(P)
    T = np.zeros((P, 16), np.float32)
    size = np.where(np.arange(P)[:, None] % 7 == 3, [[6.0, 0.02]], [[0.15, 0.1]])
    pos = rng.uniform(-4.0, 4.0, (P, 3))
    pos[:, 2] = rng.uniform(0.0, 2.0, P)
    size[0], pos[0] = (10.0, 10.0), (0.0, 0.0, -0.01)
    T[:, 0], T[:, 5], T[:, 10], T[:, 15] = size[:, 0], size[:, 1], 1.0, 1.0
    T[:, 3], T[:, 7], T[:, 11] = pos.T
    g = ctx.scene(T, np.zeros(P, np.uint32), np.ones(P, np.uint32))
    src = [native.sun_direction(z, a) for z, a in ((1, 0), (40, 100), (80, 310))]
    try:
        ctx.set_direct_grids(True)
        sg = g.direct_sums(9, 3, src)
        ctx.set_direct_grids(False)
        sb = g.direct_sums(9, 3, src)
    finally:
        ctx.set_direct_grids(True)
    assert np.array_equal(sg, sb)
    assert sg.max() > 0


@pytest.mark.parametrize("d", [1, 7, 8, 9, 16, 33])
@pytest.mark.parametrize("predicates", ["reference", "watertight"])
def test_ray_batches(ctx, d, predicates):
    """Rays a primitive below, at and above a batch of 64: the grid's decisions are the BVH's, bit for bit."""
    s = small_canopy(41, 700)
    g = ctx.scene(s.transforms, s.types, s.twosided)
    src = [native.sun_direction(z, a) for z, a in ((3, 0), (50, 130), (87, 260))]
    try:
        ctx.set_predicates(predicates)
        ctx.set_direct_grids(True)
        sg = g.direct_sums(d, 17, src)
        ctx.set_direct_grids(False)
        sb = g.direct_sums(d, 17, src)
    finally:
        ctx.set_direct_grids(True)
        ctx.set_predicates("reference")
    assert np.array_equal(sg, sb)
