"""castRays with directions of other lengths than 1: distances count in lengths of the direction."""
import numpy as np
import pytest

from helios_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("power", [10, 50, 60, 70, 80])
def test_short_directions(ctx, power):
    """The watertight predicates take a direction of any length, and scaling it by a power of two scales every
    intermediate of theirs exactly: the same hits at distances that differ by that power, bit for bit."""
    s = scenes.random_canopy(5, 3000)
    T = s.transforms.reshape(-1, 16)
    rng = np.random.default_rng(2)
    D = np.concatenate([np.repeat(np.eye(3), 60, 0), -np.repeat(np.eye(3), 60, 0), rng.normal(size=(3000, 3))])
    D = (D / np.linalg.norm(D, axis=1, keepdims=True)).astype(np.float32)
    O = (T[rng.integers(0, s.P, len(D))][:, [3, 7, 11]] - 0.5 * D).astype(np.float32)
    g = ctx.scene(s.transforms, s.types, s.twosided)
    try:
        ctx.set_predicates("watertight")
        t, _, u = g.cast_rays(O, D)
        ts, _, us = g.cast_rays(O, np.ldexp(D, -power))
    finally:
        ctx.set_predicates("reference")
    hit = u != 0xFFFFFFFF
    assert np.count_nonzero(hit) > 2000
    assert np.array_equal(us, u)
    assert np.array_equal(np.ldexp(ts[hit], -power), t[hit])
