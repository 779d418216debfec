"""The block tree's traversals (rt_types.h, rt_traverse.h) where they can go wrong, against the oracle.

Hit words, IDs, distances and normals are compared bit for bit: the tree only decides which primitives are tested.
Cases: trees of 1 to 17 records (nodes with unused children), ray counts around the 64-entry ray queue, a chain of
boxes that halve in size (deep trees, stack rows beyond the LDS part), masks set after the build (the blocks hold
copies of the records), and cast rays along the axes, from inside and from 30 m outside the scene (a ray from
kilometres away loses the box tests' padding to FP32 rounding in any of the trees)."""
import numpy as np
import pytest

from helios_amd import native, scenes
from oracle.oracle import OracleScene

pytestmark = pytest.mark.gpu


def _patches(centres, sizes, seed=0, twosided=1):
    """Square patches at random orientations."""
    rng = np.random.default_rng(seed)
    P = len(centres)
    T = np.zeros((P, 4, 4), np.float32)
    for i in range(P):
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        T[i, :3, :3] = q * sizes[i]
        T[i, :3, 3] = centres[i]
        T[i, 3, 3] = 1.0
    return scenes.SceneArrays(T.reshape(P, 16), np.zeros(P, np.uint32), np.full(P, twosided, np.uint32))


def _cloud(P, seed=1):
    rng = np.random.default_rng(seed)
    return _patches(rng.uniform(-0.3, 0.3, (P, 3)), np.full(P, 0.25), seed)


def _chain(P=48):
    """Patches at distances and sizes that shrink by 1/3 from the first to the last."""
    f = (2.0 / 3.0) ** np.arange(P)
    return _patches(np.stack([f, 0.3 * f, 0.1 * f], 1), 0.5 * f, 3)


def _same_hits(ctx, s, n, seed=11, masks=None):
    g, o = ctx.scene(s.transforms, s.types, s.twosided, periodic=s.periodic), OracleScene.from_arrays(s)
    if masks:
        g.set_masks(*masks)
        o.set_masks(*masks)
    hg, ho = g.diffuse_hits(n, seed), o.diffuse_hits(n, seed)
    assert np.array_equal(hg, ho), f"{np.count_nonzero(hg != ho)} of {hg.size} hit words differ"
    return ho


@pytest.mark.parametrize("P", [1, 2, 3, 4, 5, 6, 17])
def test_small_trees(ctx, P):
    _same_hits(ctx, _cloud(P), 7)


@pytest.mark.parametrize("n", [1, 2, 5, 6, 8, 9, 33])
def test_ray_counts(ctx, n):
    """2 n^2 rays of a two-sided primitive: 2 to 2,178, among them 50, 72, 128 and 162."""
    h = _same_hits(ctx, _cloud(40), n)
    assert np.count_nonzero(h < 0x80000000) > 0


def test_deep_chain(ctx):
    s = _chain()
    g = ctx.scene(s.transforms, s.types, s.twosided)
    assert g.info()["depth4"] >= 8
    h = _same_hits(ctx, s, 16)
    assert np.count_nonzero((h & 0x7FFFFFFF) < s.P) > 0


def test_masks_after_the_build(ctx):
    """Every other texel transparent: the blocks' records must carry the masks set after they were built."""
    s = _cloud(60)
    mask = (np.indices((8, 8)).sum(0) % 2).astype(np.uint8)
    masks = ([mask], np.where(np.arange(s.P) % 3 == 0, -1, 0).astype(np.int32))
    plain, masked = _same_hits(ctx, s, 6), _same_hits(ctx, s, 6, masks=masks)
    assert not np.array_equal(plain, masked)


@pytest.mark.parametrize("distance", [0.0, 30.0])
def test_cast_axis_parallel_and_far_rays(ctx, distance):
    s = scenes.random_canopy(5, 3000)
    g, o = ctx.scene(s.transforms, s.types, s.twosided), OracleScene.from_arrays(s)
    T = s.transforms.reshape(-1, 16)
    rng = np.random.default_rng(2)
    D = np.concatenate([np.repeat(np.eye(3), 60, 0), -np.repeat(np.eye(3), 60, 0), rng.normal(size=(300, 3))])
    D /= np.linalg.norm(D, axis=1, keepdims=True)
    aim = T[rng.integers(0, s.P, len(D))][:, [3, 7, 11]]
    O = (aim - D * distance).astype(np.float32)
    D = D.astype(np.float32)
    t, nrm, u = g.cast_rays(O, D)
    to, no, uo = o.cast_rays(O, D)
    assert np.array_equal(u, uo)
    hit = u != 0xFFFFFFFF
    assert hit.any()
    assert np.array_equal(t[hit], to[hit]) and np.array_equal(nrm[hit], no[hit])


@pytest.mark.parametrize("far", [1e30, 1e34, 1e37])
def test_one_primitive_far_away(ctx, far):
    """Extents beyond the nodes' largest steps: such a scene is traced without a block tree."""
    s = _cloud(60)
    s.transforms[7, 3] = far
    g, o = ctx.scene(s.transforms, s.types, s.twosided), OracleScene.from_arrays(s)
    rng = np.random.default_rng(4)
    O, D = rng.uniform(-0.5, 0.5, (500, 3)).astype(np.float32), rng.normal(size=(500, 3))
    D = (D / np.linalg.norm(D, axis=1, keepdims=True)).astype(np.float32)
    t, nrm, u = g.cast_rays(O, D)
    to, no, uo = o.cast_rays(O, D)
    hit = u != 0xFFFFFFFF
    assert np.array_equal(u, uo) and hit.sum() > 100
    assert np.array_equal(t[hit], to[hit]) and np.array_equal(nrm[hit], no[hit])


@pytest.mark.parametrize("bad", [np.inf, -np.inf])
def test_infinite_coordinates_are_refused(ctx, bad):
    s = _cloud(60)
    s.transforms[7, 3] = bad
    with pytest.raises(native.RTError, match="not finite"):
        ctx.scene(s.transforms, s.types, s.twosided)
