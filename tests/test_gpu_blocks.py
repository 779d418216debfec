"""The block tree's traversals (rt_types.h, rt_traverse.h) where they can go wrong, against the oracle.

Hit words, IDs, distances and normals are compared bit for bit: the tree only decides which primitives are tested.
Cases: trees of 1 to 17 records (nodes with unused children), ray counts around the 64-entry ray queue, a chain of
boxes that halve in size (deep trees, stack rows beyond the LDS part), masks set after the build (the blocks hold
copies of the records), and cast rays along the axes, from inside and from 30 m outside the scene (a ray from
kilometres away loses the box tests' padding to FP32 rounding in any of the trees)."""
import numpy as np
import pytest

from helios_amd import native, scenes
from oracle.oracle import OracleScene, predicates

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


def _nested_clusters(levels, f, scale):
    """Clusters of 16 patches that shrink by f towards a point: each level of the tree opens its own cluster before
    the smaller ones, so the wide tree is more than half as deep as the binary one."""
    rng = np.random.default_rng(3)
    r = scale * np.repeat(f ** np.arange(levels), 16)
    c = np.stack([r, 0 * r, 0 * r], 1) + rng.uniform(-0.12, 0.12, (levels * 16, 3)) * r[:, None]
    return _patches(c, 0.036 * r, 3)


@pytest.mark.parametrize("levels, f, scale", [(48, 0.7, 1e6), (56, 0.6, 1.0)])
def test_trees_with_wide_links(ctx, levels, f, scale):
    """Trees too deep for RT_STACK stack rows (from 22 levels on): their links are wide and the kernels that walk them
    are instances of their own.  56 levels: the binary tree is the fallback builder's.  Rays to lamps walk the binary
    tree here, as the counting kernels do.  Casts start next to the cluster they aim at, and into the first scene alone:
    castRays widens a patch of side a by 1e-8 / a and a far origin blurs it, both past the box of the smallest patches,
    where a tree (the oracle's too) finds other hits than a test of every primitive."""
    s = _nested_clusters(levels, f, scale)
    g, o = ctx.scene(s.transforms, s.types, s.twosided), OracleScene.from_arrays(s)
    assert g.info()["depth4"] >= 22
    rng = np.random.default_rng(6)
    D = rng.normal(size=(4000, 3))
    D = (D / np.linalg.norm(D, axis=1, keepdims=True)).astype(np.float32)
    k = rng.integers(0, s.P, len(D))
    O = (s.transforms.reshape(-1, 16)[k][:, [3, 7, 11]] - 0.3 * scale * f ** (k // 16)[:, None] * D).astype(np.float32)
    lamp = ([[0.6 * scale, 0.3 * scale, 0.8 * scale]], [native.SOURCE_SPHERE], [(0.2 * scale, 0.2 * scale)], [(0.0, 0.0, 0.0)])
    for mode in ("reference", "watertight"):
        try:
            ctx.set_predicates(mode)
            with predicates(mode):
                assert np.array_equal(g.diffuse_hits(6, 3), o.diffuse_hits(6, 3))
                if scale > 1.0:
                    (t, nrm, u), (to, no, uo) = g.cast_rays(O, D), o.cast_rays(O, D)
                    hit = u != 0xFFFFFFFF
                    assert np.array_equal(u, uo) and hit.sum() > 400
                    assert np.array_equal(t[hit], to[hit]) and np.array_equal(nrm[hit], no[hit])
            a = g.direct_sums_src(8, 5, *lamp)
            ctx.set_counting(True)
            b = g.direct_sums_src(8, 5, *lamp)
            assert np.array_equal(a, b) and a.max() > 0
        finally:
            ctx.set_counting(False)
            ctx.set_predicates("reference")
    mask = (np.indices((8, 8)).sum(0) % 2).astype(np.uint8)
    masks = ([mask], np.where(np.arange(s.P) % 3 == 0, -1, 0).astype(np.int32))
    g.set_masks(*masks)
    o.set_masks(*masks)
    assert np.array_equal(g.diffuse_hits(6, 3), o.diffuse_hits(6, 3))


def test_more_blocks_than_byte_offsets_reach(ctx):
    """48 copies of the orchard: 64 M blocks and more.  The scene has a block tree (its bytes are in the footprint), and
    casts and diffuse rays over it have the results of the binary tree."""
    one, k = scenes.orchard(1), 48
    T0 = one.transforms.reshape(-1, 16)
    n, ext = len(T0), T0[:, [3, 7]].max(0) - T0[:, [3, 7]].min(0) + 1
    T = np.tile(T0, (k, 1))
    for j in range(k):
        T[j * n:(j + 1) * n, 3] += (j % 7) * ext[0]
        T[j * n:(j + 1) * n, 7] += (j // 7) * ext[1]
    g = ctx.scene(T, np.tile(one.types, k), np.tile(one.twosided, k))
    i = g.info()
    assert i["depth4"] <= 21  # the depth does not ask for wide links
    blocks = i["device_bytes"] - n * k * 112 - i["nleaves"] * 64 - (i["nleaves"] - 1) * (64 + 128)
    assert blocks > 64 * 2 ** 26
    rng = np.random.default_rng(1)
    lo, hi = T[:, [3, 7, 11]].min(0), T[:, [3, 7, 11]].max(0)
    O = (lo + (hi - lo) * rng.random((400000, 3))).astype(np.float32)
    D = rng.normal(size=O.shape)
    D = (D / np.linalg.norm(D, axis=1, keepdims=True)).astype(np.float32)
    try:
        a, ha = g.cast_rays(O, D), g.diffuse_hits(1, 5)
        ctx.set_counting(True)
        b, hb = g.cast_rays(O, D), g.diffuse_hits(1, 5)
    finally:
        ctx.set_counting(False)
        g.close()
    hit = a[2] != 0xFFFFFFFF
    assert hit.mean() > 0.2
    for x, y in zip(a, b):
        assert np.array_equal(x[hit], y[hit])
    assert np.array_equal(a[2], b[2])
    assert np.array_equal(ha, hb)


@pytest.mark.parametrize("far", [1e30, 1e34, 1e37])
def test_one_primitive_far_away(ctx, far):
    """Extents beyond the nodes' largest steps (the last two): such a scene is traced without a block tree, by the
    kernels over the binary tree."""
    s = _cloud(60)
    s.transforms[7, 3] = far
    g, o = ctx.scene(s.transforms, s.types, s.twosided), OracleScene.from_arrays(s)
    rng = np.random.default_rng(4)
    O, D = rng.uniform(-0.5, 0.5, (500, 3)).astype(np.float32), rng.normal(size=(500, 3))
    D = (D / np.linalg.norm(D, axis=1, keepdims=True)).astype(np.float32)
    mask = (np.indices((8, 8)).sum(0) % 2).astype(np.uint8)
    masks = ([mask], np.where(np.arange(s.P) % 3 == 0, -1, 0).astype(np.int32))
    lamp = ([[0.1, 0.2, 0.9]], [native.SOURCE_DISK], [(0.2, 0.2)], [(np.pi, 0.0, 0.0)])
    for masked in (False, True):
        if masked:
            g.set_masks(*masks)
            o.set_masks(*masks)
        for mode in ("reference", "watertight"):
            try:
                ctx.set_predicates(mode)
                with predicates(mode):
                    assert np.array_equal(g.diffuse_hits(6, 3), o.diffuse_hits(6, 3))
                    (t, nrm, u), (to, no, uo) = g.cast_rays(O, D), o.cast_rays(O, D)
                    assert np.allclose(g.direct_sums_src(6, 5, *lamp), o.direct_sums_src(6, 5, *lamp), rtol=1e-5, atol=1e-7)
            finally:
                ctx.set_predicates("reference")
            hit = u != 0xFFFFFFFF
            assert np.array_equal(u, uo) and hit.sum() > 100
            assert np.array_equal(t[hit], to[hit]) and np.array_equal(nrm[hit], no[hit])


@pytest.mark.parametrize("bad", [np.inf, -np.inf])
def test_infinite_coordinates_are_refused(ctx, bad):
    s = _cloud(60)
    s.transforms[7, 3] = bad
    with pytest.raises(native.RTError, match="not finite"):
        ctx.scene(s.transforms, s.types, s.twosided)
