"""Work queue of the persistent launches: one chunk a wave without a counter, one counter, eight segments."""
import numpy as np
import pytest

from helios_amd import native
from tests.helpers import small_canopy, two_band_request

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [1, 7, 255, 257, 1023, 1024, 1025, 3001])
@pytest.mark.parametrize("chunk", [1, 3, 256])
def test_every_item_once(ctx, P, chunk):
    """One wave a workgroup and one workgroup a CU (256 waves: the queues of the direct and diffuse kernels are split
    from 1,024 chunks on) give the bits of the default shape: every primitive is handed out exactly once."""
    s = small_canopy(31, 3100)
    s.transforms, s.types, s.twosided = s.transforms[-P:], s.types[-P:], s.twosided[-P:]
    assert s.P == P
    g = ctx.scene(s.transforms, s.types, s.twosided)
    src = [native.sun_direction(z, a) for z, a in ((20, 40), (65, 200))]
    req = two_band_request(s, depth=1, nrays=9)

    def results():
        return g.diffuse_hits(3, 5), g.direct_sums(3, 5, src), native.run_band(g, req)

    ref = results()
    cfg = [ctx.get_launch_cfg(k) for k in range(3)]
    try:
        for k in range(3):
            ctx.set_launch_cfg(k, 1, 1, chunk)
        got = results()
    finally:
        for k in range(3):
            ctx.set_launch_cfg(k, *cfg[k])
    assert np.array_equal(got[0], ref[0])
    assert np.array_equal(got[1], ref[1])
    assert np.array_equal(np.asarray(got[2]), np.asarray(ref[2]))


@pytest.mark.parametrize("P", [4095, 4096, 4097, 9001])
@pytest.mark.parametrize("chunk", [1, 2])
def test_segmented_gather(ctx, P, chunk):
    """A gather's workgroups always hold four waves: one workgroup a CU is 1,024 waves, and its queue is split from
    4,096 chunks on."""
    s = small_canopy(32, 9100)
    s.transforms, s.types, s.twosided = s.transforms[-P:], s.types[-P:], s.twosided[-P:]
    g = ctx.scene(s.transforms, s.types, s.twosided)
    req = two_band_request(s, depth=1, nrays=9)
    ref = native.run_band(g, req)
    cfg = ctx.get_launch_cfg(2)
    try:
        ctx.set_launch_cfg(2, 4, 1, chunk)
        got = native.run_band(g, req)
    finally:
        ctx.set_launch_cfg(2, *cfg)
    assert np.array_equal(got, ref)
