"""Gather over every channel count with a kernel of its own, and the counts on either side of the last one."""
import numpy as np
import pytest

from helios_amd import native
from oracle.oracle import OracleScene
from tests.helpers import rel_err, small_canopy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 2, 3, 4, 5, 7, 8, 9, 11, 13, 15, 16, 17])
def test_channel_counts(ctx, B):
    """81 rays a face (a full step of 64 lanes and a remainder), distinct materials and fluxes in every band.  The
    oracle's bound of the solve tests: 1e-4 relative, 1 W/m2 floor."""
    s = small_canopy(51, 260)
    rng = np.random.default_rng(B)
    leaf = (s.twosided == 1)[:, None]
    rho = np.where(leaf, rng.uniform(0.05, 0.45, (1, B)), 0.2).astype(np.float32)
    tau = np.where(leaf, rng.uniform(0.05, 0.4, (1, B)), 0.0).astype(np.float32)
    bands = [native.BandSpec(f"b{b}", 2, False, float(rng.uniform(50, 150))) for b in range(B)]
    req = native.BandRequest(s.P, bands, rho=rho, tau=tau, direct_rays=25, diffuse_rays=81,
                             source_dirs=[native.sun_direction(40.0, 120.0)],
                             source_flux=[rng.uniform(200, 600, B).tolist()], direct_seed=21,
                             diffuse_seeds=[31, 32, 33])
    R = native.run_band(ctx.scene(s.transforms, s.types, s.twosided), req)
    Ro = OracleScene(s.transforms, s.types, s.twosided).run_band(req)
    assert rel_err(R, Ro, floor=1.0).max() <= 1e-4
