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


def _request(s, B, bands, sky):
    """Bands `bands` of a B-band request; every second band has a Prague sky, the others a power law."""
    rng = np.random.default_rng(100 + B)
    leaf = (s.twosided == 1)[:, None]
    rho = np.where(leaf, rng.uniform(0.05, 0.45, (1, B)), 0.2).astype(np.float32)
    tau = np.where(leaf, rng.uniform(0.05, 0.4, (1, B)), 0.0).astype(np.float32)
    flux, dflux = rng.uniform(200, 600, B), rng.uniform(50, 150, B)
    kw = {}
    if sky:
        peak = rng.normal(size=(B, 3)) * [0.5, 0.5, 0.2] + [0.0, 0.0, 0.8]
        peak /= np.linalg.norm(peak, axis=1, keepdims=True)
        odd = np.arange(B) % 2 == 1
        prague = np.stack([rng.uniform(1, 3, B), rng.uniform(20, 40, B), rng.uniform(1, 2, B), 0.21 * odd], 1)
        kw = {"sky_extinction": np.where(odd, 0.0, rng.uniform(0.3, 0.9, B))[bands], "sky_peak_dir": peak[bands],
              "sky_norm": np.where(odd, 0.0, 0.35)[bands], "sky_prague": prague[bands]}
    return native.BandRequest(s.P, [native.BandSpec(f"b{b}", 2, False, float(dflux[b])) for b in bands],
                              rho=rho[:, bands], tau=tau[:, bands], direct_rays=25, diffuse_rays=81,
                              source_dirs=[native.sun_direction(40.0, 120.0)], source_flux=[flux[bands].tolist()],
                              direct_seed=21, diffuse_seeds=[31, 32, 33], **kw)


@pytest.mark.parametrize("sky", [False, True])
@pytest.mark.parametrize("B", [2, 3, 4, 6, 8, 9, 10, 12, 14, 16, 17])
def test_sky_and_energy(ctx, B, sky):
    """Directional skies and the energy bookkeeping have kernels of their own for every channel count.  Fluxes against
    the oracle (the solve tests' bound), the same bits with the bookkeeping on; its rows, which sum in FP64 what the
    passes gather in FP32, against solves of each band alone: three passes of compensated sums grouped differently stay
    within a few units in the last place each, 5e-6 of the energy put in."""
    s = small_canopy(52, 260)
    g = ctx.scene(s.transforms, s.types, s.twosided)
    req = _request(s, B, list(range(B)), sky)
    R = native.run_band(g, req)
    Ro = OracleScene(s.transforms, s.types, s.twosided).run_band(req)
    assert rel_err(R, Ro, floor=1.0).max() <= 1e-4
    native.set_energy_accounting(ctx, True)
    try:
        assert np.array_equal(native.run_band(g, req), R)
        e = native.energy_fp64(ctx, B)
        for b in range(B):
            native.run_band(g, _request(s, B, [b], sky))
            one = native.energy_fp64(ctx, 1)
            put_in = one["source"][0] + one["sky"][0]
            assert put_in > 0
            for row in native.ENERGY_ROWS:
                assert abs(e[row][b] - one[row][0]) <= 5e-6 * put_in, (row, b)
            assert np.abs(e["passes"][:, :, b] - one["passes"][:, :, 0]).max() <= 5e-6 * put_in, b
    finally:
        native.set_energy_accounting(ctx, False)
