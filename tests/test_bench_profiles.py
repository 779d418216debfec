"""bench.py takes a kernel's traffic only from a profile of that kernel in its present shape."""
import json
import os

import pytest

import bench


@pytest.mark.parametrize("kernel, name, flags, taken", [
    ("k_cast", "void rt::k_cast<4, 0>", 0, True),
    ("k_cast", "void rt::k_cast<4, 2>", 0, False),            # watertight predicates
    ("k_cast", "void rt::k_cast<64, false, 0>", 0, False),    # <STK, COUNT, FLAGS> of an earlier build
    ("k_cast", "void rt::k_cast_bin<64, false, 0>", 0, False),
    ("k_diffuse", "void rt::k_diffuse<2, 1>", 1, True),
    ("k_diffuse", "void rt::k_diffuse<2, 16>", 0, False),     # wide links
    ("k_diffuse", "void rt::k_diffuse<2, 64, false, 0>", 0, False),
    ("k_direct", "void rt::k_direct<2, 32, false, 0>", 0, True),
    ("k_direct", "void rt::k_direct<4, 32, true, 0>", 0, False),  # counting
    ("k_direct", "void rt::k_direct_q<2, 0>", 0, False),
    ("k_camera", "void rt::k_camera<64, false, 0, false>", 0, True),
])
def test_profile_of_the_launched_kernel(tmp_path, monkeypatch, kernel, name, flags, taken):
    os.mkdir(tmp_path / "profiles")
    counts = {"FETCH_SIZE": {"max_bytes": 3.0}, "WRITE_SIZE": {"max_bytes": 1.0}}
    (tmp_path / "profiles" / "p.json").write_text(json.dumps({"kernels": {name: counts}}))
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    got = bench.pmc_profile(kernel, "p.json", flags)
    assert (got["bytes"] if got else None) == (4.0 if taken else None)


def test_committed_profiles_hold_kernels_of_known_shapes():
    """Every committed profile that a roofline reads has its kernel."""
    for kernel, profile, flags in (("k_diffuse", "pmc_traffic_config3_diurnal.json", 0),
                                   ("k_diffuse", "pmc_traffic_config2.json", 0),
                                   ("k_diffuse", "pmc_traffic_homogeneous_canopy.json", 1),
                                   ("k_cast", "pmc_traffic_config5_castrays.json", 0),
                                   ("k_camera", "pmc_traffic_config5_camera.json", 0)):
        assert bench.pmc_profile(kernel, profile, flags), (kernel, profile)
