"""Work that programs on this framework do, as measurable cases: whole radiation solves (plain, batched over suns,
served, driven call by call), closest-hit ray casts, a camera image and a scene update.

Every case is one call sequence through the public Python binding (``helios_amd.native``) on a seeded synthetic
scene of ``helios_amd.scenes``.  ``listed()`` holds the cases, ``draw()`` gives others of the same ranges,
``prepare()`` makes what a program holds before the call, ``run()`` is one pass, ``work()`` the bytes and
operations a pass cannot do without and ``exact()`` the same results by brute force in 64 bits where the sizes
allow it.
"""
import math

import numpy as np
import torch

from helios_amd import native, scenes
from helios_amd import workloads as W

SIGMA = 5.6703744e-8


def listed():
    return [
        # The smallest solve: one plant's leaves over a ground patch, one band, three scattering passes.  Solved
        # again for every hour or leaf state of a small model, so launches and latency count.
        {"name": "solve_small", "kind": "solve", "scene": "leaves", "prims": 1601, "bands": 1, "rays": 100, "depth": 3,
         "sky": False},
        # A stand of triangle leaves with periodic sides, two shortwave bands and a power-law sky: the usual
        # plot-scale canopy (periodic wraps in every pass, direct rays through the tree).
        {"name": "solve_periodic", "kind": "solve", "scene": "periodic", "prims": 60400, "bands": 2, "rays": 400,
         "depth": 2, "sky": True},
        # One instant of an orchard of a million primitives in three bands (thermal emission among them).
        {"name": "solve_orchard", "kind": "solve", "scene": "orchard", "prims": 1001600, "bands": 3, "rays": 200,
         "depth": 4, "sky": False},
        # A day of that orchard's ten-tree block: 64 suns x 3 bands in one batched solve, results left on the device.
        {"name": "day_batched", "kind": "day", "prims": 401600, "suns": 64, "rays": 200, "depth": 4},
        # Leaves cut out of rectangles by a texture mask in a periodic domain, direct and then diffuse light, one
        # band a call, without scattering: the reference's homogeneous-canopy benchmark on a smaller plot.
        {"name": "masked_leaves", "kind": "masked", "prims": 140000, "rays": 1024},
        # A growth chamber under lamps (rectangle, disk and sphere sources), driven call by call as the plugin's own
        # runBand loop drives a backend, with two bands and one scattering iteration.
        {"name": "lamp_chamber", "kind": "lamps", "prims": 20100, "lamps": 3, "rays": 256, "depth": 1},
        # A request server over four resident canopies: a burst of single-sun requests, answered in batches.
        {"name": "serve_burst", "kind": "serve", "prims": 150000, "models": 4, "requests": 16, "rays": 100, "depth": 2},
        # A radiation camera's image and its pixel labels over the orchard, three bands.
        {"name": "camera_image", "kind": "camera", "prims": 1001600, "side": 512, "samples": 16},
        # A handful of rays (line-of-sight and collision queries), host arrays: the smallest call there is.
        {"name": "cast_few", "kind": "cast", "prims": 20000, "rays": 1000},
        # One frame of a terrestrial laser scan, host arrays: pulses of seven sub-rays from one scanner position.
        {"name": "lidar_scan", "kind": "lidar", "prims": 400000, "rays": 700000},
        # Twenty million incoherent rays through five million triangles, everything on the device.
        {"name": "cast_bulk", "kind": "cast_device", "prims": 5008000, "rays": 20000000},
        # Leaves that moved between two steps: the scene is set up anew and a few thousand rays are cast into it.
        {"name": "scene_update", "kind": "update", "prims": 300000, "rays": 12000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "day", "masked", "lamps", "serve", "camera", "cast", "lidar", "cast_device",
                       "update"])
    if kind == "solve":
        scene = rng.choice(["leaves", "periodic", "orchard"])
        prims = _log(rng, *{"leaves": (500, 60000), "periodic": (3000, 60000), "orchard": (20000, 400000)}[scene])
        return {"kind": "solve", "scene": scene, "prims": prims, "bands": rng.randint(1, 3), "rays": _log(rng, 30, 400),
                "depth": rng.randint(0, 3), "sky": rng.random() < 0.3}
    if kind == "day":
        return {"kind": "day", "prims": _log(rng, 20000, 200000), "suns": rng.randint(3, 64), "rays": _log(rng, 50, 200),
                "depth": rng.randint(1, 4)}
    if kind == "masked":
        return {"kind": "masked", "prims": _log(rng, 12000, 140000), "rays": _log(rng, 100, 1024)}
    if kind == "lamps":
        return {"kind": "lamps", "prims": _log(rng, 1500, 20000), "lamps": rng.randint(1, 6), "rays": _log(rng, 30, 256),
                "depth": rng.randint(0, 2)}
    if kind == "serve":
        return {"kind": "serve", "prims": _log(rng, 10000, 150000), "models": rng.randint(1, 4),
                "requests": rng.randint(2, 16), "rays": _log(rng, 30, 100), "depth": rng.randint(0, 2)}
    if kind == "camera":
        return {"kind": "camera", "prims": _log(rng, 20000, 1000000), "side": rng.randint(100, 512),
                "samples": rng.randint(1, 16)}
    if kind == "cast":
        return {"kind": "cast", "prims": _log(rng, 1000, 100000), "rays": _log(rng, 10, 20000)}
    if kind == "lidar":
        return {"kind": "lidar", "prims": _log(rng, 20000, 400000), "rays": 7 * _log(rng, 3000, 100000)}
    if kind == "cast_device":
        return {"kind": "cast_device", "prims": _log(rng, 200000, 2000000), "rays": _log(rng, 100000, 20000000)}
    return {"kind": "update", "prims": _log(rng, 5000, 300000), "rays": _log(rng, 500, 12000)}


# ---- scenes ---------------------------------------------------------------------------------------------------


def _leaves(seed, prims):
    """Square 0.1 m leaves over one ground patch (the 1,600-leaf plant), more of them over a larger plot."""
    if prims == 1601:
        return scenes.config1(seed)
    side = 2.0 * math.sqrt(prims / 1600.0)
    return scenes.patch_canopy(seed, prims - 1, 0.1, side, 1.0, 1)


def _orchard(seed, prims):
    """Rows of trees of 40,000 triangles over 1,600 ground patches; smaller trees below a block of five."""
    trees = min(25, max(5, prims // 40000))
    per = (prims - 1600) // trees
    tubes = max(8, per // 20)
    return scenes.orchard(seed, nx=5, ny=max(1, trees // 5), leaves_per_tree=max(8, per - tubes), tube_tris=tubes)


def _scene(case, seed):
    if case["scene"] == "leaves":
        return _leaves(seed, case["prims"])
    if case["scene"] == "periodic":
        return scenes.config2(seed, nleaves=case["prims"] - 400)
    return _orchard(seed, case["prims"])


# ---- prepare --------------------------------------------------------------------------------------------------


def prepare(case, seed):
    seed = int(seed) % (1 << 24) + 1
    rng = np.random.default_rng(seed)
    ctx = native.Context(0)
    st = {"case": case, "ctx": ctx, "kind": case["kind"]}
    st.update(_PREPARE[case["kind"]](case, seed, rng, ctx))
    return st


def _resident(ctx, s):
    return ctx.scene(s.transforms, s.types, s.twosided, periodic=s.periodic)


def _sun(rng):
    return native.sun_direction(rng.uniform(15.0, 60.0), rng.uniform(90.0, 270.0))


def _prepare_solve(case, seed, rng, ctx):
    s = _scene(case, seed)
    bands = ["PAR", "NIR", "LW"][: case["bands"]]
    rho, tau, eps = W.optical_arrays(s, bands)
    emits = "LW" in bands
    B, depth = len(bands), case["depth"]
    spec = [native.BandSpec(b, depth, b == "LW", float(q)) for b, q in zip(bands, (110.0, 75.0, 330.0))]
    flux = np.array([[520.0, 430.0, 0.0][:B]], np.float32)
    sun = _sun(rng)
    sky = {}
    if case["sky"]:
        # power law of the angle from the sun, normalised over the hemisphere by the caller as the plugin does
        k = 0.35
        sky = {"sky_extinction": [k] * B, "sky_peak_dir": [sun] * B, "sky_norm": [_power_law_norm(k)] * B}
    req = native.BandRequest(s.P, spec, rho=rho, tau=tau, eps=eps if emits else None,
                             temperature=rng.uniform(290.0, 300.0, s.P).astype(np.float32) if emits else None,
                             direct_rays=case["rays"], diffuse_rays=case["rays"], source_dirs=[sun], source_flux=flux,
                             direct_seed=seed * 7 + 1, diffuse_seeds=[seed * 11 + 3 + k for k in range(depth + 1)], **sky)
    return {"scene": _resident(ctx, s), "req": req, "arrays": s}


def _power_law_norm(k, n=64):
    """1 / (1/pi x the hemisphere integral of psi^-k cos(theta)) for a peak at the zenith."""
    th = (np.arange(n) + 0.5) * (math.pi / 2 / n)
    psi = np.maximum(th, math.pi / 180)
    return 1.0 / float(np.sum(psi ** -k * np.cos(th) * np.sin(th)) * (math.pi / 2 / n) * 2.0)


def _prepare_day(case, seed, rng, ctx):
    s = _orchard(seed, case["prims"])
    req = W.diurnal_request(s, rays=case["rays"], depth=case["depth"])
    dirs, flux, sky, seeds = W.diurnal_suns(case["suns"], seed)
    out = torch.empty((case["suns"], s.P, req.B), dtype=torch.float32, device="cuda")
    return {"scene": _resident(ctx, s), "req": req, "suns": (dirs, flux, sky, seeds + np.uint32(seed)), "out": out}


def _prepare_masked(case, seed, rng, ctx):
    leaf = 0.05 * 0.05 * math.pi / 4
    side = math.sqrt(max(case["prims"] - 10000, 400) / 4 * leaf)
    s, masks, ids, uv, uv_ids = scenes.homogeneous_canopy(seed, D=side, mask_res=800)
    g = _resident(ctx, s)
    g.set_masks(masks, ids, uv, uv_ids)
    zero = np.zeros((s.P, 1), np.float32)
    direct = native.BandRequest(s.P, [native.BandSpec("direct", 0, False, 0.0)], rho=zero, tau=zero,
                                direct_rays=case["rays"], diffuse_rays=0, source_dirs=[_sun(rng)],
                                source_flux=[[1.0]], direct_seed=seed)
    diffuse = native.BandRequest(s.P, [native.BandSpec("diffuse", 0, False, 1.0)], rho=zero, tau=zero, direct_rays=0,
                                 diffuse_rays=case["rays"], diffuse_seeds=[seed + 5])
    return {"scene": g, "reqs": (direct, diffuse)}


def _prepare_lamps(case, seed, rng, ctx):
    P = case["prims"]
    side = 0.02 * math.sqrt(P)
    s = scenes.patch_canopy(seed, P - 100, 0.05, side, 0.8, 10)
    n = case["lamps"]
    kinds = [native.SOURCE_RECTANGLE, native.SOURCE_DISK, native.SOURCE_SPHERE]
    types = [kinds[k % 3] for k in range(n)]
    pos = np.stack([rng.uniform(-0.4 * side, 0.4 * side, n), rng.uniform(-0.4 * side, 0.4 * side, n),
                    rng.uniform(1.5, 1.8, n)], 1)
    widths = [{native.SOURCE_RECTANGLE: (0.6, 0.3), native.SOURCE_DISK: (0.2, 0.2)}.get(t, (0.12, 0.12)) for t in types]
    rot = np.stack([np.full(n, math.pi), rng.uniform(-0.1, 0.1, n), rng.uniform(0, math.pi, n)], 1)
    rho, tau, _ = W.optical_arrays(s, ["PAR", "NIR"])
    be = native.Backend(ctx)
    be.update_geometry(s.transforms, s.types, s.twosided)
    be.build_acceleration_structure()
    be.update_materials(np.repeat(rho[None], n, 0), np.repeat(tau[None], n, 0))
    be.update_sources(pos, types, widths, rot)
    return {"backend": be, "onesided": s.twosided == 0, "flux": np.tile([[900.0, 300.0]], (n, 1)).astype(np.float32),
            "seed": seed}


def _prepare_serve(case, seed, rng, ctx):
    models = []
    for m in range(case["models"]):
        s = scenes.mixed_canopy(seed + m, case["prims"] >> m)
        bands = ["PAR", "NIR", "PAR", "NIR"][: 1 + m]
        rho, tau, _ = W.optical_arrays(s, bands)
        req = native.BandRequest(s.P, [native.BandSpec(b, case["depth"], False, 100.0) for b in bands], rho=rho, tau=tau,
                                 direct_rays=case["rays"], diffuse_rays=case["rays"], source_dirs=[[0.0, 0.0, 1.0]],
                                 source_flux=[[500.0] * len(bands)], direct_seed=1,
                                 diffuse_seeds=[seed + 10 * m + k for k in range(case["depth"] + 1)])
        models.append((s, req))
    srv = native.Server(ctx, slots=3, max_batch_suns=32)
    held = [_resident(ctx, s) for s, _ in models]
    ids = [srv.add_model(g, req) for g, (_, req) in zip(held, models)]
    reqs = []
    for k in range(case["requests"]):
        req = models[k % len(models)][1]
        reqs.append((ids[k % len(models)], [_sun(rng)], req.sflux * np.float32(rng.uniform(0.5, 1.5)),
                     req.dflux * np.float32(rng.uniform(0.5, 1.5)), int(rng.integers(1, 1 << 31))))
    return {"server": srv, "held": held, "models": models, "requests": reqs}


def _prepare_camera(case, seed, rng, ctx):
    s = _orchard(seed, case["prims"])
    be = native.Backend(ctx)
    B = 3
    be.update_geometry(s.transforms, s.types, s.twosided)
    be.build_acceleration_structure()
    be.update_materials(np.full((s.P, B), 0.1, np.float32), np.full((s.P, B), 0.05, np.float32))
    sun = _sun(rng)
    be.update_sources([sun])
    be.zero_radiation_buffers(B)
    be.upload_radiation_out(rng.uniform(0, 300, (s.P, B)).astype(np.float32),
                            rng.uniform(0, 100, (s.P, B)).astype(np.float32))
    be.upload_source_fluxes(np.array([[400.0, 300.0, 500.0]], np.float32))
    be.update_sky_model(np.tile(np.array([2.0, 30.0, 1.5, 0.25], np.float32), (B, 1)),
                        np.array([20.0, 15.0, 30.0], np.float32), sun, np.array([4e3, 3e3, 5e3], np.float32),
                        math.cos(math.radians(0.27)), np.zeros(B, np.float32), np.zeros(B, np.uint32))
    T = s.transforms.reshape(-1, 16)
    x0, x1, y0, y1 = float(T[:, 3].min()), float(T[:, 3].max()), float(T[:, 7].min()), float(T[:, 7].max())
    cam = native.Camera(((x0 + x1) / 2, y0 - 0.3 * (y1 - y0), 8.0), (math.radians(115.0), 0.0),
                        (case["side"], case["side"]), viewplane_length=0.5 / math.tan(math.radians(30.0)),
                        antialiasing_samples=case["samples"])
    return {"backend": be, "camera": cam, "seed": seed}


def _box(s):
    T = s.transforms.reshape(-1, 16)
    return [float(T[:, 3].min()), float(T[:, 7].min()), 0.0], [float(T[:, 3].max()), float(T[:, 7].max()),
                                                              float(T[:, 11].max())]


def _prepare_cast(case, seed, rng, ctx):
    s = scenes.mixed_canopy(seed, case["prims"])
    O, D = scenes.rays(seed + 1, case["rays"], *_box(s))
    return {"scene": _resident(ctx, s), "rays": (O, D), "arrays": s}


def _prepare_lidar(case, seed, rng, ctx):
    s = scenes.mixed_canopy(seed, case["prims"])
    lo, hi = _box(s)
    beams = case["rays"] // 7
    nph = max(1, int(math.sqrt(beams * 3.0)))
    k = np.arange(beams)
    th = math.radians(60.0) + (k // nph) * (math.radians(70.0) / max(1, beams // nph))
    ph = (k % nph) * (2 * math.pi / nph)
    beam = np.stack([np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th)], 1)
    D = np.repeat(beam, 7, 0) + rng.normal(0, 1e-3, (beams * 7, 3))
    D /= np.linalg.norm(D, axis=1, keepdims=True)
    O = np.tile([[0.5 * (lo[0] + hi[0]), 0.5 * (lo[1] + hi[1]), hi[2] + 0.3]], (beams * 7, 1))
    return {"scene": _resident(ctx, s), "rays": (O.astype(np.float32), D.astype(np.float32))}


def _prepare_cast_device(case, seed, rng, ctx):
    P = case["prims"]
    s = scenes.orchard(seed, tiles=5, jitter=0.05) if P == 5008000 else _orchard(seed, P)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n = case["rays"]
    lo, hi = (torch.tensor(v, device="cuda") for v in _box(s))
    O = lo + (hi - lo) * torch.rand((n, 3), device="cuda", generator=gen)
    D = torch.nn.functional.normalize(torch.randn((n, 3), device="cuda", generator=gen), dim=1)
    out = [torch.zeros(n, device="cuda"), torch.zeros((n, 3), device="cuda"),
           torch.zeros(n, dtype=torch.int32, device="cuda")]
    torch.cuda.synchronize()
    return {"scene": _resident(ctx, s), "rays": (O, D), "out": out}


def _prepare_update(case, seed, rng, ctx):
    s = scenes.mixed_canopy(seed, case["prims"])
    O, D = scenes.rays(seed + 1, case["rays"], *_box(s))
    return {"arrays": s, "rays": (O, D)}


_PREPARE = {"solve": _prepare_solve, "day": _prepare_day, "masked": _prepare_masked, "lamps": _prepare_lamps,
            "serve": _prepare_serve, "camera": _prepare_camera, "cast": _prepare_cast, "lidar": _prepare_lidar,
            "cast_device": _prepare_cast_device, "update": _prepare_update}


# ---- run ------------------------------------------------------------------------------------------------------


def run(st):
    return _RUN[st["kind"]](st)


def _run_solve(st):
    return native.run_band(st["scene"], st["req"])


def _run_day(st):
    dirs, flux, sky, seeds = st["suns"]
    native.run_band_batch(st["scene"], st["req"], dirs, flux, sky, seeds, out_device_ptr=st["out"].data_ptr())
    return st["out"]


def _run_masked(st):
    return [native.run_band(st["scene"], r) for r in st["reqs"]]


def _run_lamps(st):
    """The pass loop of RadiationModel::runBand over the backend's calls: direct light, the scattered part handed on,
    one diffuse launch per face and iteration, and the sum of what stayed."""
    be, one, rays, depth, seed = (st["backend"], st["onesided"], st["case"]["rays"], st["case"]["depth"], st["seed"])
    B = st["flux"].shape[1]
    sky, dark = np.full(B, 5.0, np.float32), np.zeros(B, np.float32)
    be.zero_radiation_buffers(B)
    be.upload_source_fluxes(st["flux"])
    be.launch_direct_rays(rays, seed, B)
    r = be.get_radiation_results()
    top, bottom = r["scatter_buff_top"], r["scatter_buff_bottom"]
    both = top[one] + bottom[one]
    top[one], bottom[one] = both, both
    be.upload_radiation_out(top, bottom)
    be.zero_scatter_buffers()
    for face in (1, 0):
        be.launch_diffuse_rays(rays, seed + 1, B, face, diffuse_flux=sky, radiation_out=(top, bottom))
    for k in range(depth):
        if k:
            be.copy_scatter_to_radiation()
        be.zero_scatter_buffers()
        r = be.get_radiation_results()
        out = (r["radiation_out_top"], r["radiation_out_bottom"])
        for face in (1, 0):
            be.launch_diffuse_rays(rays, seed + 2 + k, B, face, diffuse_flux=dark, radiation_out=out)
    r = be.get_radiation_results()
    return r["radiation_in"] + r["scatter_buff_top"] + r["scatter_buff_bottom"]


def _run_serve(st):
    srv = st["server"]
    tickets = [srv.submit(*q) for q in st["requests"]]
    return [srv.wait(t)[0] for t in tickets]


def _run_camera(st):
    be, cam = st["backend"], st["camera"]
    be.zero_camera_pixel_buffers(cam.resolution)
    be.launch_camera_rays(cam, seed=st["seed"])
    be.launch_pixel_label_rays(cam)
    return be.get_camera_results(cam.resolution)


def _run_cast(st):
    return st["scene"].cast_rays(*st["rays"])


def _run_lidar(st):
    return st["scene"].lidar_cast_rays(*st["rays"], packet_size=7, miss_t=1001.0)


def _run_cast_device(st):
    (O, D), (t, n, u) = st["rays"], st["out"]
    st["scene"].cast_rays_device(O.data_ptr(), D.data_ptr(), O.shape[0], -1.0, t.data_ptr(), n.data_ptr(), u.data_ptr())
    return st["out"]


def _run_update(st):
    s = st["arrays"]
    g = st["ctx"].scene(s.transforms, s.types, s.twosided)
    out = g.cast_rays(*st["rays"])
    g.close()
    return out


_RUN = {"solve": _run_solve, "day": _run_day, "masked": _run_masked, "lamps": _run_lamps, "serve": _run_serve,
        "camera": _run_camera, "cast": _run_cast, "lidar": _run_lidar, "cast_device": _run_cast_device,
        "update": _run_update}


# ---- work -----------------------------------------------------------------------------------------------------


def _rays_of(P, n, passes):
    """Rays of diffuse passes over P primitives: n x n (n = ceil sqrt of the count) from each of two faces."""
    k = math.ceil(math.sqrt(n)) ** 2
    return 2 * P * k * passes


def work(case):
    """Bytes: the scene's geometry (64 B a primitive) and a pass's own inputs, read once, its results written once.
    Operations: each ray's generation, one descent of a four-wide tree (its depth x four boxes) and one primitive."""
    P, kind = case["prims"], case["kind"]
    per_ray = 60 + 48 * max(1.0, math.log(max(P, 4), 4)) + 50
    if kind in ("solve", "day"):
        B, K = (3, case["suns"]) if kind == "day" else (case["bands"], 1)
        direct = K * P * math.ceil(math.sqrt(case["rays"])) ** 2
        rays = direct + _rays_of(P, case["rays"], 1 + case["depth"])
        gathered = _rays_of(P, case["rays"], 1 + case["depth"]) * K * B
        return {"bytes": P * (76 + 8 * B + 4 * K * B), "flops": rays * per_ray + 2 * gathered}
    if kind == "masked":
        n = math.ceil(math.sqrt(case["rays"])) ** 2
        return {"bytes": P * (76 + 32 + 24), "flops": 3 * P * n * per_ray}
    if kind == "lamps":
        n = math.ceil(math.sqrt(case["rays"])) ** 2
        return {"bytes": P * (76 + 56), "flops": (case["lamps"] * P * n + _rays_of(P, n, 1 + case["depth"])) * per_ray}
    if kind == "serve":
        n = case["requests"]
        mean = sum(P >> m for m in range(case["models"])) / case["models"]
        rays = mean * (math.ceil(math.sqrt(case["rays"])) ** 2) * n + _rays_of(mean, case["rays"], 1 + case["depth"]) * case["models"]
        return {"bytes": case["models"] * mean * 76 + n * mean * 10, "flops": rays * per_ray}
    if kind == "camera":
        rays = case["side"] ** 2 * (case["samples"] + 1)
        return {"bytes": P * (64 + 24) + case["side"] ** 2 * 20, "flops": rays * per_ray}
    if kind == "update":
        return {"bytes": P * (72 + 64 + 64 + 21) + case["rays"] * 44, "flops": P * 200 + case["rays"] * per_ray}
    return {"bytes": P * 64 + case["rays"] * 44, "flops": case["rays"] * per_ray}


# ---- the same results by brute force in 64 bits ---------------------------------------------------------------


def exact(case, seed):
    """Small solves over patches and casts of a few rays; None where every ray against every primitive takes too long."""
    if case["kind"] in ("cast", "update") and case["rays"] * case["prims"] < 4e9:
        st = prepare(case, seed)
        return _exact_cast(st["arrays"], *st["rays"])
    if case["kind"] == "solve" and case["scene"] == "leaves" and case["bands"] == 1 and not case["sky"]:
        if _rays_of(case["prims"], case["rays"], 1 + case["depth"]) * case["prims"] < 6e9:
            st = prepare(case, seed)
            return _exact_solve(st["arrays"], st["req"])
    return None


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _world(s):
    """Corner and edges of every primitive [P][3] and which are patches: a patch spans local (-0.5, -0.5) to (0.5,
    0.5), a triangle has the local vertices (0, 0), (0, 1) and (1, 1)."""
    T = torch.tensor(s.transforms.reshape(-1, 4, 4), dtype=torch.float64, device=_device())
    patch = torch.tensor((s.types == 0) | (s.types == 3), device=_device())
    x, y, c = T[:, :3, 0], T[:, :3, 1], T[:, :3, 3]
    corner = torch.where(patch[:, None], c - 0.5 * (x + y), c)
    e1 = torch.where(patch[:, None], x, y)
    e2 = torch.where(patch[:, None], y, x + y)
    return corner, e1, e2, patch


def _closest(world, O, D, tmin, skip=None, edge=0.0, chunk=1 << 24):
    """Distance (inf: none) and index of each ray's closest primitive beyond tmin, every ray against every primitive;
    triangles reach out by `edge` in their barycentric coordinates and are missed where |direction . (e1 x e2)| is
    below it."""
    v0, e1, e2, patch = world
    n = torch.linalg.cross(e1, e2)
    # a point v0 + u e1 + v e2 of the plane: u = w . a, v = w . b with the dual basis of (e1, e2)
    nn = (n * n).sum(1, keepdim=True)
    a, b = torch.linalg.cross(e2, n) / nn, torch.linalg.cross(n, e1) / nn
    nd, va, vb = (v0 * n).sum(1), (v0 * a).sum(1), (v0 * b).sum(1)
    top = torch.where(patch, 2.0, 1.0 + edge)
    edge = torch.where(patch, 0.0, edge)
    T, I = [], []
    step = max(1, chunk // v0.shape[0])
    for k in range(0, O.shape[0], step):
        o, d = O[k:k + step], D[k:k + step]
        dn = d @ n.T
        t = (nd - o @ n.T) / dn
        u = o @ a.T + t * (d @ a.T) - va
        v = o @ b.T + t * (d @ b.T) - vb
        ok = (t > tmin) & (dn.abs() > edge) & (u >= -edge) & (v >= -edge) & (u <= 1 + edge) & (v <= 1 + edge) & (u + v <= top)
        if skip is not None:
            ok &= torch.arange(v0.shape[0], device=t.device) != skip[k:k + step, None]
        t = torch.where(ok, t, math.inf)
        best = t.min(1)
        T.append(best.values)
        I.append(best.indices)
    return torch.cat(T), torch.cat(I)


def _exact_cast(s, O, D):
    world = _world(s)
    O, D = (torch.tensor(x, dtype=torch.float64, device=_device()) for x in (O, D))
    t, i = _closest(world, O, D, 1e-6, edge=1e-5)  # the triangle test of castRays
    n = torch.linalg.cross(world[1], world[2])[i]
    n = n / n.norm(dim=1, keepdim=True)
    n = torch.where((n * D).sum(1, keepdim=True) > 0, -n, n)
    miss = torch.isinf(t)
    t[miss] = math.nan
    n[miss] = math.nan
    return t, n, None


def _tea(v0, v1):
    """16 rounds of the Tiny Encryption Algorithm on 32-bit words (held in int64)."""
    m, s = 0xFFFFFFFF, 0
    for _ in range(16):
        s = (s + 0x9E3779B9) & m
        v0 = (v0 + ((((v1 << 4) & m) + 0xA341316C & m) ^ (v1 + s & m) ^ ((v1 >> 5) + 0xC8013EA4 & m))) & m
        v1 = (v1 + ((((v0 << 4) & m) + 0xAD90777D & m) ^ (v0 + s & m) ^ ((v0 >> 5) + 0x7E95761E & m))) & m
    return v0


def _uniform(state):
    """Next 24-bit uniform numbers of linear congruential states: (numbers, states)."""
    state = (1664525 * state + 1013904223) & 0xFFFFFFFF
    return (state & 0xFFFFFF).double() / 16777216.0, state


def _exact_solve(s, req):
    """One band, one distant sun, an even sky, patches only: direct light, the primary diffuse pass and the scattering
    iterations on the request's own rays (the primary pass's scatter is not handed on, as the schedule has it)."""
    dev, P = _device(), s.P
    world = _world(s)
    v0, e1, e2, _ = world
    normal = torch.linalg.cross(e1, e2)
    normal = normal / normal.norm(dim=1, keepdim=True)
    two = torch.tensor(s.twosided != 0, device=dev)
    rho, tau = (torch.tensor(x[:, 0], dtype=torch.float64, device=dev) for x in (req.rho, req.tau))
    prim = torch.arange(P, device=dev)

    def state(n, seed):
        r = torch.arange(n * n, device=dev)
        return r, _tea(((r[None] + n * n * prim[:, None]) & 0xFFFFFFFF), torch.full((P, n * n), seed & 0xFFFFFFFF, device=dev))

    # direct light: stratified points, lit when nothing lies towards the sun
    n = math.ceil(math.sqrt(req.direct_rays))
    r, z = state(n, req.direct_seed)
    x, z = _uniform(z)
    y, z = _uniform(z)
    x, y = ((r % n)[None] + x) / n, ((r // n)[None] + y) / n
    o = (v0[:, None] + x[..., None] * e1[:, None] + y[..., None] * e2[:, None]).reshape(-1, 3)
    sun = torch.tensor(req.sdir[0], dtype=torch.float64, device=dev)
    sun = sun / sun.norm()
    t, _ = _closest(world, o, sun.expand_as(o), 1e-4, prim.repeat_interleave(n * n))
    cosine = normal @ sun
    lit = torch.isinf(t).reshape(P, n * n).double().mean(1) * cosine.abs() * float(req.sflux[0, 0])
    up = cosine > 0
    lit = torch.where(up | two, lit, torch.zeros_like(lit))
    light = [torch.where(up, lit, 0.0), torch.where(up, 0.0, lit)]
    stays = sum(light) * (1 - rho - tau)
    out = [light[0] * rho + light[1] * tau, light[0] * tau + light[1] * rho]
    if max(req.depth) > 0:
        out = [torch.where(two, q, out[0] + out[1]) for q in out]
        scatter = [torch.zeros_like(rho)] * 2
    else:
        scatter, out = out, [torch.zeros_like(rho)] * 2

    # rotation of the zenith onto each normal: elevation from its z, azimuth from its x and y
    ce, se = normal[:, 2], (1 - normal[:, 2] ** 2).clamp(min=0).sqrt()
    az = torch.atan2(normal[:, 1], normal[:, 0])
    ca, sa = az.cos(), az.sin()
    n = math.ceil(math.sqrt(req.diffuse_rays))
    for k in range(1 + int(max(req.depth))):
        if k > 1:
            out = scatter
        if k > 0:
            scatter = [torch.zeros_like(rho)] * 2
        sky = float(req.dflux[0]) if k == 0 else 0.0
        r, z = state(n, int(req.dseeds[k]))
        x, z = _uniform(z)
        y, z = _uniform(z)
        rt, z = _uniform(z)
        rp, z = _uniform(z)
        o = (v0[:, None] + x[..., None] * e1[:, None] + y[..., None] * e2[:, None]).reshape(-1, 3)
        rt, phi = ((r % n)[None] + rt) / n, 2 * math.pi * ((r // n)[None] + rp) / n
        lx, ly, lz = rt.sqrt() * phi.cos(), rt.sqrt() * phi.sin(), (1 - rt).sqrt()
        c = [q[:, None] for q in (ce, se, ca, sa)]
        d = torch.stack([lx * c[0] * c[2] - ly * c[3] + lz * c[1] * c[2], lx * c[0] * c[3] + ly * c[2] + lz * c[1] * c[3],
                         -lx * c[1] + lz * c[0]], -1).reshape(-1, 3)
        come = []
        for sign in (1.0, -1.0):
            t, i = _closest(world, o, sign * d, 1e-5, prim.repeat_interleave(n * n))
            seen = torch.where((normal[i] * d).sum(1) * sign < 0, out[0][i], out[1][i])
            come.append(torch.where(torch.isinf(t), sky, seen).reshape(P, n * n).mean(1))
        come[1] = torch.where(two, come[1], 0.0)
        stays = stays + (come[0] + come[1]) * (1 - rho - tau)
        scatter = [scatter[0] + come[0] * rho + come[1] * tau, scatter[1] + come[0] * tau + come[1] * rho]
    return (stays + scatter[0] + scatter[1])[:, None]
