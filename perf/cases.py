"""The work a user of this framework has it do, as cases that can be timed.

A case goes through the public Python entry points of woxel_amd as a program would
call them: frames and ray lists against a resident grid, shaded frames, batches of
requests over one or several grids, and the build of a scene up to its first frame.
Sizes come from the benchmark's configurations and the tests, with odd ones beside
the round ones.

  listed()            the cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) what the program holds before the call (grid, camera, buffers)
  run(state)          one pass, returning what it computes
  work(case)          bytes and floating-point operations a pass cannot do without

Hit records and rgba8 pixels are bytes and words: they are the same on every
correct build. The float colours of the shaded f32 frames have no 64-bit
counterpart: a ray traced in 64 bits takes other steps than one in 32 bits and can
meet another voxel, so exact() gives no value for them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import woxel_amd as wx
from woxel_amd import scenes

# Scenes: "ball" is one solid sphere seen from outside its node, "spheres" a set of
# spheres in a cubic domain, "noise" a value-noise isosurface (device-built).


def listed():
    return [
        # a thumbnail of the single-sphere scene: a launch of a few waves, all latency
        dict(name="thumbnail_64x48", kind="camera", scene="ball", side=256, width=64, height=48),
        # the single-sphere frame at its ordinary size
        dict(name="frame_ball_640x480", kind="camera", scene="ball", side=256, width=640, height=480),
        # the headline frame: an orbit camera over 2000 spheres in a 4096^3 domain
        dict(name="frame_spheres_1080p", kind="camera", scene="spheres", side=4096, count=2000, width=1920, height=1080),
        # a large frame of an odd size close to 4K, over a dense isosurface
        dict(name="frame_noise_3837x2157", kind="camera", scene="noise", side=1024, occupancy=0.15, width=3837,
             height=2157),
        # picking and line-of-sight queries: a few hundred arbitrary rays
        dict(name="rays_501", kind="rays", scene="noise", side=512, occupancy=0.1, rays=501, pattern="scattered"),
        # a panorama from inside the scene: a camera the library has not, given as its rays in
        # scan order
        dict(name="rays_panorama_1023x511", kind="rays", scene="spheres", side=2048, count=1000, rays=522753,
             pattern="panorama"),
        # the incoherent pass of the benchmark: 16 Mi rays over the sphere set
        dict(name="rays_16777216", kind="rays", scene="spheres", side=4096, count=2000, rays=16777216,
             pattern="scattered"),
        # a shaded frame, primary and sun shadow rays, as rgba8
        dict(name="render_diffuse_1080p", kind="render", scene="spheres", side=4096, count=2000, width=1920, height=1080,
             mode=3, f32=False),
        # a shaded frame with two reflection bounces, as float colours, an odd size
        dict(name="render_glossy_1279x717", kind="render", scene="noise", side=768, occupancy=0.08, width=1279,
             height=717, mode=4, f32=True),
        # many small requests over several resident grids in one call
        dict(name="batch_small_24", kind="batch", scene="noise", side=384, occupancy=0.1, grids=4, requests=24, lo=96,
             hi=384, shadow=True),
        # larger requests with shadow rays over one big grid in one call
        dict(name="batch_shadow_12", kind="batch", scene="spheres", side=4096, count=2000, grids=1, requests=12, lo=256,
             hi=1920, shadow=True),
        # a scene from its parameters to its first frame: voxels, grid SDF, device grid
        dict(name="build_noise_768", kind="build", scene="noise", side=768, occupancy=0.15, width=640, height=480),
    ]


def _log(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def _scene(rng, noise_max=1024):
    if rng.random() < 0.5:
        side = int(round(_log(rng, 1024, 4096) / 8)) * 8
        return dict(scene="spheres", side=side, count=int(_log(rng, 200, 2000)))
    return dict(scene="noise", side=int(round(_log(rng, 256, noise_max) / 8)) * 8,
                occupancy=round(rng.uniform(0.01, 0.2), 3))


def draw(rng):
    kind = rng.choice(["camera", "camera", "rays", "rays", "render", "batch", "build"])
    c = dict(kind=kind)
    if kind == "camera":
        c.update(dict(scene="ball", side=256) if rng.random() < 0.25 else _scene(rng))
        w = int(_log(rng, 48, 3800))
        c.update(width=w, height=max(1, int(w * rng.uniform(0.5, 0.57))))
    elif kind == "rays":
        c.update(_scene(rng))
        if c["scene"] == "spheres" and rng.random() < 0.5:
            w = int(_log(rng, 32, 2900))
            c.update(rays=w * (w // 2), pattern="panorama")
        else:
            c.update(rays=int(_log(rng, 1, 16000000)), pattern="scattered")
    elif kind == "render":
        c.update(_scene(rng))
        w = int(_log(rng, 64, 1920))
        c.update(width=w, height=max(1, int(w * rng.uniform(0.5, 0.57))), mode=rng.choice([0, 1, 2, 3, 3, 4, 4]),
                 f32=rng.random() < 0.3)
    elif kind == "batch":
        c.update(_scene(rng, noise_max=640))
        big = c["scene"] == "spheres"
        c.update(grids=1 if big else rng.randint(1, 4), requests=rng.randint(2, 12 if big else 32), lo=64,
                 hi=int(_log(rng, 128, 1920 if big else 512)), shadow=rng.random() < 0.7)
    else:
        c.update(scene="noise", side=int(round(_log(rng, 128, 768) / 8)) * 8, occupancy=round(rng.uniform(0.01, 0.15), 3),
                 width=int(_log(rng, 64, 800)), height=int(_log(rng, 48, 600)))
    return c


# ---------------- scenes ----------------

def _build(case, seed):
    """The unfinished and then finished tree of a case's scene, and its device grid."""
    v = wx.Vdb345()
    side = case["side"]
    if case["scene"] == "ball":
        v.add_spheres(scenes.single_sphere())
        v.compute_sdf()
    elif case["scene"] == "spheres":
        v.add_spheres(scenes.sphere_set(seed, count=case["count"], domain=side), (0, 0, 0), (side, side, side))
        v.compute_sdf(device=True)
    else:
        v.add_noise(seed, (0, 0, 0), (side, side, side), 8.0 / side, case["occupancy"], device=True)
        v.compute_sdf(device=True)
    return wx.Grid(v)


def _spec(case, rng, width, height):
    """A camera around the case's scene: the ball from its usual distance, the other
    scenes from 1.46 sides away, looking at the centre of the domain."""
    side = case["side"]
    c = 128.0 if case["scene"] == "ball" else side / 2.0
    az, el = rng.uniform(0.0, 2.0 * math.pi), math.radians(rng.uniform(-40.0, 40.0))
    d = np.array([math.cos(el) * math.cos(az), math.sin(el), math.cos(el) * math.sin(az)])
    r, fov = (460.0, 60.0) if case["scene"] == "ball" else (1.46 * side, 45.0)
    return scenes.look_at_spec(np.array([c, c, c]) + r * d, (c, c, c), width, height, fov)


def _sizes(case):
    """The images of a batch: widths spread evenly over the logarithm of lo..hi, in
    an order of large and small mixed, 16:9."""
    m = case["requests"]
    widths = [int(round(case["lo"] * (case["hi"] / case["lo"]) ** (k / max(1, m - 1)))) for k in range(m)]
    order = sorted(range(m), key=lambda k: k * 0.618034 % 1.0)
    return [(widths[k], max(1, int(round(widths[k] * 0.5625)))) for k in order]


def _records(n):
    return torch.empty((n, 32), dtype=torch.uint8, device="cuda")


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    st = dict(case=case, seed=seed)
    if kind == "build":
        st["cam"] = scenes.basis(_spec(case, rng, case["width"], case["height"]))
        st["out"] = _records(case["width"] * case["height"])
        return st
    if kind == "batch":
        st["grids"] = [_build(case, seed * 16 + k) for k in range(case["grids"])]
        reqs, n = [], 0
        for k, (w, h) in enumerate(_sizes(case)):
            reqs.append((k % case["grids"], scenes.basis(_spec(case, rng, w, h)), w, h, n))
            n += w * h
        st["out"] = _records(n)
        st["shadow"] = _records(n) if case["shadow"] else None
        st["requests"] = [
            wx.camera_request(g, cam, w, h, st["out"][at:at + w * h],
                              shadow_out=st["shadow"][at:at + w * h] if case["shadow"] else None)
            for g, cam, w, h, at in reqs]
        return st
    st["grid"] = _build(case, seed)
    if kind == "rays":
        st["rays"] = _panorama(case, rng) if case["pattern"] == "panorama" else _scattered(case, seed)
        st["out"] = _records(case["rays"])
        return st
    w, h = case["width"], case["height"]
    st["cam"] = scenes.basis(_spec(case, rng, w, h))
    if kind == "camera":
        st["out"] = _records(w * h)
    else:
        st["shade"] = wx.shade(case["mode"])
        st["out"] = (torch.empty((w * h, 4), dtype=torch.float32, device="cuda") if case["f32"]
                     else torch.empty(w * h, dtype=torch.int32, device="cuda"))
    return st


def _panorama(case, rng):
    """Every direction from one eye near the middle of the domain, twice as wide as
    high, row by row."""
    h = int(math.sqrt(case["rays"] / 2.0))
    w = case["rays"] // h
    eye = case["side"] * rng.uniform(0.4, 0.6, 3)
    i = torch.arange(case["rays"], device="cuda")
    az = ((i % w).float() + 0.5) * (2.0 * math.pi / w)
    el = math.pi / 2.0 - ((i // w).float() + 0.5) * (math.pi / h)
    d = torch.stack([el.cos() * az.cos(), el.sin(), el.cos() * az.sin()], dim=1)
    o = torch.tensor(eye, dtype=torch.float32, device="cuda").expand_as(d)
    return torch.cat([o, d], dim=1).contiguous()


def _scattered(case, seed):
    """Origins uniform on the domain's bounding sphere, directions uniform: rays that
    have nothing to do with their neighbours in the list."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    n, c = case["rays"], case["side"] / 2.0
    o = torch.randn((n, 3), generator=g, device="cuda", dtype=torch.float32)
    d = torch.randn((n, 3), generator=g, device="cuda", dtype=torch.float32)
    o = c + c * math.sqrt(3.0) * o / o.norm(dim=1, keepdim=True)
    d = d / d.norm(dim=1, keepdim=True)
    d = torch.where(d.abs() < 1e-7, torch.where(d < 0, -1e-7, 1e-7), d)
    return torch.cat([o, d], dim=1).contiguous()


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "camera":
        return st["grid"].trace_camera(st["cam"], case["width"], case["height"], 0.5, clip=True, out=st["out"])
    if kind == "rays":
        return st["grid"].trace_rays(st["rays"], clip=True, out=st["out"])
    if kind == "render":
        return st["grid"].render_camera(st["cam"], case["width"], case["height"], st["shade"], 0.5, clip=True,
                                        f32=case["f32"], out=st["out"])
    if kind == "batch":
        wx.trace_batch(st["grids"], st["requests"])
        return [st["out"], st["shadow"]] if case["shadow"] else st["out"]
    g = _build(case, st["seed"])
    st["grid"] = g  # the program goes on with the new grid; the one before is dropped
    out = g.trace_camera(st["cam"], case["width"], case["height"], 0.5, clip=True, out=st["out"])
    return [out, *g.counts]


# Floating-point operations of one traversal step: bound test, three quotients and
# remainders, three distances, their minimum, the advance and the nudge.
STEP_FLOPS = 50.0
# Traversal steps of a ray on average, about: a frame's ray, a scattered ray.
FRAME_STEPS = {"ball": 15.0, "spheres": 37.0, "noise": 30.0}
RAY_STEPS = {"spheres": 12.0, "noise": 15.0}


def work(case):
    kind = case["kind"]
    if kind == "rays":
        n = float(case["rays"])
        steps = FRAME_STEPS[case["scene"]] if case["pattern"] == "panorama" else RAY_STEPS[case["scene"]]
        return dict(bytes=n * (24 + 32), flops=n * steps * STEP_FLOPS)
    if kind == "batch":
        n = float(sum(w * h for w, h in _sizes(case)))
        return dict(bytes=n * 32 * (2 if case["shadow"] else 1),
                    flops=n * FRAME_STEPS[case["scene"]] * STEP_FLOPS * (1.1 if case["shadow"] else 1.0))
    n = float(case["width"] * case["height"])
    steps = FRAME_STEPS[case["scene"]] * STEP_FLOPS
    if kind == "camera":
        return dict(bytes=n * 32, flops=n * steps)
    if kind == "render":
        rays = 1.0 if case["mode"] <= 2 else (1.3 if case["mode"] == 3 else 2.0)
        return dict(bytes=n * (16 if case["f32"] else 4), flops=n * steps * rays)
    # a build: every leaf's mask and layout words once, 13 neighbours twice per voxel of
    # the leaves, and the frame
    leaves = 1.25 * case["occupancy"] * (case["side"] / 8.0) ** 3
    return dict(bytes=leaves * (64 + 256) + n * 32, flops=leaves * 512 * 2 * 13 + n * steps)


def exact(case, seed):
    """No 64-bit value: records and words are compared as they are (see the top)."""
    return None
