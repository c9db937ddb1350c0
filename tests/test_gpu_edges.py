"""Edges of the rules that choose a path, each against the oracle or the general path, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_trace import assert_hits_equal
from woxel_amd import scenes

pytestmark = pytest.mark.gpu


def same_but_nan(gpu, ora, what):
    """Every byte of the records, but for t where it is NaN on both sides (its bits are the hardware's)."""
    nan = np.isnan(ora["t"])
    assert np.array_equal(np.isnan(gpu["t"]), nan), what
    gpu, ora = gpu.copy(), ora.copy()
    gpu["t"][nan] = ora["t"][nan] = 0.0
    assert_hits_equal(gpu, ora, what)


@pytest.mark.parametrize("past", [-1, 0, 1])
def test_general_step_in_long_lists(wx, oracle_mod, cuda, past):
    """Lists one ray short of the length at which scattered sets of 64 go to the refilled waves,
    and past it; rays of the general step that run on (a start of -0) and that turn NaN (a
    direction component of -0) in scattered and in kept sets."""
    n = 64 * 64 * cuda.cuda.get_device_properties(0).multi_processor_count - 64 + past
    print(f"general step, {n} rays", flush=True)
    rng = np.random.default_rng(abs(past) + 3)
    sp = np.array([[2000.0, 1500.0, 1800.0, 60.0], [700.0, 900.0, 2500.0, 45.0], [300.0, 200.0, 250.0, 90.0]])
    p = wx.Vdb345()
    p.add_spheres(sp)
    p.compute_sdf()
    o = oracle_mod.Vdb()
    for s in sp:
        o.add_sphere(s[:3], s[3])
    o.compute_sdf()
    m = (n + 63) // 64 * 64
    eye = rng.uniform(-3000, 4000, (m, 3))
    d = sp[rng.integers(0, 3, m), :3] + rng.uniform(-60, 60, (m, 3)) - eye
    rays = np.concatenate([eye, d], 1).reshape(-1, 64, 6)
    rays[::3, :, :3] = rays[::3, :1, :3]  # one eye, neighbouring directions
    rays[::3, :, 3:] = rays[::3, :1, 3:] + rng.uniform(-20, 20, rays[::3, :, 3:].shape)
    rays = rays.reshape(m, 6)[:n]
    rays[:, 3:] /= np.linalg.norm(rays[:, 3:], axis=1, keepdims=True)
    rays = rays.astype(np.float32)
    zero = rng.choice(n, 8000, replace=False)
    rays[zero, rng.integers(0, 3, 8000)] = -0.0
    nan = rng.integers(0, n, 3000)
    rays[nan, 3 + rng.integers(0, 3, 3000)] = -0.0
    t = cuda.from_numpy(rays).cuda()
    g = wx.Grid(p)
    for clip in (False, True):
        ora, _ = o.trace_rays(rays, clip=clip)
        gpu = wx.hits_to_numpy(g.trace_rays(t, clip=clip))
        same_but_nan(gpu, ora, f"{n} rays, clip={clip}")
        ran = zero[~np.isnan(ora["t"][zero]) & (ora["steps"][zero].sum(1) > 3)]
        scattered = (ran // 64) % 3 != 0
        assert scattered.sum() > 1000 and (~scattered).sum() > 500
        assert (ora["state"][ran] == wx.HIT).sum() > 50


@pytest.mark.parametrize("bound", [4096.0, 2.0 ** 21])
def test_degenerate_rays_in_every_shape(wx, oracle_mod, cuda, bound):
    """Zeros, infinities, denormals and NaNs, quiet and signalling, in any component: every
    shape gives the oracle's records (t where it is NaN aside), with and without the clip."""
    print(f"degenerate rays, bound {bound}", flush=True)
    rng = np.random.default_rng(5)
    n = 64 * 300
    sp = np.array([[40.0, 30.0, 45.0, 22.0], [90.0, 60.0, 20.0, 14.0], [-45.0, 40.0, 30.0, 19.0]])
    r = np.concatenate([rng.uniform(-120, 120, (n, 3)), rng.standard_normal((n, 3))], 1).astype(np.float32)
    odd = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-40, -1e-39, 3e38, -3e38, 2.0 ** -64, -2.0 ** -66], np.float32)
    m = rng.random(r.shape) < 0.12
    r[m] = rng.choice(odd, m.sum())
    bits = r.view(np.uint32)
    m = np.isnan(r)
    bits[m] = (rng.integers(0, 2, m.sum()).astype(np.uint32) << 31) | 0x7F800000 | rng.integers(1, 1 << 23, m.sum()).astype(np.uint32)
    t = cuda.from_numpy(r).cuda()
    tune = wx.tune_get()
    for roots in (2, 3):
        p = wx.Vdb345()
        p.add_spheres(sp[:roots])
        p.compute_sdf()
        o = oracle_mod.Vdb()
        for s in sp[:roots]:
            o.add_sphere(s[:3], s[3])
        o.compute_sdf()
        g = wx.Grid(p, bound)
        for clip in (False, True):
            ora, _ = o.trace_rays(r, bound=bound, clip=clip)
            for persistent in (0, 1):
                print(f"{roots} spheres, clip {clip}, shape {persistent}", flush=True)
                tune.persistent = persistent
                for grids in ([g], [g, g]):
                    out = [cuda.empty((n, 32), dtype=cuda.uint8, device="cuda") for _ in grids]
                    wx.trace_batch(grids, [wx.rays_request(k, t, out[k], clip=clip) for k in range(len(grids))], tune)
                    for x in out:
                        same_but_nan(wx.hits_to_numpy(x), ora, f"{roots} {clip} {persistent} {len(grids)}")


def far_layout(wx, p):
    """The tree's layout with every second node-4 record finding its leaves in a copy further on."""
    lay = p.layout_arrays()
    n5, n4, n3 = lay["n"]
    rec4 = lay["n4"].copy()
    rec4[::2, 1] += n3 + 5000
    leaves = np.concatenate([lay["leaves"], np.zeros((5000, 64), np.uint32), lay["leaves"]])
    return lay["root"], lay["n5"], rec4, leaves


def grid_of(wx, root, n5, n4, leaves, bound=4096.0):
    keep = [np.ascontiguousarray(root, np.int32)] + [np.ascontiguousarray(a, np.uint32) for a in (n5, n4, leaves)]
    d = wx.GridDesc()
    d.n5, d.n4, d.n3, d.bound = keep[1].size // 16384, keep[2].size // 1024, keep[3].size // 64, bound
    d.root = keep[0].ctypes.data_as(C.POINTER(C.c_int32))
    d.n5_records, d.n4_records, d.leaves = [a.ctypes.data_as(C.POINTER(C.c_uint32)) for a in keep[1:]]
    return wx.Grid.from_desc(d)


def test_persistent_batches_of_every_form(wx, cuda):
    """Batches with shadow rays on one grid of each form and on grids of all forms together:
    the persistent shape gives the records of the one-lane shape, request by request."""
    print("persistent batches", flush=True)
    sp = np.array([[400.0, 300.0, 450.0, 120.0], [700.0, 600.0, 260.0, 90.0]])
    trees = []
    for shift in (0.0, -500.0):  # one node-5, eight
        p = wx.Vdb345()
        p.add_spheres(sp + [shift, shift, shift, 0.0])
        p.compute_sdf()
        trees.append(p)
    every = [wx.Grid(trees[0]), wx.Grid(trees[1]), grid_of(wx, *far_layout(wx, trees[0])), wx.Grid(trees[0], 2.0 ** 20 + 1)]
    w, h = 161, 93
    for grids in ([every[0]], [every[1]], [every[2]], [every[3]], every):
        print(f"{len(grids)} grids", flush=True)
        got = {}
        for persistent in (0, 1):
            out = [cuda.zeros((w * h, 32), dtype=cuda.uint8, device="cuda") for _ in range(8)]
            reqs = []
            for k in range(4):
                g = k % len(grids)
                shift = 500.0 if grids[g] is every[1] else 0.0
                cam = wx.camera_basis((1200 - 90 * k - shift, 900 - shift, -700 - shift), (500 - shift, 450 - shift, 380 - shift),
                                      (0, 1, 0), w / h, 45.0, float(w))
                reqs.append(wx.camera_request(g, cam, w, h, out[2 * k], shadow_out=out[2 * k + 1],
                                              light=(900.0 - shift, 2000.0 - shift, 300.0 - shift)))
            wx.trace_batch(grids, reqs, wx.Tune(persistent=persistent, refill=16, chunk=128, waves_per_cu=16, xcd_split=1))
            got[persistent] = [x.cpu().numpy() for x in out]
        hits = 0
        for a, b in zip(got[0], got[1]):
            assert np.array_equal(a, b)
            hits += int((a.view(wx.HIT_DTYPE)["state"] == wx.HIT).sum())
        assert hits > 1000


def test_autotune_of_one_request_leaves_the_queue_alone(wx, cuda):
    """One request without shadow rays has no work queue: its chunk and XCD split stay the defaults."""
    print("autotune of one request", flush=True)
    p = wx.Vdb345()
    p.add_spheres(scenes.sphere_set(2, count=300))
    p.compute_sdf()
    g = wx.Grid(p)
    rays = cuda.from_numpy(scenes.incoherent_rays(1 << 18)).cuda().repeat(16, 1)  # the persistent shape wins
    out = cuda.empty((len(rays), 32), dtype=cuda.uint8, device="cuda")
    old = wx.tune_get()
    try:
        for _ in range(4):
            t, _ = wx.autotune([g], [wx.rays_request(0, rays, out)])
            print(t.as_dict(), flush=True)
            assert (t.chunk, t.xcd_split) == (256, 1)
    finally:
        wx.tune_set(old)


@pytest.mark.parametrize("freq", [0.11, 2e5, 3e5, 1e6, 3e8, 1e38])
def test_noise_threshold_of_any_frequency(wx, cuda, freq):
    """The device's threshold is the host's also where a lattice coordinate leaves int32, which
    the two convert differently (the frequencies lie on both sides of 2^30 / 4 / 1000)."""
    print(f"noise threshold at frequency {freq}", flush=True)
    for lo, hi in (((0, 0, 0), (1000, 40, 30)), ((-1000, 5, -7), (-900, 60, 20))):
        th = wx.Vdb345().add_noise(9, lo, hi, freq, 0.3, threads=2)
        td = wx.Vdb345().add_noise(9, lo, hi, freq, 0.3, device=True)
        assert np.float32(th).view(np.uint32) == np.float32(td).view(np.uint32)


def test_root_keys_of_any_size(wx, cuda):
    """A descriptor's only node-5 may have any int32 key; one that no voxel has (2^20 past the
    scene's, which is the same coordinate mod 2^32) leaves every lookup a root miss."""
    print("root keys", flush=True)
    p = wx.Vdb345()
    p.add_spheres(np.array([[400.0, 300.0, 450.0, 120.0]]))
    p.compute_sdf()
    lay = p.layout_arrays()
    cam = wx.camera_basis((1200, 900, -700), (400, 300, 450), (0, 1, 0), 1.5, 45.0, 96.0)

    def records(key, persistent):
        root = lay["root"].copy().reshape(-1, 4)
        root[0, :3] = key
        g = grid_of(wx, root, lay["n5"], lay["n4"], lay["leaves"])
        out = [cuda.empty((96 * 64, 32), dtype=cuda.uint8, device="cuda") for _ in range(2)]
        tune = wx.Tune(persistent=persistent, refill=16, chunk=128, waves_per_cu=16, xcd_split=1)
        wx.trace_batch([g], [wx.camera_request(0, cam, 96, 64, out[0])], tune)
        wx.trace_batch([g], [wx.camera_request(0, cam, 96, 64, x) for x in out], tune)
        return wx.hits_to_numpy(out[1])

    assert (records((0, 0, 0), 0)["state"] == wx.HIT).any()
    away = records((3, 0, 0), 0)  # inside what a key can be, outside the rays' box
    assert (away["state"] != wx.HIT).all() and (away["lookups"] == 0).all()
    for key in ((1 << 20, 0, 0), (0, -(1 << 20), 0), (0, 0, -(1 << 31)), ((1 << 20) + 1, 1 << 20, 0)):
        for persistent in (0, 1):
            assert_hits_equal(records(key, persistent), away, f"key {key}")


@pytest.mark.parametrize("entries", [2, 16, 17, 40])
def test_first_of_equal_root_keys(wx, cuda, entries):
    """A descriptor's root table may name a key twice: the first entry is the node, in tables
    scanned from LDS (up to 16 entries) and from memory, in every shape."""
    print(f"{entries} root entries", flush=True)
    p = wx.Vdb345()
    p.add_spheres(np.array([[400.0, 300.0, 450.0, 120.0]]))
    p.compute_sdf()
    lay = p.layout_arrays()
    n5 = lay["n5"].reshape(1, -1)
    solid = np.zeros_like(n5)  # every slot an active tile: a hit wherever it is looked up
    nodes = np.concatenate([n5] + [solid] * (entries - 1))
    cam = wx.camera_basis((1200, 900, -700), (400, 300, 450), (0, 1, 0), 1.5, 45.0, 96.0)

    def records(where, persistent):
        root = np.zeros((entries, 4), np.int32)
        root[:, 0] = 5 + np.arange(entries)  # keys no ray meets
        root[:, 3] = np.arange(entries)
        root[where, :3] = lay["root"].reshape(-1, 4)[0, :3]
        # the sphere's node first among the equal keys
        root[where[0], 3], root[0, 3] = 0, where[0]
        g = grid_of(wx, root, nodes, lay["n4"], lay["leaves"])
        out = [cuda.empty((96 * 64, 32), dtype=cuda.uint8, device="cuda") for _ in range(3)]
        tune = wx.Tune(persistent=persistent, refill=16, chunk=128, waves_per_cu=16, xcd_split=1)
        wx.trace_batch([g], [wx.camera_request(0, cam, 96, 64, out[0])], tune)
        wx.trace_batch([g], [wx.camera_request(0, cam, 96, 64, out[1])] * 2, tune)
        wx.trace_batch([g, g], [wx.camera_request(k, cam, 96, 64, out[2]) for k in (1, 0)], tune)
        a = [wx.hits_to_numpy(x) for x in out]
        assert_hits_equal(a[1], a[0], "batch")
        assert_hits_equal(a[2], a[0], "batch of several grids")
        return a[0]

    want = wx.hits_to_numpy(wx.Grid(p).trace_camera(cam, 96, 64, 0.5, clip=True))
    assert (want["state"] == wx.HIT).any()
    for where in ([0], [entries - 1], [0, entries - 1], [0, 1], [entries // 2, entries - 1]):
        for persistent in (0, 1):
            assert_hits_equal(records(sorted(set(where)), persistent), want, f"{where} {persistent}")
