"""The traversal loop's fast step against the oracle, bit for bit, at the edges of the
rule that chooses it: zero direction components, -0 and tiny starts, starts next to cell
borders, and bounds on both sides of 2^20."""
import numpy as np
import pytest

from test_gpu_trace import assert_hits_equal

pytestmark = pytest.mark.gpu


def edge_rays():
    """Waves of 64 rays, one kind each, then the same rays mixed."""
    rng = np.random.default_rng(11)

    def unit(n):
        d = rng.standard_normal((n, 3))
        return d / np.linalg.norm(d, axis=1, keepdims=True)

    groups = []
    # axis- and plane-aligned directions (+0 components) from starts on both sides of zero
    d = np.zeros((64, 3))
    d[np.arange(64), np.arange(64) % 3] = 1.0
    d[32:, 0] += 0.5
    groups.append(np.concatenate([rng.uniform(-120, 120, (64, 3)), d], 1))
    # the same with one start just below zero on an axis that does not move
    g = groups[0].copy()
    g[5, :3], g[5, 3:] = (-30.0, -0.001, 20.0), (1.0, 0.0, 0.0)
    groups.append(g)
    # -0 starts, tiny starts of both signs (a quotient that underflows, one that does not)
    g = np.concatenate([rng.uniform(-60, 60, (64, 3)), unit(64)], 1)
    g[np.arange(64), np.arange(64) % 3] = np.array([-0.0, 1e-40, -1e-40, -2.0 ** -70, 2.0 ** -70, -1e-45, 0.0])[
        np.arange(64) % 7]
    groups.append(g)
    g = g.copy()
    g[:, :3][g[:, :3] == 0] = 0.0  # no -0: the wave may take the fast step
    groups.append(g)
    # one float below, on and above a cell border
    o = (rng.integers(-24, 24, (64, 3)) * 8).astype(np.float32)
    o[:, 0] = np.nextafter(o[:, 0], np.float32(-1e9), dtype=np.float32)
    o[:, 1] = np.nextafter(o[:, 1], np.float32(1e9), dtype=np.float32)
    groups.append(np.concatenate([o, unit(64)], 1))
    # far starts: up to and past 2^20 and 2^21, toward the scene
    o = unit(64) * np.float64(2.0) ** rng.uniform(12, 22, (64, 1))
    d = rng.uniform(-60, 60, (64, 3)) - o
    groups.append(np.concatenate([o, d / np.linalg.norm(d, axis=1, keepdims=True)], 1))
    r = np.concatenate(groups).astype(np.float32)
    return np.concatenate([r, r[rng.permutation(len(r))]])


@pytest.mark.parametrize("bound", [4096.0, 2.0 ** 20, 2.0 ** 20 + 1.0])
@pytest.mark.parametrize("roots", ["one", "several"])
def test_fast_step_edges(wx, oracle_mod, cuda, bound, roots):
    sp = np.array([[40.0, 30.0, 45.0, 22.0], [90.0, 60.0, 20.0, 14.0]])
    if roots == "several":
        sp = np.concatenate([sp, -sp * [1, 1, 1, -1], [[-45.0, 40.0, 30.0, 19.0]]])
    print(f"fast step, bound {bound}, {roots} roots", flush=True)
    p = wx.Vdb345()
    p.add_spheres(sp)
    p.compute_sdf()
    o = oracle_mod.Vdb()
    for s in sp:
        o.add_sphere(s[:3], s[3])
    o.compute_sdf()
    g = wx.Grid(p, bound)
    rays = edge_rays()
    t = cuda.from_numpy(rays).cuda()
    for clip in (False, True):
        for simple in (False, True):
            gpu = wx.hits_to_numpy(g.trace_rays(t, clip=clip, simple=simple))
            ora, _ = o.trace_rays(rays, bound=bound, clip=clip)
            assert_hits_equal(gpu, ora, f"bound={bound} clip={clip} simple={simple}")
    assert (gpu["state"] == wx.HIT).any()


def test_layouts_without_consecutive_children(wx, oracle_mod, cuda):
    """Layouts whose children are not consecutive within a node (4-byte entries), or whose
    only node-5 does not start at node-4 0 (compact, with its base): the same records as
    the builder's layout, from every kernel that traces rays."""
    import ctypes as C

    sp = np.array([[400.0, 300.0, 450.0, 120.0], [700.0, 600.0, 260.0, 90.0]])
    p = wx.Vdb345()
    p.add_spheres(sp)
    p.compute_sdf()
    lay = p.layout_arrays()
    n5, n4, n3 = lay["n"]
    rng = np.random.default_rng(5)
    tgt = sp[rng.integers(0, 2, 5000), :3] + rng.uniform(-80, 80, (5000, 3))
    eye = rng.uniform(-1500, 2500, (5000, 3))
    d = tgt - eye
    rays = np.concatenate([eye, d / np.linalg.norm(d, axis=1, keepdims=True)], 1).astype(np.float32)
    rays[70, 4] = -0.0  # one wave in the general step
    t = cuda.from_numpy(rays).cuda()
    want = wx.hits_to_numpy(wx.Grid(p).trace_rays(t, clip=True, simple=True))
    o = oracle_mod.Vdb()
    for s in sp:
        o.add_sphere(s[:3], s[3])
    o.compute_sdf()
    assert_hits_equal(want, o.trace_rays(rays, clip=True)[0], "builder's layout")
    assert (want["state"] == wx.HIT).sum() > 1000

    def grid(rec5, rec4, leaves):
        arrays = [np.ascontiguousarray(a, np.uint32) for a in (rec5, rec4, leaves)]
        root = np.ascontiguousarray(lay["root"], np.int32)
        g = wx.GridDesc()
        g.n5, g.n4, g.n3, g.bound = n5, arrays[1].size // 1024, arrays[2].size // 64, 4096.0
        g.root = root.ctypes.data_as(C.POINTER(C.c_int32))
        g.n5_records, g.n4_records, g.leaves = [a.ctypes.data_as(C.POINTER(C.c_uint32)) for a in arrays]
        return wx.Grid.from_desc(g), (root, arrays)

    # every second node-4 record finds its leaves in a copy 5000 leaves further on
    far4 = lay["n4"].copy()
    far4[::2, 1] += n3 + 5000
    leaves = np.concatenate([lay["leaves"], np.zeros((5000, 64), np.uint32), lay["leaves"]])
    # the node-4 nodes after three unused ones
    late5 = lay["n5"].copy()
    late5[:, 1] += 3
    late4 = np.concatenate([np.zeros((3 * 256, 4), np.uint32), lay["n4"]])
    old = wx.tune_get()
    for name, args in (("far leaves", (lay["n5"], far4, leaves)), ("late nodes", (late5, late4, lay["leaves"]))):
        g, keep = grid(*args)
        for persistent in (0, 1):
            print(f"{name}, shape {persistent}", flush=True)
            tune = wx.tune_get()
            tune.persistent = persistent
            out = cuda.empty((len(rays), 32), dtype=cuda.uint8, device="cuda")
            out2 = cuda.empty_like(out)
            wx.trace_batch([g], [wx.rays_request(0, t, out)], tune)
            assert_hits_equal(wx.hits_to_numpy(out), want, f"{name} {persistent}")
            wx.trace_batch([g], [wx.rays_request(0, t, out), wx.rays_request(0, t, out2)], tune)
            assert_hits_equal(wx.hits_to_numpy(out2), want, f"{name} batch {persistent}")
    assert wx.tune_get().as_dict() == old.as_dict()


@pytest.mark.parametrize("n", [(1 << 20) - 1, (1 << 20) + 37])
def test_long_ray_lists(wx, oracle_mod, cuda, n):
    """Lists on both sides of the length at which scattered sets of 64 rays go to the
    refilled waves: sets of one direction and scattered ones in turn, rays of the general
    step and rays that meet the step cap among both."""
    print(f"{n} rays", flush=True)
    rng = np.random.default_rng(n)
    org = np.array([(x, 0, 0) for x in range(0, 4096, 8)], np.int32)
    masks = np.full((org.shape[0], 8), np.uint64(0xFF))
    p = wx.Vdb345()
    p.add_leaf_masks(org >> 3, masks)
    p.add_spheres(np.array([[2000.0, 1500.0, 1800.0, 60.0], [700.0, 900.0, 2500.0, 45.0]]))
    p.compute_sdf()
    o = oracle_mod.Vdb()
    o.add_leaf_masks(org, masks)
    for s in ([2000.0, 1500.0, 1800.0, 60.0], [700.0, 900.0, 2500.0, 45.0]):
        o.add_sphere(np.array(s[:3]), s[3])
    o.compute_sdf()
    g = wx.Grid(p)
    m = (n + 63) // 64 * 64
    eye = rng.uniform(-3000, 6000, (m, 3))
    d = rng.uniform(-60, 60, (m, 3)) + np.where(rng.random((m, 1)) < 0.5, [[2000, 1500, 1800]], [[700, 900, 2500]]) - eye
    rays = np.concatenate([eye, d], 1).reshape(-1, 64, 6)
    rays[::3, :, :3] = rays[::3, :1, :3]  # one eye, neighbouring directions
    rays[::3, :, 3:] = rays[::3, :1, 3:] + rng.uniform(-20, 20, rays[::3, :, 3:].shape)
    rays = rays.reshape(m, 6)[:n].astype(np.float32)
    rays[:, 3:] /= np.linalg.norm(rays[:, 3:], axis=1, keepdims=True)
    k = rng.integers(0, n, 3000)
    rays[k, 3 + rng.integers(0, 3, 3000)] = -0.0
    k = rng.integers(0, n, 3000)
    rays[k] = np.stack([np.full(3000, 0.5), 1.5 + k % 7, np.full(3000, 4.5), np.ones(3000), np.zeros(3000),
                        np.zeros(3000)], 1)  # beside the wall: the step cap
    t = cuda.from_numpy(rays).cuda()
    ora, _ = o.trace_rays(rays, clip=True)
    nan = np.isnan(ora["t"])
    for simple in (False, True):
        gpu = wx.hits_to_numpy(g.trace_rays(t, clip=True, simple=simple))
        assert np.array_equal(np.isnan(gpu["t"]), nan)
        assert_hits_equal(gpu[~nan], ora[~nan], f"{n} rays, simple={simple}")
    assert {wx.HIT, wx.OOB, wx.MAXSTEPS} <= set(np.unique(gpu["state"]).tolist())
