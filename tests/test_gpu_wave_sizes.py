"""Launches on both sides of the sizes at which a wave takes fewer rays: ray lists,
frames, batches and shaded frames against the oracle, bit for bit."""
import numpy as np
import pytest

from test_gpu_fast_step import edge_rays
from test_gpu_trace import assert_hits_equal

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(wx, oracle_mod, cuda):
    sp = np.array([[40.0, 30.0, 45.0, 22.0], [90.0, 60.0, 20.0, 14.0], [-45.0, 40.0, 30.0, 19.0]])
    p = wx.Vdb345()
    p.add_spheres(sp)
    p.compute_sdf()
    o = oracle_mod.Vdb()
    for s in sp:
        o.add_sphere(s[:3], s[3])
    o.compute_sdf()
    return wx.Grid(p), o


@pytest.mark.parametrize("n", [1, 4096, 4097, 8193, 16385, 65537, 131071, 131072, 131073 + 131072])
def test_ray_lists(wx, cuda, scene, n):
    print(f"{n} rays", flush=True)
    g, o = scene
    rays = edge_rays()
    want, _ = o.trace_rays(rays, bound=4096.0, clip=True)
    k = np.arange(n) % len(rays)
    t = cuda.from_numpy(rays[k]).cuda()
    assert_hits_equal(wx.hits_to_numpy(g.trace_rays(t, clip=True)), want[k], f"{n} rays")
    out = cuda.empty((n, 32), dtype=cuda.uint8, device="cuda")
    wx.trace_batch([g, g], [wx.rays_request(1, t, out, clip=True)])
    assert_hits_equal(wx.hits_to_numpy(out), want[k], f"{n} rays in a batch")


@pytest.mark.parametrize("w,h", [(64, 64), (241, 17), (91, 90), (129, 127), (181, 183), (257, 255), (361, 365), (513, 515)])
def test_frames(wx, cuda, scene, w, h):
    print(f"{w}x{h} pixels", flush=True)
    g, o = scene
    cam = wx.camera_basis((300, 250, -260), (40, 35, 30), (0, 1, 0), w / h, 40.0, float(w))
    want, _ = o.trace_camera(cam.as_array(), w, h, 0.5)
    assert_hits_equal(wx.hits_to_numpy(g.trace_camera(cam, w, h, 0.5)), want, f"{w}x{h}")
    out = [cuda.empty((w * h, 32), dtype=cuda.uint8, device="cuda") for _ in range(2)]
    wx.trace_batch([g, g], [wx.camera_request(k, cam, w, h, out[k], clip=False) for k in range(2)])
    for t in out:
        assert_hits_equal(wx.hits_to_numpy(t), want, f"{w}x{h} in a batch")
    lay = o.layout()
    for mode in (3, 4):
        shade = wx.shade(mode, sun_dir=(0.3, -0.8, 0.52), intensity=0.9)
        f = g.render_camera(cam, w, h, shade, 0.5, f32=True).cpu().numpy()
        rf, _ = lay.render_camera(cam.as_array(), w, h, shade, 0.5)
        assert np.array_equal(f.view(np.uint32), rf.view(np.uint32)), mode


@pytest.mark.parametrize("n_grids,n_reqs", [(1, 2), (12, 24), (12, 25), (13, 24), (13, 25)])
def test_batch_tables(wx, cuda, scene, n_grids, n_reqs):
    """Both sides of the counts up to which a batch's tables are kernel arguments."""
    print(f"{n_reqs} requests on {n_grids} grids", flush=True)
    _, o = scene
    g = [scene[0]] * n_grids
    reqs, outs, want = [], [], []
    for k in range(n_reqs):
        w, h = 9 + 3 * k, 31 - k
        cam = wx.camera_basis((300 - 9 * k, 250, -260 + 5 * k), (40, 35, 30), (0, 1, 0), w / h, 40.0, float(w))
        outs.append(cuda.empty((w * h, 32), dtype=cuda.uint8, device="cuda"))
        reqs.append(wx.camera_request((7 * k + n_grids - 1) % n_grids, cam, w, h, outs[-1], clip=True))
        want.append(o.trace_camera(cam.as_array(), w, h, 0.5, clip=True)[0])
    wx.trace_batch(g, reqs)
    for k, (t, ora) in enumerate(zip(outs, want)):
        assert_hits_equal(wx.hits_to_numpy(t), ora, f"request {k}")
