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
    assert (gpu["state"] == wx.HIT).sum() > 20
