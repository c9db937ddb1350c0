"""The host rules of woxel_amd/csrc/launch_shape.hpp: every ray of a list is traced exactly
once, whatever the list's length and the GPU's compute units (a partition has fewer)."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CUS = [16, 32, 64, 128, 256, 304]

PROGRAM = """
#include <cstdio>
#include "launch_shape.hpp"
int main() {
    unsigned long long rays;
    unsigned cus, fast;
    while (std::scanf("%llu %u %u", &rays, &cus, &fast) == 3) {
        const wxk::ListShape s = wxk::list_shape(rays, cus, fast != 0u);
        std::printf("%u %u\\n", s.lg, s.split ? 1u : 0u);
    }
}
"""


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    d = tmp_path_factory.mktemp("launch_shape")
    (d / "p.cpp").write_text(PROGRAM)
    csrc = os.path.join(HERE, "..", "woxel_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", csrc, str(d / "p.cpp"), "-o", str(d / "p")], check=True)

    def ask(pairs, fast=1):
        r = subprocess.run([str(d / "p")], input="".join(f"{n} {c} {fast}\n" for n, c in pairs),
                           capture_output=True, text=True, check=True)
        return [tuple(int(x) for x in line.split()) for line in r.stdout.splitlines()]

    return ask


def lengths(cus):
    """Lengths around every threshold: powers of two of the ray count per compute unit."""
    near = [c << k for c in (cus, 256) for k in range(1, 14)]
    return sorted({max(1, n + d) for n in near for d in (-65, -64, -63, -1, 0, 1, 37, 63, 64)})


@pytest.mark.parametrize("cus", CUS)
def test_split_lists_take_whole_sets(shape, cus):
    ns = lengths(cus)
    got = shape([(n, cus) for n in ns])
    assert any(s for _, s in got) and not all(s for _, s in got)
    for n, (lg, split) in zip(ns, got):
        assert not split or lg == 6, (n, cus, lg)


@pytest.mark.parametrize("cus", CUS)
def test_grids_without_the_fast_step_keep_their_lists(shape, cus):
    ns = lengths(cus)
    assert set(shape([(n, cus) for n in ns], fast=0)) == {(6, 0)}


@pytest.mark.parametrize("cus", CUS)
def test_small_waves_only_where_they_fit(shape, cus):
    """A wave takes fewer than 64 rays only while four waves per SIMD hold them all."""
    ns = lengths(cus)
    for n, (lg, _) in zip(ns, shape([(n, cus) for n in ns])):
        assert lg == 6 or n >> lg <= 16 * cus, (n, cus, lg)


@pytest.mark.parametrize("cus", CUS)
def test_every_ray_is_traced_once(shape, cus):
    """The two kernels' rules on a list of mixed directions: k_simple_rays takes 2^lg rays a wave
    and, in a split list, votes over the 64 from its first; k_persist1 votes over sets of 64."""
    rng = np.random.default_rng(cus)
    edge = [n for n in lengths(cus) if 4000 < n <= 600000][::3]
    for n, (lg, split) in zip(edge, shape([(n, cus) for n in edge])):
        near = rng.random(n + 64) < 0.5  # whether a ray goes the way of the first of its set
        near[n:] = False

        def together(first):
            w = near[first[:, None] + np.arange(64)]
            inside = np.minimum(n - first, 64)
            return 2 * w.sum(1) >= inside

        times = np.zeros(n, np.int64)
        first = np.arange(0, n, 1 << lg)
        on = together(first) if split else np.ones(len(first), bool)
        rays = (first[on, None] + np.arange(1 << lg)).ravel()
        np.add.at(times, rays[rays < n], 1)
        if split:
            sets = np.arange(0, n, 64)
            rays = (sets[~together(sets), None] + np.arange(64)).ravel()
            np.add.at(times, rays[rays < n], 1)
        assert (times == 1).all(), (n, cus, int((times == 0).sum()))
