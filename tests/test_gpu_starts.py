"""Rays that start behind their origin (a negative tmin or focal offset).

A packet leaves out what lies deeper than every ray's hit; depths count from
where the rays start, hit distances from their origins.  Scenes in which every
ray of a packet hits, at many depths before and behind the origin, single rays
and fans of them, frames and batches: all equal the oracle's bit for bit.
"""
import numpy as np
import pytest

import oracle
from compound_ray_amd import eyerenderer as er
from compound_ray_amd import scenes
from test_gpu_wide import check, eye_of, random_axes, soup

pytestmark = pytest.mark.gpu


def closed(n, seed, size=0.08):
    """n triangles around the origin within a box whose walls every ray meets."""
    pos, col = soup(n, seed, size=size, spread=2.5)
    g = np.linspace(-6, 6, 25, dtype=np.float32)
    walls = []
    for a in range(3):
        for s in (-6.0, 6.0):
            for i in range(24):
                for j in range(24):
                    q = np.empty((4, 3), np.float32)
                    q[:, a] = s
                    q[:, (a + 1) % 3] = g[[i, i + 1, i + 1, i]]
                    q[:, (a + 2) % 3] = g[[j, j, j + 1, j + 1]]
                    walls.append(q[[0, 1, 2, 0, 2, 3]])
    walls = np.concatenate(walls)
    shade = np.concatenate([np.random.default_rng(seed).uniform(0, 1, (len(walls), 3)), np.ones((len(walls), 1))], 1)
    return np.concatenate([pos, walls]), np.concatenate([col, shade]).astype(np.float32)


def load(lib, tmp_path, pos, col):
    idx = np.arange(len(pos), dtype=np.uint32).reshape(-1, 3)
    sc = scenes.Scene([scenes.Mesh("m", pos, idx, col)], eyes=[scenes.Eye("eye", eye_of(random_axes(4, 1), 0.0, 0.1))])
    lib.loadGlTFscene(str(scenes.write_gltf(tmp_path, "s", sc)).encode())
    assert er.last_error(lib) == ""
    return oracle.OracleScene.from_scene(sc)


# 600 rays walk one by one, 16,800 in packets of eight (test_gpu_pieces.py)
@pytest.mark.parametrize("n", [600, 16800])
@pytest.mark.parametrize("tmin", [-0.5, -1.5, -4.0, -1e6, -1e30, -np.inf])
def test_free_rays(lib, tmp_path, n, tmin):
    O = load(lib, tmp_path, *closed(20000, 3))
    rng = np.random.default_rng(n)
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = np.repeat(rng.uniform(-2, 2, (n // 8, 3)), 8, 0)
    rays[:, 4:7] = np.repeat(rng.normal(size=(n // 8, 3)), 8, 0) + rng.normal(size=(n, 3)) * 0.01
    rays[:, 4:7] *= rng.uniform(0.5, 2.0, (n, 1))
    rays[:, 3] = tmin
    rays[:, 7] = 1e16
    if n == 600:
        rays[::7, 3] = 0.25   # beside rays that start beyond theirs
    ids, tbb = er.trace_np(lib, rays)
    # without a tree: what any walk of one has to find
    want, wt = O.trace(rays, bvh=False)
    assert (want >= 0).all()
    assert np.array_equal(ids, want)
    assert np.array_equal(tbb.view(np.uint32), wt.view(np.uint32))


@pytest.mark.parametrize("spp", [7, 64, 130])
@pytest.mark.parametrize("focal", [-0.5, -1.5, -5.0])
@pytest.mark.parametrize("split", [True, False])
def test_eyes(lib, tmp_path, spp, focal, split):
    pos, col = closed(20000, 4, size=0.15)
    axes = random_axes(60, 5)
    want = check(lib, tmp_path, pos, col, eye_of(axes, 0.3 * axes, 0.1, focal), spp, split=split, modes=(2, 0))
    assert (want["samples"].reshape(-1, 4)[:, 3] != -1.0).all()
