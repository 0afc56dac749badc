"""Hits at the corners of boxes, from origins far from them.

Flat triangles in axis planes fill their boxes' corners; rays aimed at their
vertices meet a box by less than the rounding of its test, which the boxes'
padding has to cover wherever the origin is.  All hits equal brute force.
"""
import numpy as np
import pytest

import oracle
from compound_ray_amd import eyerenderer as er
from compound_ray_amd import scenes
from test_gpu_wide import eye_of, random_axes

pytestmark = pytest.mark.gpu

FLAT = 24


def flat_triangles(seed):
    """In the middle of a scene of radius 2, each four times: a leaf of its own."""
    rng = np.random.default_rng(seed)
    tris = []
    for k in range(FLAT):
        v = rng.uniform(-0.25, 0.25, 3)
        s = rng.uniform(0.02, 0.06) * rng.choice([-1, 1], 2)
        t = np.repeat(v[None], 3, 0)
        t[1, (k + 1) % 3] += s[0]
        t[2, (k + 2) % 3] += s[1]
        tris += [t] * 4
    for c in (-1.0, 1.0):
        tris += [c + np.float64([[0, 0, 0], [0.01, 0, 0], [0, 0.01, 0]])] * 4
    return np.concatenate(tris).astype(np.float32)


# the last: one ray of its 4 M was lost while boxes were padded for 4 radii
@pytest.mark.parametrize("radii,seed,n", [(0.9, 1, 500000), (1.45, 2, 500000), (1.55, 3, 500000), (3.0, 4, 500000),
                                          (40.0, 5, 500000), (3.9, 2, 4000000)])
def test_rays_at_vertices(lib, tmp_path, radii, seed, n):
    pos = flat_triangles(seed)
    sc = scenes.Scene([scenes.Mesh("m", pos, np.arange(len(pos), dtype=np.uint32).reshape(-1, 3),
                                   np.ones((len(pos), 4), np.float32))],
                      eyes=[scenes.Eye("eye", eye_of(random_axes(4, 1), 0.0, 0.1))])
    lib.loadGlTFscene(str(scenes.write_gltf(tmp_path, "s", sc)).encode())
    assert er.last_error(lib) == ""
    O = oracle.OracleScene.from_scene(sc)
    rng = np.random.default_rng(seed)
    corner = pos[:12 * FLAT].reshape(-1, 3, 3)[::4].reshape(-1, 3)
    to = corner[rng.integers(0, len(corner), n)].astype(np.float64)
    o = rng.uniform(-1, 1, (n, 3))
    o /= np.abs(o).max(1, keepdims=True)
    o *= 2.0 * radii
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = o
    d = to - rays[:, 0:3]
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays[:, 7] = 1e16
    ids, tbb = er.trace_np(lib, rays)
    want, wt = O.trace(rays, bvh=False)
    assert (want >= 0).mean() > 0.3
    assert np.array_equal(ids, want)
    hit = want >= 0
    assert np.array_equal(tbb[hit].view(np.uint32), wt[hit].view(np.uint32))
