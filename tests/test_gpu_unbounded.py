"""Scenes with vertices that are infinite, not numbers or too large to add.

The boxes above such a triangle have centres and depths that are not numbers or
not inside them, and a packet of the 64-wide walk orders its children by depth.
These scenes have no 64-wide tree: rays and eyes of the default traversal find
what the 4-wide tree's walk finds.  A scene just within the bound has one.
"""
import numpy as np
import pytest

import oracle
from compound_ray_amd import eyerenderer as er
from compound_ray_amd import scenes
from test_gpu_wide import eye_of, random_axes, soup

pytestmark = pytest.mark.gpu

MARK = np.float32(1234.5)   # in the file's vertices, replaced in its buffer


def load(lib, tmp_path, pos, col, bad, omm):
    """The scene with the vertices of `bad` (row -> three floats) in its buffer."""
    marked = pos.copy()
    for row in bad:
        marked[row] = MARK
    idx = np.arange(len(pos), dtype=np.uint32).reshape(-1, 3)
    sc = scenes.Scene([scenes.Mesh("m", marked, idx, col)], eyes=[scenes.Eye("eye", omm)])
    path = scenes.write_gltf(tmp_path, "s", sc)
    raw = np.fromfile(path.with_suffix(".bin"), np.float32)
    real = pos.copy()
    for row, v in bad.items():
        real[row] = v
    assert np.array_equal(raw[:pos.size].reshape(-1, 3), marked)
    raw[:pos.size] = real.ravel()
    raw.tofile(path.with_suffix(".bin"))
    lib.loadGlTFscene(str(path).encode())
    assert er.last_error(lib) == ""
    er.gotoFirstCompoundEye(lib)
    n = len(idx)
    return oracle.OracleScene(real, col[:, :3].copy(), np.zeros(n, np.uint32), sc.sky_mode())


def bad_vertices(kind, n, count, seed):
    rng = np.random.default_rng(seed)
    rows = rng.choice(3 * n, count, replace=False)
    big = {"infinite": np.inf, "not numbers": np.nan, "huge": 3e38, "far": 2e18, "within": 1e18}[kind]
    out = {}
    for k, row in enumerate(rows):
        v = rng.uniform(-1, 1, 3)
        which = rng.random(3) < 0.6
        which[rng.integers(3)] = True
        v[which] = big * np.where(rng.random(3) < 0.5, -1.0, 1.0)[which]
        out[int(row)] = v.astype(np.float32)
        if k % 3 == 0:   # all corners of the triangle
            for r in range(int(row) // 3 * 3, int(row) // 3 * 3 + 3):
                out[r] = v.astype(np.float32)
    return out


@pytest.mark.parametrize("kind", ["infinite", "not numbers", "huge", "far", "within"])
@pytest.mark.parametrize("n,count", [(300, 1), (300, 40), (20000, 3), (20000, 400)])
def test_rays_and_eyes(lib, tmp_path, kind, n, count):
    pos, col = soup(n, n, size=0.08)
    axes = random_axes(60, 1)
    omm = eye_of(axes, 0.3 * axes, 0.2)
    O = load(lib, tmp_path, pos, col, bad_vertices(kind, n, count, count), omm)
    rng = np.random.default_rng(2)
    rays = np.zeros((20000, 8), np.float32)
    rays[:, 0:3] = np.repeat(rng.uniform(-1.5, 1.5, (2500, 3)), 8, 0)
    rays[:, 4:7] = np.repeat(rng.normal(size=(2500, 3)), 8, 0) + rng.normal(size=(20000, 3)) * 0.02
    rays[:, 7] = 1e16
    want, wt = O.trace(rays)
    assert (want >= 0).any() and (want < 0).any()
    for m in (600, 20000):   # a ray per wave, and eight
        ids, tbb = er.trace_np(lib, rays[:m])
        assert np.array_equal(ids, want[:m])
        hit = ids >= 0
        assert np.array_equal(tbb[hit].view(np.uint32), wt[:m][hit].view(np.uint32))
    er.set_ommatidia_np(lib, omm)
    lib.setSampleRecording(True)
    try:
        for spp, split in ((9, True), (9, False), (65, True)):
            lib.setSplitLaunches(split)
            lib.setCurrentEyeSamplesPerOmmatidium(spp)
            lib.setCameraPose(0, 0, 0, 0, 0, 0)
            lib.setCurrentEyeFrameIndex(0)
            eye_rays = er.rays_np(lib)
            assert lib.renderFrame() >= 0, er.last_error(lib)
            ids, t = O.trace(eye_rays)
            got = er.samples_np(lib)[:, 3]
            assert np.array_equal(got, np.where(ids >= 0, t[:, 0], np.float32(-1.0)))
    finally:
        lib.setSplitLaunches(True)
        lib.setSampleRecording(False)
