"""The per-ommatidium constants of ray generation, prepared once per upload.

Samples equal the oracle's bit for bit, which derives everything per ray:
counts around the preparing kernel's block, axes along and near the axis that
has no perpendicular, axes that are not of unit length, closed cones, lenses
away from the rays' start, and a second upload of another size.
"""
import numpy as np
import pytest

import oracle
from compound_ray_amd import eyerenderer as er
from compound_ray_amd import scenes
from test_gpu_wide import eye_of, random_axes, soup

pytestmark = pytest.mark.gpu


def ommatidia(n, seed):
    rng = np.random.default_rng(seed)
    axes = random_axes(n, seed) * rng.uniform(0.2, 3.0, (n, 1)).astype(np.float32)
    special = [(0, 1, 0), (0, -2, 0), (0, 1, 1e-20), (1e-4, -1, 0), (1, 0, -1), (0, 0, 1), (-1, 0, 0)]
    for i, a in enumerate(special):
        axes[i % n::11 + i] = a
    acc = rng.choice([0.0, 0.01, 0.3, 2.0], n)
    return eye_of(axes, rng.normal(size=(n, 3)) * 0.5, acc, rng.choice([0.0, 0.25, -0.5], n))


@pytest.mark.parametrize("n", [1, 2, 63, 255, 256, 257, 1025])
def test_cones(lib, tmp_path, n):
    pos, col = soup(400, 5)
    idx = np.arange(len(pos), dtype=np.uint32).reshape(-1, 3)
    sc = scenes.Scene([scenes.Mesh("m", pos, idx, col)], eyes=[scenes.Eye("eye", ommatidia(3, 1))])
    lib.loadGlTFscene(str(scenes.write_gltf(tmp_path, "s", sc)).encode())
    assert er.last_error(lib) == ""
    er.gotoFirstCompoundEye(lib)
    lib.setCameraPose(0.1, -0.2, 0.3, 0.4, 0.5, 0.6)
    lib.setSampleRecording(True)
    try:
        for k, m in enumerate((n, n + 5, max(1, n // 2))):
            omm = ommatidia(m, 10 + k)
            er.set_ommatidia_np(lib, omm)
            lib.setCurrentEyeSamplesPerOmmatidium(7)
            lib.setCurrentEyeFrameIndex(0)
            want = oracle.OracleScene.from_scene(sc).render(omm, er.pose_np(lib), spp=7, want_samples=True)
            assert lib.renderFrame() >= 0, er.last_error(lib)
            assert np.array_equal(er.samples_np(lib).view(np.uint32), want["samples"].view(np.uint32)), m
    finally:
        lib.setSampleRecording(False)
