"""Rays along the axes through scenes of large coordinates.

The reciprocal of a direction's component near 0 times a coordinate beyond
3.4e8 is not finite: rays that run inside a box's slab have to enter it all the
same, whatever the scene's unit is.
"""
import numpy as np
import pytest

import oracle
from compound_ray_amd import eyerenderer as er
from compound_ray_amd import scenes
from test_gpu_wide import eye_of

pytestmark = pytest.mark.gpu


def blocks(unit, away, count):
    """Squares of several heights around (away, 0, 0), in `unit`s; a count of 1: one
    triangle whose middle is the origin."""
    rng = np.random.default_rng(5)
    if count == 1:
        return (np.float64([[-16, 0, -16], [16, 0, -16], [-1, 0, 16]]) * unit).astype(np.float32)
    quad = np.float64([[0, 0, 0], [1, 0, 0], [1, 0, 1], [0, 0, 0], [1, 0, 1], [0, 0, 1]])
    at = rng.uniform(-8, 8, (700, 1, 3)) * [1, 0.2, 1]
    return ((at + quad * rng.uniform(0.3, 2.0, (700, 1, 1)) + [away, 0, 0]) * unit).reshape(-1, 3).astype(np.float32)


@pytest.mark.parametrize("unit", [1.0, 1e7, 1e9, 1e12, 1e16])
@pytest.mark.parametrize("away,count", [(0.0, 700), (40.0, 700), (0.0, 1)])
def test_axis_rays(lib, tmp_path, unit, away, count):
    pos = blocks(unit, away, count)
    col = np.concatenate([np.random.default_rng(1).uniform(0, 1, (len(pos), 3)), np.ones((len(pos), 1))],
                         1).astype(np.float32)
    n = 400
    rng = np.random.default_rng(6)
    rays = np.zeros((4 * n, 8), np.float32)
    rays[:, 0:3] = (rng.uniform(-8, 8, (4 * n, 3)) * [1, 0.1, 1] + [away, 3.0, 0]) * unit
    rays[:, 5] = -1.0                                   # straight down
    rays[n:2 * n, 4] = rng.choice([1e-38, -1e-30, 1e-29, -1e-12], n)
    rays[2 * n:3 * n, 6] = rng.choice([-0.0, 1e-25, -1e-31], n)
    rays[3 * n:, 4:7] = rng.normal(size=(n, 3)) * [0.3, 0.1, 0.3] - [0, 1, 0]
    rays[:, 7] = 1e30
    omm = eye_of(np.tile(np.float32([[0, -1, 0]]), (50, 1)), rays[:50, 0:3], 0.0)
    sc = scenes.Scene([scenes.Mesh("m", pos, np.arange(len(pos), dtype=np.uint32).reshape(-1, 3), col)],
                      eyes=[scenes.Eye("eye", omm)])
    sc.cameras = [scenes.Camera("flat", "orthographic", xmag=float(6 * unit), ymag=float(6 * unit))]
    lib.loadGlTFscene(str(scenes.write_gltf(tmp_path, "s", sc)).encode())
    assert er.last_error(lib) == ""
    O = oracle.OracleScene.from_scene(sc)
    ids, tbb = er.trace_np(lib, rays)
    want, wt = O.trace(rays, bvh=False)
    hit = want >= 0
    # beyond that the triangle test's products of three lengths overflow: no walk hits anything
    assert hit.reshape(4, n).any(axis=1).all() == (unit * (2 if count > 1 else 32) < 1e13)
    assert np.array_equal(ids, want)
    assert np.array_equal(tbb[hit].view(np.uint32), wt[hit].view(np.uint32))
    # an eye whose ommatidia look straight down
    er.gotoFirstCompoundEye(lib)
    er.set_ommatidia_np(lib, omm)
    lib.setCurrentEyeSamplesPerOmmatidium(3)
    lib.setCameraPose(0, 0, 0, 0, 0, 0)
    assert lib.renderFrame() >= 0, er.last_error(lib)
    ref = O.render(omm, er.pose_np(lib), spp=3)["colour_gpu_order"][0]
    assert np.array_equal(er.colours_np(lib), ref)
    # an orthographic camera above, looking down
    lib.gotoCameraByName(b"flat")
    lib.setCameraPose(float(away * unit), float(3 * unit), 0.0, float(-np.pi / 2), 0.0, 0.0)
    er.setRenderSize(lib, 60, 40)
    try:
        cam = np.zeros((2400, 8), np.float32)
        assert lib.getCurrentCameraRays(cam.ctypes.data, 2400) == 2400
        assert lib.renderFrame() >= 0, er.last_error(lib)
        frame = np.array(lib.getFramePointer(), copy=True).reshape(-1, 4)
        assert np.array_equal(frame, oracle.make_color(O.radiance(cam)))
    finally:
        er.setRenderSize(lib, 400, 400)
