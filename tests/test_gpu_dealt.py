"""Frames and cameras whose rays are dealt to more and narrower packets.

How many waves share a task, and how large a camera's tiles are, follows from
the launch's size; every division has to give each sample to exactly one
wave, so samples, colours and pixels equal the oracle's bit for bit.  Frames
around the counts where the number of waves changes (up to 12,288 packets in a
small scene); cameras of one pixel, around the pixel counts where the tile
grows (16,384 times the tile's pixels) and of sizes that no tile divides.
"""
import numpy as np
import pytest

import oracle
from compound_ray_amd import eyerenderer as er
from compound_ray_amd import scenes
from test_gpu_cameras import pinhole_scale
from test_gpu_wide import check, eye_of, random_axes, soup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 37, 192, 193, 768, 1535, 1537])
@pytest.mark.parametrize("spp", [2, 3, 7, 31, 33, 64, 65, 130, 260])
def test_frames(lib, tmp_path, n, spp):
    pos, col = soup(300, 3)
    axes = random_axes(n, n)
    check(lib, tmp_path, pos, col, eye_of(axes, -1.5 * axes, 0.4), spp, modes=(2,))


@pytest.mark.parametrize("size", [(1, 1), (2, 1), (1, 3), (127, 129), (128, 128), (128, 129), (181, 181), (257, 256),
                                  (363, 363), (513, 511), (725, 723), (1025, 1023)])
@pytest.mark.parametrize("kind", [0, 2])
def test_cameras(lib, tmp_path, size, kind):
    pos, col = soup(300, 4)
    idx = np.arange(len(pos), dtype=np.uint32).reshape(-1, 3)
    name = ("perspective", "orthographic", "panoramic")[kind]
    cam = scenes.Camera("c", name, yfov=0.9, translation=(0.1, 0.2, -0.1), yaw=0.4)
    sc = scenes.Scene([scenes.Mesh("m", pos, idx, col)], eyes=[], cameras=[cam])
    lib.loadGlTFscene(str(scenes.write_gltf(tmp_path, "s", sc)).encode())
    assert er.last_error(lib) == ""
    lib.gotoCamera(0)
    w, h = size
    er.setRenderSize(lib, w, h)
    try:
        lib.setCameraPose(0.1, 0.2, -0.1, 0.1, 0.5, 0.0)
        scale = pinhole_scale(cam.yfov) if kind == 0 else np.zeros(3, np.float32)
        rays = oracle.camera_rays(kind, er.pose_np(lib), scale, w, h)
        assert lib.renderFrame() >= 0, er.last_error(lib)
        frame = np.array(lib.getFramePointer(), copy=True).reshape(h * w, 4)
        assert np.array_equal(frame, oracle.make_color(oracle.OracleScene.from_scene(sc).radiance(rays)))
    finally:
        er.setRenderSize(lib, 400, 400)
