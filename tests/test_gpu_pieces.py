"""Results that cross to the host in pieces or through pinned memory.

Hits of free rays around the counts where the packets (16,384) and the pieces
(131,072) change; colours and pixels of frames after each other, of eyes that
grow, shrink and change place, whose host copies the frame kernels write; and
batches around the size (65,536 units) up to which pinned memory is used.
All equal the oracle's bit for bit.
"""
import numpy as np
import pytest

import oracle
from compound_ray_amd import eyerenderer as er
from compound_ray_amd import scenes
from test_gpu_wide import eye_of, random_axes, soup

pytestmark = pytest.mark.gpu


def load(lib, tmp_path, n_eyes=1):
    pos, col = soup(500, 8)
    idx = np.arange(len(pos), dtype=np.uint32).reshape(-1, 3)
    eyes = [scenes.Eye(f"eye{k}", eye_of(random_axes(4, k), 0.0, 0.1)) for k in range(n_eyes)]
    sc = scenes.Scene([scenes.Mesh("m", pos, idx, col)], eyes=eyes)
    lib.loadGlTFscene(str(scenes.write_gltf(tmp_path, "s", sc)).encode())
    assert er.last_error(lib) == ""
    er.gotoFirstCompoundEye(lib)
    return oracle.OracleScene.from_scene(sc)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 16383, 16384, 16385, 131071, 131072, 131073, 262145])
@pytest.mark.parametrize("order", ["none", "fans"])
def test_free_rays(lib, tmp_path, n, order):
    O = load(lib, tmp_path)
    rng = np.random.default_rng(n)
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = rng.uniform(-2, 2, (n, 3))
    rays[:, 4:7] = rng.normal(size=(n, 3))
    if order == "fans":   # runs of 100 rays from one place in one direction
        rays = rays[(np.arange(n) // 100) * 100 % n]
        rays[:, 4:7] += rng.normal(size=(n, 3)) * 0.05
    rays[:, 4:7] *= rng.uniform(0.1, 4.0, (n, 1)).astype(np.float32)
    rays[:, 3] = rng.choice([0.0, 0.3], n)
    rays[:, 7] = rng.choice([1e16, 2.0], n)
    ids = np.empty(n, np.int32)
    tbb = np.empty((n, 3), np.float32)
    assert lib.traceRays(rays, n, ids, tbb) == 0, er.last_error(lib)
    want, wt = O.trace(rays)
    assert np.array_equal(ids, want)
    hit = want >= 0
    assert np.array_equal(tbb[hit].view(np.uint32), wt[hit].view(np.uint32))


def test_frames_of_changing_eyes(lib, tmp_path):
    O = load(lib, tmp_path, n_eyes=2)
    er.setRenderSize(lib, 50, 3)
    first = lib.getCurrentCameraIndex()
    try:
        for step, (eye, n, spp) in enumerate([(0, 40, 5), (1, 70, 65), (0, 40, 5), (0, 90, 3), (1, 7, 200), (0, 20, 1)]):
            lib.gotoCamera(first + eye)
            omm = eye_of(random_axes(n, step), np.random.default_rng(step).normal(size=(n, 3)), 0.3)
            er.set_ommatidia_np(lib, omm)
            lib.setCurrentEyeSamplesPerOmmatidium(spp)
            lib.setCurrentEyeFrameIndex(0)
            before = np.array(lib.getFramePointer(), copy=True).reshape(3, 50, 4) if step % 2 else None
            assert lib.renderFrame() >= 0, er.last_error(lib)
            want = O.render(omm, er.pose_np(lib), spp=spp, eye=eye, want_samples=False)["colour_gpu_order"][0]
            assert np.array_equal(er.colours_np(lib), want), step
            frame = np.array(lib.getFramePointer(), copy=True).reshape(3, 50, 4)
            m = min(n, 50)
            assert np.array_equal(frame[0, :m], oracle.make_color(want)[:m]), step
            if before is not None:
                assert np.array_equal(frame[0, m:], before[0, m:]) and np.array_equal(frame[1:], before[1:]), step
    finally:
        er.setRenderSize(lib, 400, 400)


@pytest.mark.parametrize("poses,n", [(1, 1), (4, 100), (256, 256), (1, 65537), (257, 256)])
def test_batches(lib, tmp_path, poses, n):
    O = load(lib, tmp_path)
    omm = eye_of(random_axes(n, 3), 0.0, 0.2)
    er.set_ommatidia_np(lib, omm)
    lib.setCurrentEyeSamplesPerOmmatidium(2)
    lib.setCurrentEyeFrameIndex(0)
    p = np.random.default_rng(poses).uniform(-1, 1, (poses, 6)).astype(np.float32)
    _, got = er.render_batch_np(lib, p)
    want = O.render(omm, np.stack([oracle.pose12(q) for q in p]), spp=2)["colour_gpu_order"]
    assert np.array_equal(got, want)
