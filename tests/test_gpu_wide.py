"""The 64-wide packet tree (trace mode 2) at the edges of its build and walk.

Whatever tree is walked, a ray's hit is the (t, id) minimum over the triangles
it meets, so samples equal the oracle's bit for bit: tiny scenes around the
leaf and node sizes, coincident triangles, flat and point-like scenes, rays
along the axes, cones wider than a packet, origins far outside the scene and
behind the lens, and waves that mix ommatidia of several places and
directions.
"""
import numpy as np
import pytest

import oracle
from compound_ray_amd import eyerenderer as er
from compound_ray_amd import scenes

pytestmark = pytest.mark.gpu


def soup(n, seed, size=0.25, spread=1.0):
    """n random triangles around the origin."""
    rng = np.random.default_rng(seed)
    centre = rng.uniform(-spread, spread, (n, 1, 3))
    pos = (centre + rng.uniform(-size, size, (n, 3, 3))).reshape(-1, 3).astype(np.float32)
    col = np.concatenate([rng.uniform(0, 1, (3 * n, 3)), np.ones((3 * n, 1))], 1).astype(np.float32)
    return pos, col


def eye_of(axes, positions, acceptance, focal=0.0):
    n = len(axes)
    omm = np.zeros((n, 8), np.float32)
    omm[:, 0:3] = positions
    omm[:, 3:6] = axes
    omm[:, 6] = acceptance
    omm[:, 7] = focal
    return omm


def random_axes(n, seed):
    a = np.random.default_rng(seed).normal(size=(n, 3))
    return (a / np.linalg.norm(a, axis=1, keepdims=True)).astype(np.float32)


def check(lib, tmp_path, pos, col, omm, spp, split=True, modes=(2, 1, 0)):
    idx = np.arange(len(pos), dtype=np.uint32).reshape(-1, 3)
    sc = scenes.Scene([scenes.Mesh("m", pos, idx, col)], eyes=[scenes.Eye("eye", omm)])
    lib.loadGlTFscene(str(scenes.write_gltf(tmp_path, "s", sc)).encode())
    assert er.last_error(lib) == ""
    er.gotoFirstCompoundEye(lib)
    er.set_ommatidia_np(lib, omm)
    lib.setCurrentEyeSamplesPerOmmatidium(spp)
    lib.setCameraPose(0, 0, 0, 0, 0, 0)
    want = oracle.OracleScene.from_scene(sc).render(omm, er.pose_np(lib), spp=spp, want_samples=True)
    lib.setSampleRecording(True)
    lib.setSplitLaunches(split)
    try:
        for mode in modes:
            lib.setTraversalMode(mode)
            lib.setCurrentEyeFrameIndex(0)
            assert lib.renderFrame() >= 0, er.last_error(lib)
            assert np.array_equal(er.samples_np(lib).view(np.uint32), want["samples"].view(np.uint32)), mode
            assert np.array_equal(er.colours_np(lib), want["colour_gpu_order"][0]), mode
    finally:
        lib.setTraversalMode(2)
        lib.setSplitLaunches(True)
        lib.setSampleRecording(False)
    return want


@pytest.mark.parametrize("n", [1, 3, 4, 5, 8, 63, 64, 65, 255, 256, 257, 1021, 4097])
def test_scene_sizes(lib, tmp_path, n):
    """Around the leaf size (4), a full node of leaves and two levels."""
    pos, col = soup(n, n)
    axes = random_axes(70, 2)
    want = check(lib, tmp_path, pos, col, eye_of(axes, -2.5 * axes, 0.05), 33)
    assert n < 64 or (want["samples"].reshape(-1, 4)[:, 3] >= 0).any()


@pytest.mark.parametrize("kind", ["coincident", "flat", "one centre"])
def test_degenerate_scenes(lib, tmp_path, kind):
    """Equal Morton codes (ties by id), no height, no extent at all."""
    if kind == "coincident":
        one, col1 = soup(1, 5)
        pos, col = np.tile(one, (300, 1)), soup(300, 6)[1]
    elif kind == "flat":
        pos, col = soup(700, 7)
        pos[:, 1] = np.float32(-0.5)
    else:
        rng = np.random.default_rng(8)
        half = rng.uniform(-1, 1, (200, 1, 3)).astype(np.float32)
        pos = np.concatenate([half, -half, np.zeros_like(half)], axis=1).reshape(-1, 3)
        pos[2::3] = rng.uniform(-1e-3, 1e-3, (200, 3)).astype(np.float32)
        col = soup(200, 9)[1]
    axes = random_axes(50, 3)
    check(lib, tmp_path, pos, col, eye_of(axes, -2.0 * axes, 0.3), 17)


def test_axis_parallel_rays(lib, tmp_path):
    """Rays exactly along the axes, some inside the planes of box faces."""
    g = np.arange(9, dtype=np.float32) - 4
    x, y = np.meshgrid(g, g)
    c = np.stack([x.ravel(), y.ravel(), np.zeros(81, np.float32)], 1)[:, None, :]
    quad = np.float32([[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 0, 0], [1, 1, 0], [0, 1, 0]])
    pos = np.concatenate([(c + quad).reshape(-1, 3), (c + quad).reshape(-1, 3)[:, [2, 0, 1]]]).astype(np.float32)
    col = np.concatenate([np.random.default_rng(1).uniform(0, 1, (len(pos), 3)), np.ones((len(pos), 1))],
                         1).astype(np.float32)
    axes, at = [], []
    for a in range(3):
        for s in (-1.0, 1.0):
            for off in (0.0, 0.5, 1.0, 2.25):
                d = np.zeros(3)
                d[a] = s
                p = np.full(3, off)
                p[a] = -6.0 * s
                axes.append(d)
                at.append(p)
    want = check(lib, tmp_path, pos, col, eye_of(np.float32(axes), np.float32(at), 0.0), 5)
    assert (want["samples"].reshape(-1, 4)[:, 3] >= 0).any()


@pytest.mark.parametrize("acceptance", [0.5, 1.5, 3.0])
def test_cones_wider_than_a_packet(lib, tmp_path, acceptance):
    """Samples of one ommatidium up to opposite directions."""
    pos, col = soup(3000, 11, size=0.05)
    axes = random_axes(20, 4)
    check(lib, tmp_path, pos, col, eye_of(axes, np.float32([0.1, 0.2, -0.1]), acceptance), 130)


@pytest.mark.parametrize("distance", [3.0, 30.0, 3000.0])
@pytest.mark.parametrize("focal", [0.0, 0.5, -1.5])
def test_origins(lib, tmp_path, distance, focal):
    """Origins out to far beyond the range that the boxes' padding covers, and
    rays that start beyond or behind theirs."""
    pos, col = soup(2000, 12, size=0.08)
    axes = random_axes(40, 5)
    want = check(lib, tmp_path, pos, col, eye_of(axes, -distance * axes, 1.0 / distance, focal), 65, modes=(2, 0))
    assert (want["samples"].reshape(-1, 4)[:, 3] >= 0).any()


@pytest.mark.parametrize("spp", [1, 3, 8, 32])
@pytest.mark.parametrize("apart", [0.0, 1e-3, 0.05, 5.0])
def test_mixed_waves(lib, tmp_path, spp, apart):
    """The unit renderer packs ommatidia of any direction and place into one
    wave: up to 64 of them, up to metres apart."""
    pos, col = soup(3000, 13, size=0.05)
    axes = random_axes(150, 6)
    at = np.random.default_rng(7).uniform(-apart, apart, (150, 3)).astype(np.float32)
    check(lib, tmp_path, pos, col, eye_of(axes, at, 0.2), spp, split=False, modes=(2, 1))


def test_rays_that_hit_nothing(lib, tmp_path):
    """Ommatidia without an axis (rays that are not numbers) beside ordinary
    ones: misses, as in every other walk."""
    pos, col = soup(500, 14)
    axes = random_axes(64, 8)
    axes[::5] = 0.0
    omm = eye_of(axes, -2.0 * axes, 0.1)
    for split in (True, False):
        check(lib, tmp_path, pos, col, omm, 9, split=split, modes=(2,))


@pytest.mark.parametrize("grab,blocks", [(0, 0), (1, 1), (5, 3), (64, 1), (7, 100000)])
@pytest.mark.parametrize("counts", [None, "uneven"])
def test_unit_grid_shapes(lib, tmp_path, grab, blocks, counts):
    """Any grab size and grid, down to one workgroup that strides over all the
    work, gives every (pose, ommatidium) unit once: batches of an ommatidium
    count that is not a power of two, at one and at several poses."""
    pos, col = soup(800, 15)
    omm = eye_of(random_axes(131, 9), -2.0 * random_axes(131, 9), 0.1)
    sc = scenes.Scene([scenes.Mesh("m", pos, np.arange(len(pos), dtype=np.uint32).reshape(-1, 3), col)],
                      eyes=[scenes.Eye("eye", omm)])
    lib.loadGlTFscene(str(scenes.write_gltf(tmp_path, "s", sc)).encode())
    er.gotoFirstCompoundEye(lib)
    er.set_ommatidia_np(lib, omm)
    n = None if counts is None else scenes.log_uniform_counts(131, 1, 130, seed=4)
    lib.setCurrentEyeSamplesPerOmmatidium(13)
    er.set_sample_counts(lib, n)
    poses6 = np.zeros((5, 6), np.float32)
    poses6[:, 0] = np.linspace(-0.2, 0.2, 5)
    poses6[:, 4] = np.arange(5)
    poses12 = np.stack([oracle.pose12(p) for p in poses6])
    lib.setRenderTuning(grab, blocks)
    try:
        for k in (1, 5):
            want = oracle.OracleScene.from_scene(sc).render(omm, poses12[:k], spp=13, counts=n,
                                                            frame=lib.getCurrentEyeFrameIndex())
            _, rgb = er.render_batch_np(lib, poses6[:k])
            assert np.array_equal(rgb, want["colour_gpu_order"]), k
    finally:
        lib.setRenderTuning(0, 0)
        er.set_sample_counts(lib, None)


@pytest.mark.parametrize("spp", [1, 64, 65, 512, 513, 575, 577, 1100])
@pytest.mark.parametrize("width", [40, 71, 90])
@pytest.mark.parametrize("split", [0, 1])
def test_frame_chunks(lib, tmp_path, spp, width, split):
    """renderFrame's 64-sample chunks on different waves, around the reduction's
    runs of eight chunks: colours, and the frame row of single_dimension_fast
    narrower and wider than the eye (pixels beyond it stay as they were)."""
    pos, col = soup(300, 16)
    omm = eye_of(random_axes(71, 10), -2.0 * random_axes(71, 10), 0.2)
    sc = scenes.Scene([scenes.Mesh("m", pos, np.arange(len(pos), dtype=np.uint32).reshape(-1, 3), col)],
                      eyes=[scenes.Eye("eye", omm)])
    lib.loadGlTFscene(str(scenes.write_gltf(tmp_path, "s", sc)).encode())
    er.gotoFirstCompoundEye(lib)
    er.set_ommatidia_np(lib, omm)
    lib.setCurrentEyeSamplesPerOmmatidium(spp)
    lib.setCameraPose(0, 0, 0, 0, 0, 0)
    er.setRenderSize(lib, width, 2)
    lib.setTaskSplit(split)
    try:
        want = oracle.OracleScene.from_scene(sc)
        for frame in range(3):
            assert lib.renderFrame() >= 0, er.last_error(lib)
            ref = want.render(omm, er.pose_np(lib), spp=spp, frame=frame)["colour_gpu_order"][0]
            assert lib.getLastRenderKernel() == b"k_render_tasks"
            assert np.array_equal(er.colours_np(lib), ref)
            pixels = np.array(lib.getFramePointer(), copy=True).reshape(2, width, 4)
            n = min(width, 71)
            assert np.array_equal(pixels[0, :n], oracle.make_color(ref)[:n])
            assert not pixels[0, n:].any() and not pixels[1].any()
    finally:
        lib.setTaskSplit(2)
        er.setRenderSize(lib, 400, 400)
