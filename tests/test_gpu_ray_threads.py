"""traceRays from several threads at a time.

The calls share the buffers that rays go through in pieces, which grow with the
longest list: every thread gets the hits of its own rays, alone or beside
frames of an eye.
"""
import threading

import numpy as np
import pytest

import oracle
from compound_ray_amd import eyerenderer as er
from compound_ray_amd import scenes
from test_gpu_wide import eye_of, random_axes, soup

pytestmark = pytest.mark.gpu


def rays_of(n, seed):
    rng = np.random.default_rng(seed)
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = rng.uniform(-2, 2, (n, 3))
    rays[:, 4:7] = rng.normal(size=(n, 3))
    rays[:, 7] = 1e16
    return rays


@pytest.mark.parametrize("counts", [(700, 700, 700, 700), (300, 20000, 140000, 300007)])
@pytest.mark.parametrize("frames", [False, True])
def test_threads(lib, tmp_path, counts, frames):
    pos, col = soup(500, 8)
    omm = eye_of(random_axes(300, 1), 0.0, 0.1)
    sc = scenes.Scene([scenes.Mesh("m", pos, np.arange(len(pos), dtype=np.uint32).reshape(-1, 3), col)],
                      eyes=[scenes.Eye("eye", omm)])
    lib.loadGlTFscene(str(scenes.write_gltf(tmp_path, "s", sc)).encode())
    assert er.last_error(lib) == ""
    er.gotoFirstCompoundEye(lib)
    er.set_ommatidia_np(lib, omm)
    lib.setCurrentEyeSamplesPerOmmatidium(20)
    O = oracle.OracleScene.from_scene(sc)
    rays = [rays_of(n, k) for k, n in enumerate(counts)]
    want = [O.trace(r) for r in rays]
    gate = threading.Barrier(len(counts) + int(frames))
    wrong = []

    def trace(k):
        gate.wait()
        for turn in range(6):
            ids, tbb = er.trace_np(lib, rays[k])
            hit = ids >= 0
            if not np.array_equal(ids, want[k][0]) or not np.array_equal(tbb[hit], want[k][1][hit]):
                wrong.append((k, turn))

    threads = [threading.Thread(target=trace, args=(k,)) for k in range(len(counts))]
    for t in threads:
        t.start()
    if frames:
        gate.wait()
        for turn in range(6):
            lib.setCurrentEyeFrameIndex(0)
            assert lib.renderFrame() >= 0
            ref = O.render(omm, er.pose_np(lib), spp=20)["colour_gpu_order"][0]
            assert np.array_equal(er.colours_np(lib), ref)
    for t in threads:
        t.join(60)
    assert not wrong and not any(t.is_alive() for t in threads)
