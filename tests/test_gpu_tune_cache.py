"""Autotune cache files written before the 64-wide walk.

Their entries were timed on other kernels: they are kept in the file, but a
batch of such a workload is tuned anew, and its colours stay the oracle's.
"""
import numpy as np
import pytest

import oracle
from compound_ray_amd import eyerenderer as er
from compound_ray_amd import scenes
from test_gpu_wide import eye_of, random_axes, soup

pytestmark = pytest.mark.gpu


def entries(path):
    return {ln.split()[0]: [float(v) for v in ln.split()[1:]] for ln in path.read_text().splitlines()
            if ln and not ln.startswith("#")}


def test_old_entries_are_not_used(lib, tmp_path):
    n, tris = 211, 523
    pos, col = soup(tris, 8)
    omm = eye_of(random_axes(n, 1), 0.0, 0.1)
    sc = scenes.Scene([scenes.Mesh("m", pos, np.arange(len(pos), dtype=np.uint32).reshape(-1, 3), col)],
                      eyes=[scenes.Eye("eye", omm)])
    lib.loadGlTFscene(str(scenes.write_gltf(tmp_path, "s", sc)).encode())
    assert er.last_error(lib) == ""
    er.gotoFirstCompoundEye(lib)
    er.set_ommatidia_np(lib, omm)
    lib.setCurrentEyeSamplesPerOmmatidium(7)
    O = oracle.OracleScene.from_scene(sc)
    old = f"tris{tris}_nodes{O.info()['nodes']}_leaf4_omm{n}_spp{7 * n}_stats0_rec0"
    cache = tmp_path / "tune.txt"
    cache.write_text(f"# key units_per_grab blocks traversal ms\n{old} 16 512 2 0.0001\n")
    poses = np.random.default_rng(3).uniform(-1, 1, (4, 6)).astype(np.float32)
    try:
        assert lib.setAutotuneCacheFile(str(cache).encode()) >= 1
        lib.setBatchAutotune(1)
        lib.setCurrentEyeFrameIndex(0)
        _, rgb = er.render_batch_np(lib, poses)
        want = O.render(omm, np.stack([oracle.pose12(p) for p in poses]), spp=7)["colour_gpu_order"]
        assert np.array_equal(rgb, want)
        now = entries(cache)
        assert now[old] == [16, 512, 2, 0.0001]
        new = [k for k in now if k.startswith(old) and k != old]
        assert len(new) == 1 and now[new[0]][3] > 0.0001
    finally:
        lib.setBatchAutotune(0)
        lib.setAutotuneCacheFile(None)
