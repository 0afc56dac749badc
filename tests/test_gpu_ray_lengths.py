"""Free rays whose directions are very long or very short.

A direction scaled by a power of two divides the distances by it, exactly: ids
are those of the directions of ordinary length, and distances theirs divided
(rounded once where they are subnormal).  Misses return the tmax given.
"""
import numpy as np
import pytest

import oracle
from compound_ray_amd import eyerenderer as er
from compound_ray_amd import scenes
from test_gpu_wide import eye_of, random_axes, soup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3000, 20000])   # a ray per wave, and eight
@pytest.mark.parametrize("exponent", [-146, -127, -110, -90, -72, -60, -20, 0, 30, 60, 100, 119, 121, 124, 126])
def test_lengths(lib, tmp_path, n, exponent):
    pos, col = soup(3000, 12, size=0.08)
    sc = scenes.Scene([scenes.Mesh("m", pos, np.arange(len(pos), dtype=np.uint32).reshape(-1, 3), col)],
                      eyes=[scenes.Eye("eye", eye_of(random_axes(4, 1), 0.0, 0.1))])
    lib.loadGlTFscene(str(scenes.write_gltf(tmp_path, "s", sc)).encode())
    assert er.last_error(lib) == ""
    O = oracle.OracleScene.from_scene(sc)
    rng = np.random.default_rng(n)
    # three bits of a direction survive the shortest lengths
    d = np.round(rng.normal(size=(n, 3)) * 2).clip(-7, 7) / 8
    d[~d.any(axis=1)] = [0.5, 0.25, 0.0]
    if exponent > -100:
        d += rng.normal(size=(n, 3)) * 0.05
        d /= np.abs(d).max(axis=1, keepdims=True) * 1.01
    plain = np.zeros((n, 8), np.float32)
    plain[:, 0:3] = rng.uniform(-1.2, 1.2, (n, 3))
    plain[:, 4:7] = d
    plain[:, 3] = rng.choice([0.0, 0.25], n)
    plain[:, 7] = rng.choice([2.0, 1e3, np.inf], n)
    rays = plain.copy()
    rays[:, 4:7] = np.ldexp(plain[:, 4:7], exponent)
    with np.errstate(over="ignore", under="ignore"):
        rays[:, 3] = np.ldexp(plain[:, 3], -exponent)
        rays[:, 7] = np.ldexp(plain[:, 7], -exponent)
    # what the rays given stand for, back at an ordinary length: their limits have been rounded
    same = plain.copy()
    same[:, 3] = np.ldexp(rays[:, 3], exponent)
    same[:, 7] = np.ldexp(rays[:, 7], exponent)
    same[np.isinf(rays[:, 7]), 7] = np.inf
    assert np.array_equal(np.ldexp(rays[:, 4:7], -exponent), plain[:, 4:7])
    want, wt = O.trace(same, bvh=False)
    assert 0.01 < (want >= 0).mean() < 0.99
    ids, tbb = er.trace_np(lib, rays)
    hit = want >= 0
    assert np.array_equal(ids, want)
    with np.errstate(over="ignore"):
        t = np.ldexp(wt[hit, 0], -exponent).astype(np.float32)
    assert np.array_equal(tbb[hit, 0], t)
    assert np.array_equal(tbb[hit, 1:], wt[hit, 1:])
    assert np.array_equal(tbb[~hit, 0], rays[~hit, 7])
