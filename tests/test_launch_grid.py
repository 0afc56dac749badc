"""Grid sizes of launches whose work may exceed one grid.

The host functions are compiled on their own: HIP launches fewer than 2^32
threads along x, and every grab of a batch of up to 2^32 - 65,537 units has to
lie under the grid's stride.
"""
import pathlib
import shutil
import subprocess

import pytest

from compound_ray_amd import eyerenderer as er
from compound_ray_amd import scenes

CSRC = pathlib.Path(__file__).resolve().parents[1] / "compound-ray_amd" / "csrc"
MOST = 2**32 - 65537

MAIN = """
#include <cstdio>
#include <cstdlib>
#include "launch_grid.h"
int main(int argc, char** argv) {
  for (int k = 1; k + 3 < argc; k += 4) {
    const eye::UnitGrid g = eye::unit_grid(strtoull(argv[k], nullptr, 10), atoi(argv[k + 1]), atoi(argv[k + 2]),
                                           atoi(argv[k + 3]));
    printf("%u %u\\n", g.blocks, g.grid);
  }
}
"""


@pytest.fixture(scope="module")
def grids(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("grid")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", str(CSRC), "-o", str(d / "main"), str(d / "main.cpp")], check=True)

    def of(calls):
        args = [str(v) for c in calls for v in c]
        out = subprocess.run([str(d / "main"), *args], capture_output=True, text=True, check=True).stdout
        return [tuple(int(v) for v in line.split()) for line in out.splitlines()]

    return of


def test_unit_grids(grids):
    calls = [(units, grab, threads, fixed)
             for units in (1, 63, 64, 65, 2**26 - 1, 2**26, 2**26 + 1, 2**28 + 3, 2**31, MOST)
             for grab in (1, 6, 16, 64) for threads in (64, 256) for fixed in (0, 1, 1000, 2**31 - 1)]
    for (units, grab, threads, fixed), (blocks, grid) in zip(calls, grids(calls)):
        case = (units, grab, threads, fixed)
        per_block = grab * (threads // 64)
        assert blocks == -(-units // per_block), case
        assert 1 <= grid <= blocks and grid * threads < 2**32, case
        # the kernel's index of 32 bits stays below 2^32
        assert blocks + grid <= 2**32, case
        asked = fixed * (256 // threads) if fixed else blocks
        # as many as asked for, unless there is less work or no more can be launched
        assert grid == min(asked, blocks, (2**32 - 1) // threads, 2**32 - blocks), case


@pytest.mark.gpu
def test_batch_of_more_grabs_than_a_grid_takes(lib, tmp_path):
    """67,207,168 units one by one, by a grid that strides: the colours of the
    same units 64 by 64, in 1,050,112 workgroups."""
    import numpy as np

    from test_gpu_wide import eye_of, random_axes, soup

    pos, col = soup(40, 8)
    omm = eye_of(random_axes(16384, 1), 0.0, 0.1)
    sc = scenes.Scene([scenes.Mesh("m", pos, np.arange(len(pos), dtype=np.uint32).reshape(-1, 3), col)],
                      eyes=[scenes.Eye("eye", omm[:4])])
    lib.loadGlTFscene(str(scenes.write_gltf(tmp_path, "s", sc)).encode())
    assert er.last_error(lib) == ""
    er.gotoFirstCompoundEye(lib)
    er.set_ommatidia_np(lib, omm)
    lib.setCurrentEyeSamplesPerOmmatidium(1)
    poses = np.zeros((4102, 6), np.float32)
    poses[:, 4] = np.linspace(0, 6, 4102)
    try:
        out = []
        for grab in (64, 1):
            lib.setRenderTuning(grab, 0)
            lib.setCurrentEyeFrameIndex(0)
            out.append(er.render_batch_np(lib, poses)[1])
        assert out[0].any()
        assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
    finally:
        lib.setRenderTuning(0, 0)
