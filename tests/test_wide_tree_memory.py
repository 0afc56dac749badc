"""A scene loads without its 64-wide tree when there is no memory for that.

The builder is linked with allocators of the test's own (host memory, no GPU),
of which the k-th call runs out: whichever it is of those before the first
kernel, the scene keeps its 4-wide tree and no error.
"""
import pathlib
import shutil
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "compound-ray_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

MAIN = """
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstdlib>
#include "device_scene.h"

static int left, held, cleared;
static hipError_t fails = hipErrorOutOfMemory;
static hipError_t take(void** p, size_t n) {
  if (left-- == 0) return fails;
  *p = malloc(n);
  ++held;
  return hipSuccess;
}
static hipError_t give(void* p) {
  free(p);
  --held;
  return hipSuccess;
}
extern "C" hipError_t __wrap_hipMalloc(void** p, size_t n) { return take(p, n); }
extern "C" hipError_t __wrap_hipHostMalloc(void** p, size_t n, unsigned) { return take(p, n); }
extern "C" hipError_t __wrap_hipFree(void* p) { return give(p); }
extern "C" hipError_t __wrap_hipHostFree(void* p) { return give(p); }
extern "C" hipError_t __wrap_hipGetLastError() { return ++cleared, hipSuccess; }

int main(int argc, char** argv) {
  if (argc > 2) fails = hipErrorInvalidValue;   // a failure of another kind
  eye::DeviceScene scene;
  scene.tri_count = 5000;
  left = atoi(argv[1]);
  std::string err;
  const bool ok = eye::build_wide_tree(&scene, nullptr, &err);
  printf("%d %d %d %d %d\\n", ok, !err.empty(), scene.wide_nodes != nullptr, held, cleared > 0);
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not pathlib.Path(HIPCC).exists():
        pytest.skip("hipcc not available")
    d = tmp_path_factory.mktemp("memory")
    (d / "main.hip").write_text(MAIN)
    wraps = ",".join(f"--wrap={n}" for n in ("hipMalloc", "hipHostMalloc", "hipFree", "hipHostFree",
                                             "hipGetLastError"))
    cmd = [HIPCC, "--offload-arch=gfx950", "-std=c++17", "-O1", "-ffp-contract=off", "-w",
           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", str(CSRC),
           "-o", str(d / "main"), str(d / "main.hip"), str(CSRC / "wide_bvh.hip"), str(CSRC / "scan.hip"),
           f"-Wl,{wraps}"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]

    def run(*args):
        out = subprocess.run([str(d / "main"), *map(str, args)], capture_output=True, text=True, timeout=60)
        assert out.returncode == 0, out.stderr[-2000:]
        return [int(v) for v in out.stdout.split()]

    return run


# the codes and their copy, the order and its copy, the histogram, ranges,
# parents and flag, then the prefix sums' three
@pytest.mark.parametrize("k", range(11))
def test_out_of_memory(program, k):
    ok, error, tree, held, cleared = program(k)
    assert ok and not error and not tree and held == 0
    assert cleared   # the next call does not report it


@pytest.mark.parametrize("k", range(11))
def test_other_failures(program, k):
    ok, error, tree, held, _ = program(k, "other")
    assert not ok and error and not tree and held == 0
