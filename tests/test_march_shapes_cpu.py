"""The autotuner of the 3-D marches, without a GPU: which work-unit shapes it tries
(march_shapes.h, compiled here with the host compiler), and that one disturbed timing of the best
shape does not lose it."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "magudi_amd", "csrc")
SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include "march_shapes.h"
int main(int argc, char** argv) {
  if (!std::strcmp(argv[1], "shapes")) {
    const int n[3] = {atoi(argv[2]), atoi(argv[3]), atoi(argv[4])};
    for (const mgd::MarchShape& s : mgd::march_shapes(n, atoi(argv[5]), atoi(argv[6]), atoi(argv[7])))
      std::printf("%d %d\n", s.tile, s.chunk);
    return 0;
  }
  // pick: shape k takes 1 + k / 50 (forward) and 1 + (n - 1 - k) / 50 (adjoint); sample `bad` of
  // every shape is half as long again
  const int n = atoi(argv[2]), bad = atoi(argv[3]);
  std::vector<int> taken(n, 0);
  int kf = -1, ka = -1;
  const bool ok = mgd::pick_march_shapes(n, [&](int k, float* f, float* a) {
    const float d = taken[k]++ == bad ? 1.5f : 1.f;
    *f = d * (1.f + k / 50.f);
    *a = d * (1.f + (n - 1 - k) / 50.f);
    return true;
  }, &kf, &ka);
  const bool failed = mgd::pick_march_shapes(n, [&](int k, float*, float*) { return k == 0; }, &kf, &ka);
  std::printf("%d %d %d %d\n", ok, failed, kf, ka);
  for (int k = 0; k < n; ++k) std::printf("%d\n", taken[k]);
}
"""


@pytest.fixture(scope="module")
def tool(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("march_shapes")
    (d / "t.cpp").write_text(SOURCE)
    exe = str(d / "t")
    subprocess.check_call([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, "-o", exe, str(d / "t.cpp")])

    def run(*args):
        out = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, check=True)
        return [tuple(map(int, line.split())) for line in out.stdout.splitlines()]
    return run


def _units(n, inst, tile, chunk):
    return inst * -(-n[0] // tile) * -(-n[1] // 16) * -(-n[2] // chunk)


@pytest.mark.parametrize("n,inst", [((256, 256, 256), 1), ((160, 160, 160), 1), ((100, 100, 100), 1),
                                    ((64, 64, 64), 1), ((64, 64, 64), 8), ((33, 20, 35), 2),
                                    ((512, 512, 512), 1), ((128, 256, 512), 1), ((9, 9, 9), 1)])
def test_candidates(tool, n, inst):
    shapes = tool("shapes", *n, inst, 0, 0)
    assert len(set(shapes)) == len(shapes) and {s[0] for s in shapes} == {16, 32}
    for tile in (16, 32):
        chunks = {z for t, z in shapes if t == tile}
        for z in (32, 64, 128):
            # every long chunk that gives half the CUs a unit, whatever just fills the GPU
            assert (z in chunks) == (_units(n, inst, tile, z) >= 128), (tile, z)
        short = {z for z in chunks if z < 32}
        if _units(n, inst, tile, 32) >= 512:
            assert not short
        else:
            assert short and min(short) >= 2
            # the shortest may leave CUs idle, the others not
            assert all(_units(n, inst, tile, z) >= 128 for z in short - {min(short)})


def test_fixed_options(tool):
    assert tool("shapes", 64, 64, 64, 1, 32, 10) == [(32, 10)]
    assert tool("shapes", 64, 64, 64, 1, 0, 10) == [(16, 10), (32, 10)]
    assert {t for t, _ in tool("shapes", 100, 100, 100, 1, 16, 0)} == {16}


@pytest.mark.parametrize("n,bad", [(1, 0), (6, -1), (6, 0), (6, 1), (6, 2), (14, 0)])
def test_a_disturbed_sample_loses_no_shape(tool, n, bad):
    (ok, failed, kf, ka), *taken = tool("pick", n, bad)
    taken = [t[0] for t in taken]
    assert ok == 1 and failed == (1 if n == 1 else 0)
    assert (kf, ka) == (0, n - 1)
    assert all(t in (2, 3) for t in taken) and taken[0] == 3 and taken[-1] == 3
    if n > 1:
        assert taken.count(2) == max(0, n - 6)     # a twentieth: three shapes at either end
