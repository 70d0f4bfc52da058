"""Launch shapes of the sweeps (csrc/launch.h, plain C++) over every block
size, workgroup size, system and window: what fits, and what one context's
shape may demand of the limits that all contexts of a process share."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "amun_amd", "csrc")

SHAPES = r"""
#include <cstdio>
#include <initializer_list>
#include "launch.h"
using namespace amun_dev;
int main() {
  for (int nd = 2; nd <= 3; nd++)
    for (int nv : {4, 5, 8, 9})
      for (int es : {4, 8})
        for (int sr = 0; sr < 2; sr++)
          for (int R = 0; R <= 3; R++)
            for (int dir = 0; dir < nd; dir++)
              for (int nc = 4; nc <= 64; nc += 4)
                for (int wg : {64, 128, 256}) {
                  const SweepCfg c{nv, es, sr != 0, R, nd, nc, 37};
                  const SweepShape s = sweep_shape(c, dir, wg);
                  std::printf("%d %d %d %d %d %d %d %d %d %d %u %zu %zu\n", nd, nv, es, sr, R, dir,
                              nc, wg, s.np, s.lanes, s.grid, s.lds, sweep_lds_limit(c, dir));
                }
}
"""


def _run(tmp_path, text):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(text)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout


@pytest.fixture(scope="module")
def shapes(tmp_path_factory):
    out = _run(tmp_path_factory.mktemp("launch"), SHAPES)
    return [[int(x) for x in line.split()] for line in out.splitlines()]


def test_shapes_cover_every_pencil(shapes):
    for nd, nv, es, sr, R, d, nc, wg, np_, lanes, grid, lds, _ in shapes:
        total = 37 * nc ** (nd - 1)
        assert np_ % 2 == 0 and np_ * (nc + 2) <= lanes <= max(wg, (2 * (nc + 2) + 63) // 64 * 64) <= 256
        assert (grid - 1) * np_ < total <= grid * np_


def test_lds_limit_does_not_depend_on_the_block_size(shapes):
    """The limit set on a kernel covers the launches of every context that
    uses it, and lies within the 160 KiB of a CU."""
    limits = {}
    for nd, nv, es, sr, R, d, nc, wg, np_, lanes, grid, lds, limit in shapes:
        assert lds <= limit <= 160 * 1024
        assert limits.setdefault((nd, nv, es, sr, R, d), limit) == limit


RULE = r"""
#include <cstdio>
#include <initializer_list>
#include "launch.h"
using namespace amun_dev;
int main() {
  for (int nd = 2; nd <= 3; nd++)
    for (int nc : {4, 8, 16, 64})
      for (int nblk : {1, 7, 64, 146, 147, 300, 4096})
        for (int dir = 0; dir < nd; dir++) {
          const SweepCfg c{9, 8, false, 2, nd, nc, nblk};
          for (int wg : {0, 64, 128, 256}) {
            const SweepShape s = launch_shape(c, dir, wg);
            std::printf("%d %d %u", wg, s.np, s.grid);
            for (int k : {64, 128, 256}) {
              const SweepShape t = sweep_shape(c, dir, k);
              std::printf(" %d %u", t.np, t.grid);
            }
            std::printf("\n");
          }
        }
}
"""


def test_a_chosen_workgroup_size_holds(tmp_path):
    """Chosen sizes run as chosen on every grid; the default is the largest
    size that gives every CU a workgroup, the smallest where none does."""
    small = 0
    for line in _run(tmp_path, RULE).splitlines():
        wg, np_, grid, *by = [int(x) for x in line.split()]
        size = {64: by[:2], 128: by[2:4], 256: by[4:]}
        small += size[256][1] < 256
        if wg:
            assert [np_, grid] == size[wg]
        else:
            want = next((k for k in (256, 128, 64) if size[k][1] >= 256), 64)
            assert [np_, grid] == size[want]
    assert small
