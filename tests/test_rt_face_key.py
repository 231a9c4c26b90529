"""The ray tracer's number of a cell face's corner, compiled for the host from the kernels' own source: two
corners, each inside the grid or one voxel outside it, have successive numbers only if they lie in one column,
one voxel apart along z (that is when a lane hands its upper taps to the next lane)."""

import os
import shutil
import subprocess

import pytest

from vamtoolbox_amd import build

CSRC = os.path.join(os.path.dirname(build.__file__), "csrc")

SOURCE = r"""
#include <cstdio>
#include <map>
#include "vamx_internal.h"
using namespace vamx;

int main() {
  int bad = 0;
  const int sizes[][3] = {{2, 2, 2}, {3, 4, 5}, {5, 3, 1}, {4, 7, 3}, {1, 2, 9}};
  for (auto& d : sizes) {
    RtDev g{};
    g.nx = d[0];
    g.ny = d[1];
    g.nz = d[2];
    struct Corner { int x, y, z; };
    std::map<unsigned, Corner> at;
    for (int x = -1; x <= g.nx; ++x)
      for (int y = -1; y <= g.ny; ++y)
        for (int z = -1; z <= g.nz; ++z)
          if (!at.insert({rt_face_key(g, x, y, z), Corner{x, y, z}}).second) ++bad;   // two corners, one number
    // receiving corners lie inside the grid along z
    for (auto& [key, c] : at) {
      const auto next = at.find(key + 1u);
      if (next == at.end() || next->second.z < 0 || next->second.z >= g.nz) continue;
      const Corner& n = next->second;
      if (n.x != c.x || n.y != c.y || n.z != c.z + 1) {
        ++bad;
        std::printf("%d x %d x %d: (%d %d %d) before (%d %d %d)\n", g.nx, g.ny, g.nz, c.x, c.y, c.z, n.x, n.y, n.z);
      }
    }
  }
  std::printf("%d faults\n", bad);
  return bad != 0;
}
"""


@pytest.mark.skipif(not shutil.which(build.HIPCC), reason="no hipcc")
def test_successive_numbers_are_one_column(tmp_path):
    src, exe = tmp_path / "key.hip", tmp_path / "key"
    src.write_text(SOURCE)
    subprocess.run([build.HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-I", CSRC, "-Wno-unused-result",
                    str(src), "-o", str(exe)], check=True, timeout=300)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stdout
