"""The back projection's nodes (lower row and weights per voxel column and angle) on the host, compiled from
the kernels' own source: every row that a node names lies in the sinogram, the opposite angle's mirrored rows
too, and the nodes of all passes give each column what np.interp gives it angle by angle -- for detectors
shifted by up to their whole width, where the two angles of a pair share no, one or several bins."""

import os
import shutil
import subprocess

import pytest

from vamtoolbox_amd import build

CSRC = os.path.join(os.path.dirname(build.__file__), "csrc")

SOURCE = r"""
#include <cstdio>
#include <vector>
#include "par_core.h"
using namespace vamx;

static int bad = 0;
static void fail(const char* what, const ParDev& g, int pix, int u) {
  if (++bad <= 20) std::printf("n %d D %d column %d unit %d: %s\n", g.n, g.pair_D, pix, u, what);
}

// a column's sum over the nodes of one pass
template <bool COMB, int PASS>
static void pass(const ParDev& g, const std::vector<double>& s, int pix, double x, double y, double& sum) {
  const int steps = COMB ? g.n_units : g.na;
  for (int u = 0; u < steps; ++u) {
    int i = u, i2 = -1;
    if (COMB) { i = g.units[2 * u]; i2 = g.units[2 * u + 1]; }
    bool single = false;
    const BpNode nd = bp_node<COMB, PASS>(g, true, i, i2, x, y, single);
    if (nd.jr < 0) continue;
    if (nd.jr > g.n - 2) { fail("row past the sinogram", g, pix, u); continue; }
    const int a = PASS == BP_TWO ? i2 : i;
    double b0 = s[nd.jr * g.na + a], b1 = s[(nd.jr + 1) * g.na + a];
    if (COMB && PASS == BP_ALL && i2 >= 0) {
      const int m = 2 * g.c + g.pair_D - nd.jr;   // mirrored bins m and m - 1
      if (m > g.n - 1 || m < 1) { fail("mirrored row past the sinogram", g, pix, u); continue; }
      b0 += s[m * g.na + i2];
      b1 += s[(m - 1) * g.na + i2];
    }
    sum += nd.w0 * b0 + nd.w1 * b1;
  }
}

int main() {
  for (int n : {2, 3, 4, 5, 8, 17, 32, 33})
    for (int D = -n; D <= n; ++D)
      for (int half : {1, 2, 6}) {
        const int na = 2 * half;
        std::vector<double> cs(2 * na), s((size_t)n * na);
        std::vector<int> units;
        for (int i = 0; i < na; ++i) {
          const double ang = i * (360.0 / na) * (M_PI / 180.0);
          cs[2 * i] = std::cos(ang);
          cs[2 * i + 1] = std::sin(ang);
        }
        for (int i = 0; i < half; ++i) { units.push_back(i); units.push_back(i + half); }
        for (size_t k = 0; k < s.size(); ++k) s[k] = 0.1 + (double)((k * 2654435761u) % 1000) / 1000.0;
        ParDev g{};
        g.n = n;
        g.nz = 32;
        g.na = na;
        g.c = n / 2;
        g.det_offset = D / 2.0;
        g.xp0 = (0 - g.c) - g.det_offset;
        g.xp_last = (n - 1 - g.c) - g.det_offset;
        g.inv_cos = 1.0;
        g.radius = (n - 1) / 2.0;
        g.cs = cs.data();
        g.units = units.data();
        g.n_units = half;
        g.pair_D = D;
        const int lo2 = std::max(0, 2 * g.c + D - (n - 1)), hi2 = std::min(n - 1, 2 * g.c + D);
        g.pair_ok = hi2 >= lo2 && std::abs(D) < n;   // as the plan's units ask
        g.fp_pair = 1;
        const bool comb = bp_combines(g);
        for (int pix = 0; pix < n * n; ++pix) {
          const double y = pix / n - g.c, x = pix % n - g.c;
          double want = 0.0, got = 0.0;
          for (int i = 0; i < na; ++i) {
            int j, j1;
            float w;
            if (interp_node(g, x * cs[2 * i] - y * cs[2 * i + 1], j, j1, w))
              want += s[j * na + i] + w * (s[j1 * na + i] - s[j * na + i]);
          }
          if (comb) {
            pass<true, BP_ALL>(g, s, pix, x, y, got);
            pass<true, BP_ONE>(g, s, pix, x, y, got);
            pass<true, BP_TWO>(g, s, pix, x, y, got);
          } else {
            pass<false, BP_ALL>(g, s, pix, x, y, got);
          }
          if (std::fabs(got - want) > 1e-6 * na) fail("another sum than angle by angle", g, pix, -1);
        }
      }
  std::printf("%d faults\n", bad);
  return bad != 0;
}
"""


@pytest.mark.skipif(not shutil.which(build.HIPCC), reason="no hipcc")
def test_nodes_stay_in_the_sinogram(tmp_path):
    src, exe = tmp_path / "nodes.hip", tmp_path / "nodes"
    src.write_text(SOURCE)
    subprocess.run([build.HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-ffp-contract=off", "-I", CSRC,
                    "-Wno-unused-result", str(src), "-o", str(exe)], check=True, timeout=300)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stdout
