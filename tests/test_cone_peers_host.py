"""The cone beam's peer table (class_peers, sgd_amd/csrc/symmetry.hpp), compiled
for the host: every view finds the views its symmetries map it onto among its
class's slots, over one and several turns; tables whose classes do not hold them
are refused rather than given slot 0."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from test_symmetry_host import ROOT, scan, turn

MAIN = r"""
#include <cstdio>
#include <vector>
#include "symmetry.hpp"
using namespace sgdct;
int main() {
  int nx, ny, nu, np, allowed, broken;
  if (scanf("%d %d %d %d %d %d", &nx, &ny, &nu, &np, &allowed, &broken) != 6) return 1;
  std::vector<ViewGeo> v(np);
  for (auto& a : v)
    if (scanf("%lf %lf %lf %lf %lf %lf", &a.px, &a.py, &a.e0x, &a.e0y, &a.pux, &a.puy) != 6) return 1;
  SymTables t = find_symmetries(v, nx, ny, nu, (unsigned)allowed, kMaxSym, 6e-9, false, false, 1);
  if (broken) std::swap(t.rep_view[0], t.rep_view[t.nh()]);
  std::vector<int> peer;
  printf("%d %d\n", t.nh(), class_peers(t, &peer) ? 1 : 0);
  auto line = [](const auto& a) { for (auto x : a) printf("%d ", (int)x); printf("\n"); };
  line(t.rep_view); line(t.view); line(peer);
}
"""


@pytest.fixture(scope="module")
def peers(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("peers")
    (d / "main.cpp").write_text(MAIN)
    subprocess.check_call([hipcc, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1",
                           "-I", os.path.join(ROOT, "sgd_amd", "csrc"), str(d / "main.cpp"), "-o", str(d / "main")])

    def run(nx, ny, angles, allowed, broken=0):
        views = scan(angles, 45)
        text = "%d %d 45 %d %d %d\n" % (nx, ny, len(views), allowed, broken)
        text += "\n".join(" ".join("%.17g" % x for x in v) for v in views)
        out = subprocess.run([str(d / "main")], input=text, capture_output=True, text=True, check=True).stdout
        rows = [np.array(s.split(), dtype=int) for s in out.split("\n")[:4]]
        return rows[0][0], bool(rows[0][1]), rows[1], rows[2], rows[3]

    return run


@pytest.mark.parametrize("nx,ny,n,per,allowed,want", [
    (12, 12, 360, 360, 0x55, 4), (12, 12, 360, 360, 0xff, 8), (12, 10, 720, 360, 0x55, 4),
    (12, 12, 720, 360, 0xff, 8), (9, 9, 1080, 360, 0xff, 8), (9, 14, 27, 9, 0x55, 2), (7, 7, 24, 12, 0xff, 8)])
def test_peers_are_the_symmetric_views(peers, nx, ny, n, per, allowed, want):
    nh, ok, rep_view, view, peer = peers(nx, ny, 2 * np.pi * np.arange(n) / per, allowed)
    assert nh == want and ok
    view, peer, classes = view.reshape(n, nh), peer.reshape(-1, nh), rep_view.reshape(-1, nh)
    for s, v in enumerate(rep_view):
        if v >= 0:
            assert np.array_equal(classes[s // nh][peer[s]], view[v]), (s, v)


def test_classes_without_their_views_are_refused(peers):
    nh, ok, *_ = peers(12, 12, turn(60), 0x55, broken=1)
    assert nh == 4 and not ok
