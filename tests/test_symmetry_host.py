"""Tables of a scan's symmetries (sgd_amd/csrc/symmetry.hpp), compiled for the
host and checked against the geometry: every symmetry permutes the views, maps
sources onto sources and bins onto bins (reversed where it mirrors), the
representative views reach every view exactly once, and the tiles of the
fundamental domain write every pixel exactly once."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAIN = r"""
#include <cstdio>
#include <vector>
#include "symmetry.hpp"
using namespace sgdct;
int main() {
  int nx, ny, nu, np, allowed, most;
  double tol;
  if (scanf("%d %d %d %d %d %d %lf", &nx, &ny, &nu, &np, &allowed, &most, &tol) != 7) return 1;
  std::vector<ViewGeo> v(np);
  for (auto& a : v)
    if (scanf("%lf %lf %lf %lf %lf %lf", &a.px, &a.py, &a.e0x, &a.e0y, &a.pux, &a.puy) != 6) return 1;
  const SymTables t = find_symmetries(v, nx, ny, nu, (unsigned)allowed, most, tol);
  auto line = [](const auto& a) { for (auto x : a) printf("%d ", (int)x); printf("\n"); };
  line(t.op); line(t.rep); line(t.rep_view); line(t.view); line(t.tile); line(t.owner);
}
"""


@pytest.fixture(scope="module")
def tables(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("sym")
    (d / "main.cpp").write_text(MAIN)
    subprocess.check_call([hipcc, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1",
                           "-I", os.path.join(ROOT, "sgd_amd", "csrc"), str(d / "main.cpp"), "-o", str(d / "main")])

    def run(nx, ny, nu, views, allowed, most=8, tol=6e-9):
        text = "%d %d %d %d %d %d %.17g\n" % (nx, ny, nu, len(views), allowed, most, tol)
        text += "\n".join(" ".join("%.17g" % x for x in v) for v in views)
        out = subprocess.run([str(d / "main")], input=text, capture_output=True, text=True, check=True).stdout
        return [np.array(s.split(), dtype=int) for s in out.split("\n")[:6]]

    return run


def scan(angles, nu, du=0.8, lsd=1000.0, lso=500.0, drho=None):
    out = []
    for k, b in enumerate(angles):
        c, s = np.cos(b), np.sin(b)
        r = -lso + (0.0 if drho is None else drho[k])
        p = np.array([r * c, r * s])
        pu = du * np.array([-s, c])
        e0 = (lsd - lso) * np.array([c, s]) - 0.5 * nu * pu - p
        out.append([*p, *e0, *pu])
    return out


def turn(n, start=0.0):
    return start + 2 * np.pi * np.arange(n) / n


def apply(op, x, y):
    a, b = (y, x) if op & 1 else (x, y)
    return (-a if op & 2 else a), (-b if op & 4 else b)


def pixel(op, nx, ny, x, y):
    a, b = (y, x) if op & 1 else (x, y)
    return (nx - 1 - a if op & 2 else a), (ny - 1 - b if op & 4 else b)


CASES = [
    # nx, ny, nu, angles, drho, allowed, most, symmetries
    (33, 33, 50, turn(60), None, 0xff, 8, 8),
    (48, 48, 64, turn(60), None, 0xff, 4, 4),
    (48, 48, 64, turn(60), None, 0xff, 2, 2),
    (40, 24, 64, turn(60), None, 0x55, 8, 4),
    (32, 32, 64, turn(30), None, 0xff, 8, 4),
    (20, 31, 64, turn(31), None, 0x55, 8, 2),
    (32, 32, 64, turn(60, 0.37), None, 0xff, 8, 4),
    (32, 32, 64, turn(31, 0.37), None, 0xff, 8, 1),
    (32, 32, 64, turn(60), 0.6 * (-1.0) ** np.arange(60), 0xff, 8, 4),   # the mirrored diagonals swap the spots
    (32, 32, 64, turn(60), np.linspace(-1, 1, 60), 0xff, 8, 1),
    (32, 32, 64, np.linspace(0, 2 * np.pi, 61), None, 0xff, 8, None),    # first view again at the end
    (32, 32, 64, turn(60) + 1e-7 * np.sin(np.arange(60)), None, 0xff, 8, 1),
    (17, 17, 64, turn(60), None, 0x1, 8, 1),
    (1, 1, 8, turn(4), None, 0xff, 8, 8),
    (16, 16, 3, turn(4, np.pi / 4), None, 0xff, 8, 8),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_symmetry_tables(tables, case):
    nx, ny, nu, ang, drho, allowed, most, want = CASES[case]
    views = np.array(scan(ang, nu, drho=drho))
    op, rep, rep_view, view, tile, owner = tables(nx, ny, nu, views, allowed, most)
    nh, n_p = len(op), len(views)
    if want is not None:
        assert nh == want, (nh, op)
    assert op[0] == 0 and nh <= most and all((allowed >> o) & 1 for o in op)
    if nh == 1:
        return
    view = view.reshape(n_p, nh)
    for h, o in enumerate(op):
        assert sorted(view[:, h]) == list(range(n_p))
        rev = (o ^ (o >> 1) ^ (o >> 2)) & 1
        for v in range(n_p):
            w = views[view[v, h]]
            assert np.allclose(apply(o, *views[v][:2]), w[:2], atol=1e-8, rtol=0)
            for k in range(0, nu + 1, max(1, nu // 5)):  # edge k -> edge k, or nu - k mirrored
                e = views[v][2:4] + k * views[v][4:6]
                assert np.allclose(apply(o, *e), w[2:4] + (nu - k if rev else k) * w[4:6], atol=1e-7, rtol=0)
    rep_view = rep_view.reshape(len(rep), nh)
    assert sorted(rep_view[rep_view >= 0]) == list(range(n_p))
    for r, row in zip(rep, rep_view):
        assert row[0] == r and all(x in (-1, view[r, h]) for h, x in enumerate(row))
    hits = np.zeros((ny, nx), int)
    owner = owner.reshape(len(tile), 16, 16)
    for t, m in zip(tile, owner):
        for j, i in zip(*np.nonzero(m)):
            x, y = (t & 0xffff) * 16 + i, (t >> 16) * 16 + j
            assert x < nx and y < ny
            for h, o in enumerate(op):
                if (m[j, i] >> h) & 1:
                    qx, qy = pixel(o, nx, ny, x, y)
                    hits[qy, qx] += 1
    assert (hits == 1).all()
