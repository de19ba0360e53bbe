// symmetry.hpp -- host code that finds the symmetries of a scan (group2d.hpp)
// and lays out the tables its kernels read.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <utility>
#include <vector>

#include "group2d.hpp"

namespace sgdct {

struct SymTables {
  std::vector<int> op{0};           // symmetries, the identity first
  std::vector<int> rep, rep_view;   // [nrep], [nrep][nh]
  std::vector<int> view;            // [np][nh]
  std::vector<int> tile;            // tiles of the fundamental domain
  std::vector<unsigned char> owner; // [ntile][edge * edge], edge = kTile unless asked otherwise
  int nh() const { return (int)op.size(); }
};

// Bins that hold the projection of every pixel tile's box in every view,
// +-1 margin.  Tile (0, 0)'s box has its centre (cx, cy) from pixel (0, 0) and
// half extents (hx, hy), the other tiles' lie kTile pixels apart.  A point d
// away from a box's centre projects to kc - (d . G) / (beta + d . grad beta), G
// = grad N_0 + kc grad beta, kc the centre's projection.  Over the image, kc is
// extreme at the corner tiles (a projective map), |G| at extreme kc, and beta,
// affine, at the corners; so four tiles per view bound every window.
inline int window_bound(const Proj2DArgs& g, const ViewGeo* views, double cx, double cy, double hx, double hy) {
  const int tx = (g.nx + kTile - 1) / kTile, ty = (g.ny + kTile - 1) / kTile;
  int w = 0;
  for (int v = 0; v < g.np; ++v) {
    const ViewGeo& vg = views[v];
    double top = 0.0, room = 1e300;
    for (int c = 0; c < 4; ++c) {
      const double wx = ((c & 1) ? (tx - 1) * kTile : 0) * g.dx + cx + vg.w0x;
      const double wy = ((c & 2) ? (ty - 1) * kTile : 0) * g.dy + cy + vg.w0y;
      const double be = vg.pux * wy - vg.puy * wx;  // < 0 in front of the source
      const double kc = -(vg.e0x * wy - vg.e0y * wx) / be;
      top = std::max(top, hx * std::fabs(vg.e0y + kc * vg.puy) + hy * std::fabs(vg.e0x + kc * vg.pux));
      room = std::min(room, -be - (hx * std::fabs(vg.puy) + hy * std::fabs(vg.pux)));
    }
    // floor(kc + hw) - floor(kc - hw) <= 2 hw + 1, the window's margins 2 more
    const double n = room > 0.0 ? std::floor(2.0 * top / room) + 4.0 : 1e9;
    w = n < g.nu ? std::max(w, (int)n) : g.nu;
  }
  return w;
}

// Views per symmetry op: perm[v] is the view op maps v onto, empty if some
// view has no partner.  Source, first edge ray (`edges`) and detector step have
// to agree within tol (the FP64 rounding of the angles); every view is the
// partner of exactly one.
inline std::vector<int> view_permutation(const std::vector<ViewGeo>& views, int nu, int op, double tol, bool edges) {
  const int np = (int)views.size();
  std::vector<std::pair<double, int>> by_angle(np);
  for (int v = 0; v < np; ++v) by_angle[v] = {std::atan2(views[v].py, views[v].px), v};
  std::sort(by_angle.begin(), by_angle.end());
  std::vector<char> used(np, 0);
  std::vector<int> perm(np, -1);
  const double kPi = 3.14159265358979323846;
  for (int v = 0; v < np; ++v) {
    const ViewGeo& a = views[v];
    const bool rev = SymOp::reverses(op);
    double p[2], e[2], d[2];
    SymOp::point(op, a.px, a.py, &p[0], &p[1]);
    SymOp::point(op, a.e0x + (rev ? nu * a.pux : 0.0), a.e0y + (rev ? nu * a.puy : 0.0), &e[0], &e[1]);
    SymOp::point(op, a.pux, a.puy, &d[0], &d[1]);
    if (rev) d[0] = -d[0], d[1] = -d[1];
    const double th = std::atan2(p[1], p[0]), eps = 1e-9;
    for (int turn = -1; turn <= 1 && perm[v] < 0; ++turn) {
      const double t = th + 2 * kPi * turn;
      auto it = std::lower_bound(by_angle.begin(), by_angle.end(), std::make_pair(t - eps, -1));
      for (; it != by_angle.end() && it->first <= t + eps && perm[v] < 0; ++it) {
        const ViewGeo& b = views[it->second];
        double err = std::max({std::fabs(b.px - p[0]), std::fabs(b.py - p[1]), nu * std::fabs(b.pux - d[0]),
                               nu * std::fabs(b.puy - d[1])});
        if (edges) err = std::max({err, std::fabs(b.e0x - e[0]), std::fabs(b.e0y - e[1])});
        if (!used[it->second] && err <= tol) {
          used[it->second] = 1;
          perm[v] = it->second;
        }
      }
    }
    if (perm[v] < 0) return {};
  }
  return perm;
}

// The symmetries of a scan of nx x ny pixels, at most `most` of them: the
// group of every grid symmetry that permutes the views, or its subgroup
// without axis swaps, or that subgroup's first element of order two.
// `allowed` has a bit for each op the grid admits; hex: a hexagonal lattice;
// edges = false: the detector's bins need not map onto each other; edge: tile
// edge of the fundamental domain.
inline SymTables find_symmetries(const std::vector<ViewGeo>& views, int nx, int ny, int nu, unsigned allowed, int most,
                                 double tol, bool hex = false, bool edges = true, int edge = kTile) {
  SymTables t;
  const int np = (int)views.size();
  std::vector<int> perm[kMaxSym];
  std::vector<int> found{0};
  for (int op = 1; op < kMaxSym && most > 1; ++op) {
    if (!((allowed >> op) & 1)) continue;
    perm[op] = view_permutation(views, nu, op, tol, edges);
    if (!perm[op].empty()) found.push_back(op);
  }
  if ((int)found.size() > most) {
    std::vector<int> plain;
    for (int op : found)
      if (!(op & SymOp::kSwap)) plain.push_back(op);
    found = plain;
  }
  if ((int)found.size() > most) found.resize(most >= 2 ? 2 : 1);
  const int nh = (int)found.size();
  if (nh != 2 && nh != 4 && nh != 8) return t;
  t.op = found;
  perm[0].resize(np);
  for (int v = 0; v < np; ++v) perm[0][v] = v;
  t.view.resize((size_t)np * nh);
  for (int v = 0; v < np; ++v)
    for (int h = 0; h < nh; ++h) t.view[(size_t)v * nh + h] = perm[found[h]][v];
  // classes of views, each represented by the member whose source is nearest
  // the y axis (its rays walk image rows)
  std::vector<char> done(np, 0);
  for (int v = 0; v < np; ++v) {
    if (done[v]) continue;
    int r = v;
    for (int h = 1; h < nh; ++h) {
      const int w = t.view[(size_t)v * nh + h];
      if (std::fabs(views[w].py) > std::fabs(views[r].py) * (1.0 + 1e-9)) r = w;
    }
    t.rep.push_back(r);
    for (int h = 0; h < nh; ++h) {
      const int w = t.view[(size_t)r * nh + h];
      t.rep_view.push_back(done[w] ? -1 : w);
      done[w] = 1;
    }
  }
  // tiles in raster order until every pixel is the image of a tile's pixel;
  // the first pair (pixel, op) that reaches a pixel writes it
  std::vector<char> covered((size_t)nx * ny, 0);
  const int tx = (nx + edge - 1) / edge, ty = (ny + edge - 1) / edge;
  for (int j = 0; j < ty; ++j)
    for (int i = 0; i < tx; ++i) {
      const int x1 = std::min(nx, (i + 1) * edge), y1 = std::min(ny, (j + 1) * edge);
      bool need = false;
      for (int y = j * edge; y < y1 && !need; ++y)
        for (int x = i * edge; x < x1 && !need; ++x) need = !covered[(size_t)y * nx + x];
      if (!need) continue;
      t.tile.push_back(j << 16 | i);
      const size_t o = t.owner.size();
      t.owner.resize(o + edge * edge, 0);
      for (int y = j * edge; y < y1; ++y)
        for (int x = i * edge; x < x1; ++x)
          for (int h = 0; h < nh; ++h) {
            int qx, qy;
            if (hex) SymOp::hex_point(found[h], nx, ny, x, y, &qx, &qy);
            else SymOp::pixel(found[h], nx, ny, x, y, &qx, &qy);
            char& c = covered[(size_t)qy * nx + qx];
            if (c) continue;
            c = 1;
            t.owner[o + (size_t)(y - j * edge) * edge + (x - i * edge)] |= (unsigned char)(1 << h);
          }
    }
  return t;
}

}  // namespace sgdct
