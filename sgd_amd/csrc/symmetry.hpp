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

// No window holds a tile's bins (window_bound).
constexpr int kNoWindow = 1 << 30;

// Bins that hold the projection of every pixel tile's box in every view,
// +-1 margin; kNoWindow where some box does not lie in front of some view's
// source: a box that the plane beta = 0 through the source cuts projects to
// both ends of the detector, whatever its corners do.  Tile (0, 0)'s box has its centre (cx, cy) from pixel (0, 0) and
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
    if (!(room > 0.0)) return kNoWindow;
    // floor(kc + hw) - floor(kc - hw) <= 2 hw + 1, the window's margins 2 more
    const double n = std::floor(2.0 * top / room) + 4.0;
    w = n < g.nu ? std::max(w, (int)n) : g.nu;
  }
  return w;
}

// The op that applies a after b.
inline int compose(int a, int b) {
  double x, y;
  SymOp::point(b, 1.0, 2.0, &x, &y);
  SymOp::point(a, x, y, &x, &y);
  const int swap = std::fabs(x) == 2.0 ? SymOp::kSwap : 0;
  return swap | (x < 0.0 ? SymOp::kFlipX : 0) | (y < 0.0 ? SymOp::kFlipY : 0);
}

// The views of a scan by where they are: a scan of several turns holds views
// that coincide up to the rounding of their angles.  Places are found by their
// first view; source, first edge ray (`edges`) and detector step have to agree
// within tol (the FP64 rounding of the angles).
struct ViewPlaces {
  static constexpr double kAngle = 1e-9;
  const std::vector<ViewGeo>& views;
  int nu;
  double tol;
  bool edges;
  std::vector<std::vector<int>> at;              // views of a place, ascending
  std::vector<std::pair<double, int>> by_angle;  // (source angle, place), sorted

  ViewPlaces(const std::vector<ViewGeo>& views_, int nu_, double tol_, bool edges_)
      : views(views_), nu(nu_), tol(tol_), edges(edges_) {
    const int np = (int)views.size();
    std::vector<std::pair<double, int>> all(np);
    for (int v = 0; v < np; ++v) all[v] = {std::atan2(views[v].py, views[v].px), v};
    std::sort(all.begin(), all.end());
    for (const auto& a : all) {
      // places are added by ascending angle, so by_angle is sorted throughout
      const int k = find(0, views[a.second]);
      if (k >= 0) {
        at[k].push_back(a.second);
      } else {
        by_angle.push_back({a.first, (int)at.size()});
        at.push_back({a.second});
      }
    }
    for (auto& p : at) std::sort(p.begin(), p.end());
  }

  // The place that op maps view a onto, -1 if there is none.
  int find(int op, const ViewGeo& a) const {
    const bool rev = SymOp::reverses(op);
    const double kPi = 3.14159265358979323846;
    double p[2], e[2], d[2];
    SymOp::point(op, a.px, a.py, &p[0], &p[1]);
    SymOp::point(op, a.e0x + (rev ? nu * a.pux : 0.0), a.e0y + (rev ? nu * a.puy : 0.0), &e[0], &e[1]);
    SymOp::point(op, a.pux, a.puy, &d[0], &d[1]);
    if (rev) d[0] = -d[0], d[1] = -d[1];
    const double th = std::atan2(p[1], p[0]);
    for (int turn = -1; turn <= 1; ++turn) {
      const double t = th + 2 * kPi * turn;
      auto it = std::lower_bound(by_angle.begin(), by_angle.end(), std::make_pair(t - kAngle, -1));
      for (; it != by_angle.end() && it->first <= t + kAngle; ++it) {
        const ViewGeo& b = views[at[it->second][0]];
        double err = std::max({std::fabs(b.px - p[0]), std::fabs(b.py - p[1]), nu * std::fabs(b.pux - d[0]),
                               nu * std::fabs(b.puy - d[1])});
        if (edges) err = std::max({err, std::fabs(b.e0x - e[0]), std::fabs(b.e0y - e[1])});
        if (err <= tol) return it->second;
      }
    }
    return -1;
  }

  // perm[v] is the view op maps v onto, the k-th view of a place onto the k-th
  // of its image, so that the permutations of several ops compose as the ops
  // do; empty if a place has no image with as many views.
  std::vector<int> permutation(int op) const {
    std::vector<int> perm(views.size(), -1);
    for (const auto& from : at) {
      const int k = find(op, views[from[0]]);
      if (k < 0 || at[k].size() != from.size()) return {};
      for (size_t i = 0; i < from.size(); ++i) perm[from[i]] = at[k][i];
    }
    return perm;
  }
};

// Whether perm[] acts on the views as the ops `found` do on the grid: closed
// under composition, every op a permutation, and perm[a after b] = perm[a]
// after perm[b].  The orbits that the tables are made of are then classes.
inline bool acts_as_group(const std::vector<int>& found, const std::vector<int>* perm) {
  for (int a : found) {
    std::vector<char> hit(perm[a].size(), 0);
    for (int w : perm[a]) {
      if (w < 0 || w >= (int)hit.size() || hit[w]) return false;
      hit[w] = 1;
    }
    for (int b : found) {
      const int ab = compose(a, b);
      if (std::find(found.begin(), found.end(), ab) == found.end()) return false;
      for (size_t v = 0; v < hit.size(); ++v)
        if (perm[a][perm[b][v]] != perm[ab][v]) return false;
    }
  }
  return true;
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
  if (most <= 1) return t;
  for (const ViewGeo& v : views)  // angles that are no numbers have no order
    if (!std::isfinite(v.px + v.py + v.e0x + v.e0y + v.pux + v.puy)) return t;
  const ViewPlaces places(views, nu, tol, edges);
  std::vector<int> perm[kMaxSym];
  std::vector<int> found{0};
  for (int op = 1; op < kMaxSym; ++op) {
    if (!((allowed >> op) & 1)) continue;
    perm[op] = places.permutation(op);
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
  perm[0].resize(np);
  for (int v = 0; v < np; ++v) perm[0][v] = v;
  if (!acts_as_group(found, perm)) return t;
  t.op = found;
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

// For every view in its class's slot s (rep_view order, -1 where a class repeats
// a view) and every symmetry k, the slot of view k v counted from the class's
// first: peer[s * nh + k] (0 in a repeated slot, which nothing reads).  False if
// some class does not hold the views its members map onto.
inline bool class_peers(const SymTables& t, std::vector<int>* peer) {
  const int nh = t.nh(), ns = (int)t.rep_view.size();
  peer->assign((size_t)ns * nh, 0);
  for (int s = 0; s < ns; ++s) {
    if (t.rep_view[s] < 0) continue;
    const auto cls = t.rep_view.begin() + s / nh * nh;
    for (int k = 0; k < nh; ++k) {
      const auto q = std::find(cls, cls + nh, t.view[(size_t)t.rep_view[s] * nh + k]);
      if (q == cls + nh) return false;
      (*peer)[(size_t)s * nh + k] = (int)(q - cls);
    }
  }
  return true;
}

}  // namespace sgdct
