// hex2d.hip -- hexagonal-lattice projectors (H0, Hl), gfx950.
//
// Lattice point (ic, il): row il at y = (il - (nl-1)/2) dyh, column ic at
// x = (ic + (il odd ? 1/2 : 0) - (nc-1)/2) dxh, dxh = sqrt(3) dt; odd rows hold
// nc-1 points (layers/A_H0.cu:172-183, A_Hl.cu:171-182).
//   H0: hexagon indicator (circumradius dt, dyh = 1.5 dt) = three rhombi; the
//       value is the bin average of the sum of the three rhombus projections
//       (box splines of two of va, vb, vc each, A_H0.cu:229-245), divided by 3
//       so that it is the hexagon's projection (the reference omits the 1/3);
//       evaluated as the hexagon's own chord length (s_h0).
//   Hl: three-direction box spline (dyh = dt/2), bin average of
//       box_|va| * box_|vb| * box_|vc| (A_Hl.cu:226-236).
// va, vb, vc = dt sin(theta + 2 pi k / 3), theta the bin's central-ray angle
// atan2(dx, dy) (A_H0.cu:229-232).  Bin ranges come from the six true hexagon
// vertices: the reference's H0 culling uses the Hl row pitch and drops
// off-centre rows (A_H0.cu:82-156 with h0_init's dy = dt/2).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "footprint.hpp"
#include "group2d_dev.hpp"
#include "projector.hpp"
#include "symmetry.hpp"

namespace sgdct {

hipError_t launch_sum_parts(const double* part, float* out, size_t n, int nparts, hipStream_t s);

// H0: the hexagon's vertices project to +-a, +-b, +-c (a = b + c, the lengths
// of its edges' projections), between which its chord length is linear.
struct H0Bin {
  float ka, kb, a, b;
  float c, d, k1, k2;    // d = b - c, 1 / (6 b c), 1 / (3 b)
  float k3, k4, pad[2];  // 1 / (6 a b), 2 / (3 a)
};

// Antiderivative of the projection of a hexagon of unit area, odd in t: the
// mean of three rhombi box_b * box_c, box_a * box_b and box_a * box_c about
// a / 2, -c / 2 and -b / 2 (layers/A_H0.cu:229-248), whose sum over the tail
// x = |t| is one quadratic per interval between vertices:
//   1/2 - S(x) = u^2 / (6 b c) + v / (3 b) + v^2 / (6 a b) + 2 w / (3 a)
// with the depths u, v, w of x into [b, a], [c, b] and [0, c].
__device__ __forceinline__ float s_h0(float t, const H0Bin& r) {
  const float x = __builtin_fabsf(t);
  const float u = __builtin_amdgcn_fmed3f(r.a - x, 0.0f, r.c);
  const float v = __builtin_amdgcn_fmed3f(r.b - x, 0.0f, r.d);
  const float w = __builtin_fmaxf(r.c - x, 0.0f);
  const float tail = __builtin_fmaf(u, u * r.k1, __builtin_fmaf(v, __builtin_fmaf(v, r.k3, r.k2), w * r.k4));
  return copysign_f(0.5f - tail, t);
}

// Hl: widths p >= q >= r (p = q + r) of box_p * box_q * box_r.
struct HlBin {
  float ka, kb, p, q, r, inv6pq, inv_r, pad;
};

// Antiderivative of box_p * box_q * box_r (p = q + r), odd in t:
//   S(x) = 1/2 - [(p-x)_+^3 - (q-x)_+^3 - (r-x)_+^3] / (6pqr),   x = |t|,
// written without the cancellations of the difference of cubes:
//   x <= q :  1/2 - (A^2 + AB + B^2)/(6pq) + C^2 (C/r)/(6pq)
//   x >  q :  1/2 - A^2 (A/r)/(6pq)
// with A = (p-x)_+, B = (q-x)_+, C = (r-x)_+  (A - B = r when x <= q).
__device__ __forceinline__ float s_hl(float t, const HlBin& r) {
  const float x = __builtin_fabsf(t);
  const float A = __builtin_fmaxf(r.p - x, 0.0f);
  const float B = __builtin_fmaxf(r.q - x, 0.0f);
  const float C = __builtin_fmaxf(r.r - x, 0.0f);
  const float a2 = A * A;
  const float v1 = (__builtin_fmaf(A, B, a2) + B * B) - C * C * (C * r.inv_r);
  const float v2 = a2 * (A * r.inv_r);
  const float v = ((x <= r.q) ? v1 : v2) * r.inv6pq;
  return copysign_f(0.5f - v, t);
}

template <int HB> struct HexTraits;

template <> struct HexTraits<BASIS_H0> {
  using Bin = H0Bin;
  __device__ static __forceinline__ float conv(const Bin& r, float ta, float tb) {
    const float cv = (s_h0(tb, r) - s_h0(ta, r)) * __builtin_amdgcn_rcpf(tb - ta);
    return cv > 0.0f ? cv : 0.0f;  // conv > 0 (layers/A_H0.cu:248)
  }
};

template <> struct HexTraits<BASIS_HL> {
  using Bin = HlBin;
  __device__ static __forceinline__ float conv(const Bin& r, float ta, float tb) {
    const float cv = (s_hl(tb, r) - s_hl(ta, r)) * __builtin_amdgcn_rcpf(tb - ta);
    return cv > 0.0f ? cv : 0.0f;  // conv > 0 (layers/A_Hl.cu:238)
  }
};

// max over the six vertices of a pointy-top hexagon of circumradius dt of
// (vertex offset) . (gx, gy)
__device__ __forceinline__ double hex_reach(double gx, double gy, double dt) {
  return dt * fmax(fabs(gy), 0.8660254037844386 * fabs(gx) + 0.5 * fabs(gy));
}

__device__ __forceinline__ float hex_reach_f(float gx, float gy, float dt) {
  return dt * fmaxf(__builtin_fabsf(gy), __builtin_fmaf(0.8660254f, __builtin_fabsf(gx), 0.5f * __builtin_fabsf(gy)));
}

struct HexArgs {
  Proj2DArgs g;  // nx = nc, ny = nl, dx = dxh, dy = dyh
  double dt;
};

// The G values of a lattice point.
template <int G>
__device__ __forceinline__ void load_point(const float* p, float (&x)[G]) {
  __builtin_memcpy(x, __builtin_assume_aligned(p, G < 4 ? 4 * G : 16), sizeof(x));
}

// A: bin-driven gather along lattice rows, or along the vertical lines k = 2 ic
// + (il & 1) (x = k dx / 2, every other row) when the wave's middle ray gives a
// strip more points per vertical line (|ray_y| dx > 2 dy |ray_x|): steep strips
// cross every row with only a point or two in each.  The choice is uniform
// over the wave.
// One wave: bins [64 chunk, 64 chunk + 64) of view v, one per lane; of every
// line's points the w-th of wn equal ranges of columns (row walk) or rows
// (vertical walk), of the lines segment seg of nseg.  Adds sum conv * x into
// acc[G] (FP32 along a line, FP64 across lines; without dx dy).  img holds G
// values per point; at G = 1, point p's value is img's at `place` p.  Lanes past
// the last bin add nothing.
// The strips lie along the lines, so splitting the points keeps every lane of
// every wave busy, where splitting the lines would leave a lane only the few
// it crosses; and a wave's lanes stay within one narrow range of columns or
// rows at a time, which keeps the lines they touch in the vector L1 (walking
// the whole lattice, near-row strips needed their rows staged in LDS for
// that).
template <int HB, int G, bool FAR>
__device__ __forceinline__ void hex_fwd_lines(const HexArgs& ha, int v, int chunk, const float* __restrict__ img, int w,
                                              int wn, int seg, int nseg, double (&acc)[G],
                                              int place = 0) {
  using T = HexTraits<HB>;
  const bool flip_x = G == 1 && (place & SymOp::kFlipX), flip_y = G == 1 && (place & SymOp::kFlipY);
  const Proj2DArgs& g = ha.g;
  const bool inside = chunk * 64 + (int)(threadIdx.x & 63) < g.nu;
  const int u = inside ? chunk * 64 + (int)(threadIdx.x & 63) : g.nu - 1;
  const ViewGeo vg = g.views[v];
  const typename T::Bin rec = reinterpret_cast<const typename T::Bin*>(g.bins)[(size_t)v * g.nu + u];

  const double eax = vg.e0x + u * vg.pux, eay = vg.e0y + u * vg.puy;
  const double ebx = eax + vg.pux, eby = eay + vg.puy;
  // N(ic', il) = s * ic' + m * il + c, ic' = ic + (il odd) / 2
  const double sa = -eay * g.dx, ma = eax * g.dy, ca = eax * vg.w0y - eay * vg.w0x;
  const double sb = -eby * g.dx, mb = ebx * g.dy, cb = ebx * vg.w0y - eby * vg.w0x;
  // pixel-set edges (clamped end bins see one more bin), as in fwd_bin_lines
  const double lax = (u == 0) ? eax - vg.pux : eax, lay = (u == 0) ? eay - vg.puy : eay;
  const double lbx = (u == g.nu - 1) ? ebx + vg.pux : ebx, lby = (u == g.nu - 1) ? eby + vg.puy : eby;
  const double sq = -lay * g.dx, mq = lax * g.dy, cq = lax * vg.w0y - lay * vg.w0x;
  const double sr = -lby * g.dx, mr = lbx * g.dy, cr = lbx * vg.w0y - lby * vg.w0x;
  // points that touch a strip's edge belong to it on either side: a hexagon's
  // footprint is not zero there (its model widens it by the bin's angle), and
  // lattices have whole columns of such points in the views along their axes,
  // which rounding would otherwise share out (H0, 1501 x 3 points, a view
  // along the columns: relative error 1.2e-5 without, 8e-6 with)
  constexpr double kTouch = 1.0 + 1e-10;
  const double rq = kTouch * hex_reach(-lay, lax, ha.dt), rr = kTouch * hex_reach(-lby, lbx, ha.dt);
  const double ka = rec.ka, kb = rec.kb;

  // Point values by 32-bit byte offsets into a buffer resource, or by address,
  // clamped to the last point: for a lattice of 4 GiB and more (FAR), and for 8
  // values, whose two 16-byte loads the vector L1 serves faster so (Hl, batch
  // 64: 7.07 ms against 7.92).
  using Off = std::conditional_t<FAR, size_t, unsigned>;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(img), (short)0, (int)(4u * G * (unsigned)g.nx * (unsigned)g.ny), 0x00020000);
  const Off last_point = 4 * (Off)G * ((Off)g.nx * g.ny - 1);
  auto fetch = [&](Off off, float (&x)[G]) {
    if constexpr (FAR || G == 8)
      load_point<G>(reinterpret_cast<const float*>(reinterpret_cast<const char*>(img) + min(off, last_point)), x);
    else
      buffer_load_n<G>(rsrc, off, x);
  };
  // One line: n points `step` bytes apart from `off`.
  auto walk = [&](Off off, int n, Off step, float ta, float tb, float dta, float dtb) {
    float accl[G], xn[G];
#pragma unroll
    for (int s = 0; s < G; ++s) accl[s] = 0.0f;
    // the next point's values are requested one step ahead, which overlaps
    // their latency with the footprint evaluation
    fetch(off, xn);
    const Off end = off + (Off)n * step;
    do {
      float xc[G];
#pragma unroll
      for (int s = 0; s < G; ++s) xc[s] = xn[s];
      off += step;
      fetch(off, xn);
      const float c = T::conv(rec, ta, tb);
#pragma unroll
      for (int s = 0; s < G; ++s) accl[s] = __builtin_fmaf(c, xc[s], accl[s]);
      ta += dta;
      tb += dtb;
    } while (off != end);
#pragma unroll
    for (int s = 0; s < G; ++s) acc[s] += (double)accl[s];
  };
  // Points n of line l in the strip, from q: N_q + R_q >= 0 and r: N_r - R_r <
  // 0 with N = slope n + cross l + c.
  StripLines lines;

  const int umid = min(chunk * 64 + 32, g.nu - 1);
  const double rmx = vg.e0x + (umid + 0.5) * vg.pux, rmy = vg.e0y + (umid + 0.5) * vg.puy;
  if (fabs(rmy) * g.dx <= 2.0 * g.dy * fabs(rmx)) {
    const int c_lo = g.nx * w / wn, c_hi = g.nx * (w + 1) / wn - 1;
    // rows the strip can reach within the columns (ic' = ic + 1/2 on odd rows)
    int il_lo, il_hi;
    strip_lines(sq, mq, -rq - cq, sr, mr, rr - cr, (double)c_lo, (double)(c_hi + 1), g.ny, &il_lo, &il_hi);
    if (nseg > 1) {
      const int len = (g.ny + nseg - 1) / nseg;
      il_lo = max(il_lo, seg * len);
      il_hi = min(il_hi, seg * len + len - 1);
    }
    if (!inside) il_hi = -1;
    lines.set(sq, mq, -rq - cq, sr, mr, rr - cr, (float)g.ny);
    const double kas = ka * sa, kam = ka * ma, kac = ka * ca, kbs = kb * sb, kbm = kb * mb, kbc = kb * cb;
    const float dta = (float)kas, dtb = (float)kbs;
    const float fc_lo = (float)c_lo, fc_hi = (float)c_hi, fc_odd = (float)min(c_hi, g.nx - 2);
    const Off step = flip_x ? -(Off)(4 * G) : (Off)(4 * G);
    for (int il = il_lo; il <= il_hi; ++il) {
      const bool odd = il & 1;  // points half a column to the right
      const float sh = odd ? 0.5f : 0.0f;
      float flo, fhi;
      if (!lines.at((float)il, sh, &flo, &fhi))
        lines.settle(sq, -rq - __builtin_fma(mq, (double)il, cq) - sq * sh, sr,
                     rr - __builtin_fma(mr, (double)il, cr) - sr * sh, (double)(g.nx - 1), &flo, &fhi);
      flo = fmaxf(ceilf(flo), fc_lo);
      fhi = fminf(floorf(fhi), odd ? fc_odd : fc_hi);
      if (!(flo <= fhi)) continue;
      const int n0 = (int)flo;
      const double dn = (double)(flo + sh), dl = (double)il;
      const int qx = flip_x ? g.nx - (il & 1) - 1 - n0 : n0, qy = flip_y ? g.ny - 1 - il : il;
      walk(4 * G * ((Off)qy * g.nx + qx), (int)fhi - n0 + 1, step,
           (float)__builtin_fma(kas, dn, __builtin_fma(kam, dl, kac)),
           (float)__builtin_fma(kbs, dn, __builtin_fma(kbm, dl, kbc)), dta, dtb);
    }
  } else {
    const int r_lo = g.ny * w / wn, r_hi = g.ny * (w + 1) / wn - 1;
    // vertical lines the strip can reach within the rows
    const int kmax = 2 * g.nx - 2;
    int k_lo, k_hi;
    strip_lines(mq, 0.5 * sq, -rq - cq, mr, 0.5 * sr, rr - cr, (double)r_lo, (double)r_hi, kmax + 1, &k_lo, &k_hi);
    if (nseg > 1) {
      const int len = (kmax + nseg) / nseg;
      k_lo = max(k_lo, seg * len);
      k_hi = min(k_hi, seg * len + len - 1);
    }
    if (!inside) k_hi = -1;
    lines.set(mq, 0.5 * sq, -rq - cq, mr, 0.5 * sr, rr - cr, (float)(kmax + 1));
    const double kam = ka * ma, kas = 0.5 * ka * sa, kac = ka * ca, kbm = kb * mb, kbs = 0.5 * kb * sb, kbc = kb * cb;
    const float dta = (float)(2.0 * kam), dtb = (float)(2.0 * kbm);
    const float fr_lo = (float)r_lo, fr_hi = (float)r_hi;
    const Off step = flip_y ? -(8 * G * (Off)g.nx) : 8 * G * (Off)g.nx;
    for (int k = k_lo; k <= k_hi; ++k) {  // ic' = k / 2
      float flo, fhi;
      if (!lines.at((float)k, 0.0f, &flo, &fhi))
        lines.settle(mq, -rq - cq - sq * (0.5 * k), mr, rr - cr - sr * (0.5 * k), (double)(g.ny - 1), &flo, &fhi);
      flo = fmaxf(ceilf(flo), fr_lo);
      fhi = fminf(floorf(fhi), fr_hi);
      if (!(flo <= fhi)) continue;
      int i0 = (int)flo, i1 = (int)fhi;
      i0 += (i0 ^ k) & 1;  // rows of the line's parity
      i1 -= (i1 ^ k) & 1;
      if (i0 > i1) continue;
      const double dk = (double)k, di = (double)i0;
      const int qx = flip_x ? g.nx - (k & 1) - 1 - (k >> 1) : k >> 1, qy = flip_y ? g.ny - 1 - i0 : i0;
      walk(4 * G * ((Off)qy * g.nx + qx), ((i1 - i0) >> 1) + 1, step,
           (float)__builtin_fma(kam, di, __builtin_fma(kas, dk, kac)),
           (float)__builtin_fma(kbm, di, __builtin_fma(kbs, dk, kbc)), dta, dtb);
    }
  }
}

// grid (nrep * nchunk, image groups, nseg): W waves take one representative
// view and 64-bin chunk, and their FP64 sums are added in wave order through
// LDS.  Chunk-major: workgroups in flight take the same bins of adjacent views,
// so they walk nearly the same points and reach the lattice together or miss
// it together.  Bound by VALU issue (~45 instructions per footprint, and about
// as many per line and lane) and, at G = 8, by the vector L1.  Per call, one
// value per footprint and one wave per (view, chunk) -> now: H0 256 x 296
// points, 1024 views, 1024 bins 840 -> 315 us (476 with three rhombi's six
// antiderivatives and FP64 divisions for every line); Hl, batch 64 30.8 -> 7.0
// ms; Hl 40 x 46, 60 views, batch 3 76 -> 18 us, 3 of them the events that order
// the interleaved points' uses.
template <int HB, int G, int W, bool FAR>
__global__ __launch_bounds__(64 * W) void hex_fwd_kernel(HexArgs ha, SymPlan sp, int m, int batch,
                                                         const float* __restrict__ img, float* __restrict__ sino,
                                                         double* __restrict__ part) {
  __shared__ double red[W][G][64];
  const Proj2DArgs& g = ha.g;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int rank = blockIdx.x / sp.nrep, rep = blockIdx.x - rank * sp.nrep;
  const int chunk = centre_out(rank, g.nchunk);
  const int v = sp.rep ? sp.rep[rep] : rep;
  double acc[G];
#pragma unroll
  for (int s = 0; s < G; ++s) acc[s] = 0.0;
  hex_fwd_lines<HB, G, FAR>(ha, v, chunk, img + (size_t)blockIdx.y * G * g.nx * g.ny, wv, W, blockIdx.z, gridDim.z, acc,
                            sp.place);
#pragma unroll
  for (int s = 0; s < G; ++s) red[wv][s][lane] = acc[s];
  __syncthreads();
  const int u = chunk * 64 + lane;
  if (u >= g.nu) return;
  fwd_group_store<G, W>(g, sp, rep, v, u, m, batch, red, g.dx, g.dy, 1.0, sino, gridDim.z > 1 ? part : nullptr);
}

// Interleaved copies of the lattices of one launch (interleave_kernel on the
// hexagonal lattice: a mirror maps the points of an odd row among its nc - 1).
template <int G>
__global__ __launch_bounds__(256) void hex_interleave_kernel(SymPlan sp, int nx, int ny, int m, int batch,
                                                             const float* __restrict__ img, float* __restrict__ rows) {
  const size_t npix = (size_t)nx * ny;
  const int img0 = blockIdx.z * m, nslot = sp.nh * min(m, batch - img0);
  const int ix = blockIdx.x * 16 + (threadIdx.x & 15), iy = blockIdx.y * 16 + (threadIdx.x >> 4);
  if (ix >= nx || iy >= ny) return;
  float x[G];
#pragma unroll
  for (int s = 0; s < G; ++s) {
    x[s] = 0.0f;
    if (s < nslot) {
      const int k = s >> sp.lg, h = s & (sp.nh - 1);
      int qx, qy;
      SymOp::hex_point(sp.op[h], nx, ny, ix, iy, &qx, &qy);
      x[s] = img[(img0 + k) * npix + (size_t)qy * nx + qx];
    }
  }
  rows += blockIdx.z * npix * G;
  __builtin_memcpy(__builtin_assume_aligned(rows + ((size_t)iy * nx + ix) * G, G < 4 ? 4 * G : 16), x, sizeof(x));
}

// Box that holds the footprints of a 16 x 16 point tile: its centre relative
// to point (0, 0) of the tile and its half extents (one circumradius and the
// half-column shift of odd rows around the points).
__host__ __device__ inline void hex_tile_box(const HexArgs& a, double* cx, double* cy, double* hx, double* hy) {
  *cx = 0.5 * kTile * a.g.dx;
  *cy = 0.5 * (kTile - 1) * a.g.dy;
  *hx = (0.5 * kTile + 0.5) * a.g.dx + a.dt;
  *hy = 0.5 * (kTile + 1) * a.g.dy + a.dt;
}

// A^T in the grouped frame (group2d_dev.hpp).
template <int HB> struct HexBwd {
  using Args = HexArgs;
  using T = HexTraits<HB>;
  using Bin = typename T::Bin;
  static constexpr int kRec = sizeof(Bin) / 16;
  static_assert(sizeof(Bin) % 16 == 0, "bin records are whole float4s");
  struct Pixel {
    double fx, fy;
  };
  __device__ static __forceinline__ const Proj2DArgs& geo(const Args& a) { return a.g; }
  __device__ static __forceinline__ void window(const Args& a, const ViewGeo& vg, int ix0, int iy0, int* lo, int* n,
                                                int cap) {
    double cx, cy, hx, hy, umin = 1e300, umax = -1e300;
    hex_tile_box(a, &cx, &cy, &hx, &hy);
#pragma unroll 1
    for (int c = 0; c < 4; ++c) {
      const double wx = ix0 * a.g.dx + cx + ((c & 1) ? hx : -hx) + vg.w0x;
      const double wy = iy0 * a.g.dy + cy + ((c & 2) ? hy : -hy) + vg.w0y;
      const double uu = -(vg.e0x * wy - vg.e0y * wx) / (vg.pux * wy - vg.puy * wx);
      umin = fmin(umin, uu);
      umax = fmax(umax, uu);
    }
    const int l = (int)fmax(floor(umin) - 1.0, 0.0), h = (int)fmin(floor(umax) + 1.0, (double)(a.g.nu - 1));
    *lo = l;
    *n = h >= l ? min(h - l + 1, cap) : 0;
  }
  __device__ static __forceinline__ Pixel pixel(const Args& a, int ic, int il) {
    return {(ic + ((il & 1) ? 0.5 : 0.0)) * a.g.dx, il * a.g.dy};
  }
  __device__ static __forceinline__ bool active(const Args& a, int ic, int il) {
    return !((il & 1) && ic == a.g.nx - 1);
  }
  __device__ static __forceinline__ void image(const Args& a, int op, int ic, int il, int* qx, int* qy) {
    SymOp::hex_point(op, a.g.nx, a.g.ny, ic, il, qx, qy);
  }
  __device__ static __forceinline__ float value(const float4 (&)[kRec], float y) { return y; }
  __device__ static __forceinline__ double result(const Args& a, double acc) { return acc * a.g.dx * a.g.dy; }

  template <int G>
  __device__ static __forceinline__ void view(const Args& a, const ViewGeo& vg, const Pixel& p,
                                              const Staged<kRec, G>& st, int base, int wlo, int wn, float (&accv)[G]) {
    const double wx = p.fx + vg.w0x, wy = p.fy + vg.w0y;
    const double n0 = vg.e0x * wy - vg.e0y * wx;
    const double be = vg.pux * wy - vg.puy * wx;
    const float bef = (float)be;
    // bin range in FP32 (it only bounds the bins visited; a bin gained or
    // lost at a rounding boundary carries a vanishing footprint)
    const float kc = -(float)n0 * __builtin_amdgcn_rcpf(bef);
    // k*(vertex) - kc = -(d . G) / (beta + d . grad beta), G = grad N_0 + kc grad beta
    const float gx = -__builtin_fmaf(kc, (float)vg.puy, (float)vg.e0y);
    const float gy = __builtin_fmaf(kc, (float)vg.pux, (float)vg.e0x);
    const float dt = (float)a.dt;
    const float hw = hex_reach_f(gx, gy, dt) *
                     __builtin_amdgcn_rcpf(__builtin_fabsf(bef) - hex_reach_f(-(float)vg.puy, (float)vg.pux, dt));
    const float last = (float)(a.g.nu - 1);
    const int ulo = max((int)fminf(fmaxf(floorf(kc - hw), 0.0f), last), wlo);
    const int uhi = min((int)fminf(fmaxf(floorf(kc + hw), 0.0f), last), wlo + wn - 1);
    float na = (float)(n0 + (double)ulo * be);
    for (int u = ulo; u <= uhi; ++u) {
      const int at = base + u - wlo;
      float4 rd[kRec];
      st.record(at, rd);
      const Bin rec = __builtin_bit_cast(Bin, rd);
      const float nb = na + bef;
      st.add(at, T::conv(rec, rec.ka * na, rec.kb * nb), accv);
      na = nb;
    }
  }
};

// Launched as bwd_group_kernel; bound by VALU issue and the LDS reads of the
// records (48 bytes per footprint for H0; 80 with three rhombi, 437 us in the
// first case).  Same cases as hex_fwd_kernel: 728 -> 257 us, 33.2 -> 5.5 ms, 39
// -> 13 us.
template <int HB, int G>
__global__ __launch_bounds__(256) void hex_bwd_group_kernel(HexArgs ha, SymPlan sp, int m, int batch,
                                                            const float* __restrict__ sino, float* __restrict__ img,
                                                            int vpg, int nvc, int win, double* __restrict__ part) {
  bwd_group_block<HexBwd<HB>, G>(ha, sp, m, batch, sino, img, vpg, nvc, win, part);
}

constexpr int kHexH0Window = 72;

// A^T where the tiles' bin windows are too wide for the grouped frame's LDS:
// lattice-point-driven gather, 16 x 16 point tiles, LDS bin windows.
// grid (tiles, tiles, batch * ngroup), H0's blocks mapped by xcd_block: z =
// b * ngroup + k takes views
// [k vpg, (k+1) vpg); with ngroup > 1 it writes its FP64 sum to
// part[(k * batch + b) * nc * nl + point], added in group order afterwards.
template <int HB>
__global__ __launch_bounds__(256) void hex_bwd_kernel(HexArgs ha, const float* __restrict__ sino,
                                                      float* __restrict__ img, int ngroup, int vpg,
                                                      double* __restrict__ part) {
  using T = HexTraits<HB>;
  using Bin = typename T::Bin;
  constexpr int BIN4 = sizeof(Bin) / 16;
  static_assert(sizeof(Bin) % 16 == 0, "bin records are whole float4s");
  // LDS bin window per view: 72 of H0's 48-byte records (14 KB a block; a 16 x
  // 16 H0 tile spans up to ~66 bins at 0.3 mm per bin); bins past the window are
  // read from global memory
  constexpr int kWin = HB == BASIS_H0 ? kHexH0Window : kMaxWindow;
  __shared__ float4 lds[kViewChunk][kWin][BIN4];
  __shared__ float ldsy[kViewChunk][kWin];
  __shared__ int win_lo[kViewChunk], win_n[kViewChunk];
  const Proj2DArgs& g = ha.g;
  // XCD-contiguous blocks (xcd_block) for H0: A^T 0.959 -> 0.939 ms (296 x
  // 256, 1024 views, 1024 bins); Hl was slower with them (0.547 -> 0.562 ms)
  const uint3 blk = HB == BASIS_H0 ? xcd_block() : make_uint3(blockIdx.x, blockIdx.y, blockIdx.z);
  const int ic0 = blk.x * kTile, il0 = blk.y * kTile;
  const int ic = ic0 + (threadIdx.x & (kTile - 1)), il = il0 + threadIdx.x / kTile;
  const int k = blk.z % ngroup, b = blk.z / ngroup, batch = gridDim.z / ngroup;
  const size_t npt = (size_t)g.nx * g.ny;
  sino += (size_t)b * g.np * g.nu;
  img += b * npt;
  const int v_begin = k * vpg, v_end = min(g.np, v_begin + vpg);
  const bool inside = ic < g.nx && il < g.ny;
  const bool valid = inside && !((il & 1) && ic == g.nx - 1);
  const Bin* bins = reinterpret_cast<const Bin*>(g.bins);
  const double sh = (il & 1) ? 0.5 : 0.0;

  double acc = 0.0;
  for (int v0 = v_begin; v0 < v_end; v0 += kViewChunk) {
    const int nv = min(kViewChunk, v_end - v0);
    if ((int)threadIdx.x < nv) {
      // window: the tile's bounding box widened by one circumradius
      const ViewGeo& vg = g.views[v0 + threadIdx.x];
      double umin = 1e300, umax = -1e300;
      for (int c = 0; c < 4; ++c) {
        double fx = (c & 1) ? (ic0 + kTile + 0.5) * g.dx + ha.dt : (ic0 - 0.5) * g.dx - ha.dt;
        double fy = (c & 2) ? (il0 + kTile) * g.dy + ha.dt : (il0 - 1) * g.dy - ha.dt;
        double wx = fx + vg.w0x, wy = fy + vg.w0y;
        double uu = -(vg.e0x * wy - vg.e0y * wx) / (vg.pux * wy - vg.puy * wx);
        umin = fmin(umin, uu);
        umax = fmax(umax, uu);
      }
      int lo = (int)fmax(floor(umin) - 1.0, 0.0), hi = (int)fmin(floor(umax) + 1.0, (double)(g.nu - 1));
      win_lo[threadIdx.x] = lo;
      win_n[threadIdx.x] = hi >= lo ? min(hi - lo + 1, kWin) : 0;
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < nv * kWin; idx += blockDim.x) {
      const int j = idx / kWin, i = idx - j * kWin;
      if (i < win_n[j]) {
        const size_t gi = (size_t)(v0 + j) * g.nu + win_lo[j] + i;
        const float4* src = reinterpret_cast<const float4*>(bins + gi);
#pragma unroll
        for (int k = 0; k < BIN4; ++k) lds[j][i][k] = src[k];
        ldsy[j][i] = sino[gi];
      }
    }
    __syncthreads();
    if (valid) {
      for (int j = 0; j < nv; ++j) {
        const int v = v0 + j;
        const ViewGeo& vg = g.views[v];
        const double wx = (ic + sh) * g.dx + vg.w0x, wy = il * g.dy + vg.w0y;
        const double n0 = vg.e0x * wy - vg.e0y * wx;
        const double be = vg.pux * wy - vg.puy * wx;
        const float bef = (float)be;
        // bin range in FP32 (it only bounds the bins visited; a bin gained or
        // lost at a rounding boundary carries a vanishing footprint)
        const float kc = -(float)n0 * __builtin_amdgcn_rcpf(bef);
        // k*(vertex) - kc = -(d . G) / (beta + d . grad beta), G = grad N_0 + kc grad beta
        const float gx = -__builtin_fmaf(kc, (float)vg.puy, (float)vg.e0y);
        const float gy = __builtin_fmaf(kc, (float)vg.pux, (float)vg.e0x);
        const float dt = (float)ha.dt;
        const float hw = hex_reach_f(gx, gy, dt) *
                         __builtin_amdgcn_rcpf(__builtin_fabsf(bef) - hex_reach_f(-(float)vg.puy, (float)vg.pux, dt));
        const float last = (float)(g.nu - 1);
        const int ulo = (int)fminf(fmaxf(floorf(kc - hw), 0.0f), last);
        const int uhi = (int)fminf(fmaxf(floorf(kc + hw), 0.0f), last);
        float na = (float)(n0 + (double)ulo * be);
        const int wlo = win_lo[j], wn = win_n[j];
        float accv = 0.0f;
        for (int u = ulo; u <= uhi; ++u) {
          const int wi = u - wlo;
          Bin rec;
          float yv;
          if (wi >= 0 && wi < wn) {
            float4* d = reinterpret_cast<float4*>(&rec);
#pragma unroll
            for (int k = 0; k < BIN4; ++k) d[k] = lds[j][wi][k];
            yv = ldsy[j][wi];
          } else {
            rec = bins[(size_t)v * g.nu + u];
            yv = sino[(size_t)v * g.nu + u];
          }
          const float nb = na + bef;
          accv = __builtin_fmaf(T::conv(rec, rec.ka * na, rec.kb * nb), yv, accv);
          na = nb;
        }
        acc += (double)accv;
      }
    }
    __syncthreads();
  }
  if (inside) {
    const double val = valid ? acc * g.dx * g.dy : 0.0;
    if (ngroup > 1) part[(size_t)k * batch * npt + b * npt + (size_t)il * g.nx + ic] = val;
    else img[(size_t)il * g.nx + ic] = (float)val;
  }
}

// Evaluation count (clamped six-vertex ranges).
__global__ __launch_bounds__(256) void hex_count_kernel(HexArgs ha, unsigned long long* out) {
  __shared__ unsigned long long part[256];
  const Proj2DArgs& g = ha.g;
  const int ic = blockIdx.x * 16 + (threadIdx.x & 15), il = blockIdx.y * 16 + (threadIdx.x >> 4);
  unsigned long long c = 0;
  if (ic < g.nx && il < g.ny && !((il & 1) && ic == g.nx - 1)) {
    const double cx = (ic + ((il & 1) ? 0.5 : 0.0)) * g.dx, cy = il * g.dy;
    for (int v = 0; v < g.np; ++v) {
      const ViewGeo& vg = g.views[v];
      double umin = 1e300, umax = -1e300;
      for (int k = 0; k < 6; ++k) {
        const double a = 1.5707963267948966 + k * 1.0471975511965976;
        const double wx = cx + ha.dt * cos(a) + vg.w0x, wy = cy + ha.dt * sin(a) + vg.w0y;
        const double uu = -(vg.e0x * wy - vg.e0y * wx) / (vg.pux * wy - vg.puy * wx);
        umin = fmin(umin, uu);
        umax = fmax(umax, uu);
      }
      const int lo = (int)fmin(fmax(floor(umin), 0.0), (double)(g.nu - 1));
      const int hi = (int)fmin(fmax(floor(umax), 0.0), (double)(g.nu - 1));
      c += (unsigned long long)(hi - lo + 1);
    }
  }
  part[threadIdx.x] = c;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(out, part[0]);
}

// Per-(view, bin) constants (host side, FP64).
void hex_bin_constants(int basis, const ViewGeo& v, int nu, double dt, void* out) {
  for (int u = 0; u < nu; ++u) {
    const double ax = v.e0x + u * v.pux, ay = v.e0y + u * v.puy;
    const double bx = ax + v.pux, by = ay + v.puy;
    const double cx = ax + 0.5 * v.pux, cy = ay + 0.5 * v.puy;
    const double len = std::sqrt(cx * cx + cy * cy);
    const double ka = -len / (ax * cx + ay * cy), kb = -len / (bx * cx + by * cy);
    // central-ray angle, rounded to FP32 like atan2f (layers/A_H0.cu:229)
    const double th = (double)(float)std::atan2(cx, cy);
    double vk[3];
    for (int k = 0; k < 3; ++k) vk[k] = dt * std::sin(th + k * 2.0 * 3.14159265358979323846 / 3.0);
    double w[3] = {std::fabs(vk[0]), std::fabs(vk[1]), std::fabs(vk[2])};
    std::sort(w, w + 3);
    if (basis == BASIS_H0) {
      H0Bin r{};
      r.ka = (float)ka;
      r.kb = (float)kb;
      const double a = w[2], b = w[1], c = w[0];
      r.a = (float)a;
      r.b = (float)b;
      r.c = (float)c;
      r.d = (float)(b - c);
      r.k1 = c > 1e-30 ? (float)(1.0 / (6.0 * b * c)) : 0.0f;
      r.k2 = (float)(1.0 / (3.0 * b));
      r.k3 = (float)(1.0 / (6.0 * a * b));
      r.k4 = (float)(2.0 / (3.0 * a));
      static_cast<H0Bin*>(out)[u] = r;
    } else {
      HlBin r{};
      r.ka = (float)ka;
      r.kb = (float)kb;
      const double p = w[2], q = w[1], rr = w[0];
      r.p = (float)p;
      r.q = (float)q;
      r.r = (float)rr;
      r.inv6pq = (float)(1.0 / (6.0 * p * q));
      r.inv_r = rr > 1e-30 ? (float)(1.0 / rr) : 0.0f;
      static_cast<HlBin*>(out)[u] = r;
    }
  }
}

size_t hex_bin_size(int basis) { return basis == BASIS_H0 ? sizeof(H0Bin) : sizeof(HlBin); }

// Bins per view that hold every tile's window (host-side).
int hex_tile_window(const Proj2DArgs& g, double dt, const ViewGeo* views) {
  const HexArgs a{g, dt};
  double cx, cy, hx, hy;
  hex_tile_box(a, &cx, &cy, &hx, &hy);
  return window_bound(g, views, cx, cy, hx, hy);
}

namespace {
template <int HB, int G, int W>
hipError_t hex_forward_g(const HexArgs& ha, const GroupRun& r, const float* img, float* sino, hipStream_t s) {
  const Proj2DArgs& g = ha.g;
  if (r.rows)
    hex_interleave_kernel<G><<<dim3((unsigned)(g.nx + 15) / 16, (unsigned)(g.ny + 15) / 16, (unsigned)r.groups()), 256,
                               0, s>>>(r.sym, g.nx, g.ny, r.m, r.batch, img, r.rows);
  const dim3 grid((unsigned)(r.sym.nrep * g.nchunk), (unsigned)r.groups(), (unsigned)r.split);
  const float* const p = r.rows ? r.rows : img;
  if (G == 1 && (size_t)g.nx * g.ny >= (size_t)1 << 30)
    hex_fwd_kernel<HB, 1, W, true><<<grid, 64 * W, 0, s>>>(ha, r.sym, r.m, r.batch, p, sino, r.part);
  else
    hex_fwd_kernel<HB, G, W, false><<<grid, 64 * W, 0, s>>>(ha, r.sym, r.m, r.batch, p, sino, r.part);
  return hipGetLastError();
}

template <int HB, int G>
hipError_t hex_backward_g(const HexArgs& ha, const GroupRun& r, const float* sino, float* img, hipStream_t s) {
  const dim3 grid((unsigned)r.sym.ntile, (unsigned)r.split, (unsigned)r.groups());
  const size_t lds = (size_t)r.nvc * r.win * (16 * HexBwd<HB>::kRec + 4 * G);
  hex_bwd_group_kernel<HB, G><<<grid, 256, lds, s>>>(ha, r.sym, r.m, r.batch, sino, img, r.vpg, r.nvc, r.win, r.part);
  return hipGetLastError();
}

// Waves per (view, chunk): as many as a launch of one image needs to fill the
// GPU, since every wave repeats a strip's set-up and shortens its lines.  A at
// 8 / 4 / 2 waves, us: H0 128 x 147, 360 views (1448 workgroups) 52 / 62 / 94;
// H0 256 x 296, 1024 views (8208) 543 / 496 / 476, batch 16 2398 / 2164 / 1963;
// Hl, batch 64 8525 / 7805 / 7107, one image without symmetries (16368) 738 /
// 619 / 570.  The choice follows the handle, not the batch, so that an image's
// sums associate alike in every batch.
int hex_waves(const Proj2DArgs& g, const GroupRun& r) {
  const long long n = (long long)r.sym.nrep * g.nchunk;
  return r.lone ? 1 : (n < 2048 ? 8 : (n < 6000 ? 4 : 2));
}

template <int HB, int G>
hipError_t hex_forward_w(const HexArgs& ha, const GroupRun& r, const float* img, float* sino, hipStream_t s) {
  switch (hex_waves(ha.g, r)) {
    case 8: return hex_forward_g<HB, G, 8>(ha, r, img, sino, s);
    case 4: return hex_forward_g<HB, G, 4>(ha, r, img, sino, s);
    case 2: return hex_forward_g<HB, G, 2>(ha, r, img, sino, s);
    default: return hex_forward_g<HB, 1, 1>(ha, r, img, sino, s);  // lone: one value per point
  }
}

template <int HB>
hipError_t hex_forward_b(const HexArgs& ha, const GroupRun& r, const float* img, float* sino, hipStream_t s) {
  if (r.lone && r.g != 1) return hipErrorInvalidValue;
  switch (r.g) {
    case 1: return hex_forward_w<HB, 1>(ha, r, img, sino, s);
    case 2: return hex_forward_w<HB, 2>(ha, r, img, sino, s);
    case 4: return hex_forward_w<HB, 4>(ha, r, img, sino, s);
    case 8: return hex_forward_w<HB, 8>(ha, r, img, sino, s);
    default: return hipErrorInvalidValue;
  }
}

template <int HB>
hipError_t hex_backward_b(const HexArgs& ha, const GroupRun& r, const float* sino, float* img, hipStream_t s) {
  switch (r.g) {
    case 1: return hex_backward_g<HB, 1>(ha, r, sino, img, s);
    case 2: return hex_backward_g<HB, 2>(ha, r, sino, img, s);
    case 4: return hex_backward_g<HB, 4>(ha, r, sino, img, s);
    case 8: return hex_backward_g<HB, 8>(ha, r, sino, img, s);
    default: return hipErrorInvalidValue;
  }
}
}  // namespace

// r.split > 1 needs r.part with split * batch * np * nu doubles.
hipError_t launch_hex_forward(int basis, const Proj2DArgs& g, double dt, const GroupRun& r, const float* img,
                              float* sino, hipStream_t s) {
  if (r.split < 1 || (r.split > 1 && !r.part)) return hipErrorInvalidValue;
  const HexArgs ha{g, dt};
  const hipError_t e = basis == BASIS_H0 ? hex_forward_b<BASIS_H0>(ha, r, img, sino, s)
                                         : hex_forward_b<BASIS_HL>(ha, r, img, sino, s);
  if (e == hipSuccess && r.split > 1 && r.sum)
    return launch_sum_parts(r.part, sino, (size_t)r.batch * g.np * g.nu, r.split, s);
  return e;
}

// r.split > 1 needs r.part with split * batch * nc * nl doubles.
hipError_t launch_hex_backward(int basis, const Proj2DArgs& g, double dt, const GroupRun& r, const float* sino,
                               float* img, hipStream_t s) {
  if (r.split < 1 || (r.split > 1 && !r.part)) return hipErrorInvalidValue;
  const HexArgs ha{g, dt};
  hipError_t e;
  if (r.win > 0) {
    e = basis == BASIS_H0 ? hex_backward_b<BASIS_H0>(ha, r, sino, img, s)
                          : hex_backward_b<BASIS_HL>(ha, r, sino, img, s);
  } else {
    if (r.sym.nh != 1) return hipErrorInvalidValue;
    const dim3 grid((g.nx + kTile - 1) / kTile, (g.ny + kTile - 1) / kTile, (unsigned)(r.batch * r.split));
    if (basis == BASIS_H0) hex_bwd_kernel<BASIS_H0><<<grid, 256, 0, s>>>(ha, sino, img, r.split, r.vpg, r.part);
    else hex_bwd_kernel<BASIS_HL><<<grid, 256, 0, s>>>(ha, sino, img, r.split, r.vpg, r.part);
    e = hipGetLastError();
  }
  if (e == hipSuccess && r.split > 1) e = launch_sum_parts(r.part, img, (size_t)r.batch * g.nx * g.ny, r.split, s);
  return e;
}

// Explicit system matrix (h0_matrix_generation / hl_matrix_generation; the
// reference's hl_matrix_generate, layers/A_Hl.cu:370-451, and its H0 twin,
// A_H0.cu:360, are never called): one lane per (view, bin) walks every
// lattice row the bin's strip can reach, points in ascending column order,
// with the same pixel-set tests and footprint as hex_fwd_kernel, and keeps
// the points whose footprint is > 0 as (p nu + u, il nc + ic, conv) --
// without the dx dy factor, as the reference's generators.  A count pass,
// host offsets, then a write pass that never writes past its count.
template <int HB, bool WRITE>
__global__ __launch_bounds__(256) void hex_matgen_kernel(HexArgs ha, unsigned int* __restrict__ counts,
                                                         const long long* __restrict__ offsets,
                                                         double* __restrict__ out) {
  using T = HexTraits<HB>;
  const Proj2DArgs& g = ha.g;
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int v = wave / g.nchunk;
  if (v >= g.np) return;
  const int u = (wave - v * g.nchunk) * 64 + lane;
  if (u >= g.nu) return;
  const ViewGeo vg = g.views[v];
  const typename T::Bin rec = reinterpret_cast<const typename T::Bin*>(g.bins)[(size_t)v * g.nu + u];
  const double eax = vg.e0x + u * vg.pux, eay = vg.e0y + u * vg.puy;
  const double ebx = eax + vg.pux, eby = eay + vg.puy;
  const double sa = -eay * g.dx, ma = eax * g.dy, ca = eax * vg.w0y - eay * vg.w0x;
  const double sb = -eby * g.dx, mb = ebx * g.dy, cb = ebx * vg.w0y - eby * vg.w0x;
  const double lax = (u == 0) ? eax - vg.pux : eax, lay = (u == 0) ? eay - vg.puy : eay;
  const double lbx = (u == g.nu - 1) ? ebx + vg.pux : ebx, lby = (u == g.nu - 1) ? eby + vg.puy : eby;
  const double sq = -lay * g.dx, mq = lax * g.dy, cq = lax * vg.w0y - lay * vg.w0x;
  const double sr = -lby * g.dx, mr = lbx * g.dy, cr = lbx * vg.w0y - lby * vg.w0x;
  const double rq = hex_reach(-lay, lax, ha.dt), rr = hex_reach(-lby, lbx, ha.dt);
  const double ka = rec.ka, kb = rec.kb;
  const double isq = sq != 0.0 ? 1.0 / sq : 0.0, isr = sr != 0.0 ? 1.0 / sr : 0.0;
  const size_t bin = (size_t)v * g.nu + u;
  const long long pos = WRITE ? offsets[bin] : 0;
  const unsigned int cap = WRITE ? counts[bin] : 0u;
  unsigned int cnt = 0;
  for (int il = 0; il < g.ny; ++il) {
    const double sh = (il & 1) ? 0.5 : 0.0;
    const double r1 = -rq - (mq * il + cq) - sq * sh;
    const double r2 = rr - (mr * il + cr) - sr * sh;
    double lo = 0.0, hi = (double)(g.nx - 1 - (il & 1));
    if (sq > 0.0) lo = fmax(lo, ceil(r1 * isq));
    else if (sq < 0.0) hi = fmin(hi, floor(r1 * isq));
    else if (r1 > 0.0) continue;
    if (sr > 0.0) hi = fmin(hi, ceil(r2 * isr) - 1.0);
    else if (sr < 0.0) lo = fmax(lo, floor(r2 * isr) + 1.0);
    else if (r2 <= 0.0) continue;
    for (int ic = (int)lo; ic <= (int)hi; ++ic) {
      const double xc = ic + sh;
      const float ta = (float)(ka * (sa * xc + ma * il + ca));
      const float tb = (float)(kb * (sb * xc + mb * il + cb));
      const float w = T::conv(rec, ta, tb);
      if (!(w > 0.0f)) continue;
      if (WRITE) {
        if (cnt >= cap) return;
        double* o = out + 3 * (pos + cnt);
        o[0] = (double)bin;
        o[1] = (double)il * g.nx + ic;
        o[2] = (double)w;
      }
      ++cnt;
    }
  }
  if (!WRITE) counts[bin] = cnt;
}

hipError_t launch_hex_matgen(int basis, const Proj2DArgs& g, double dt, bool write, unsigned int* counts,
                             const long long* offsets, double* out, hipStream_t s) {
  HexArgs ha{g, dt};
  dim3 grid((g.np * g.nchunk + 3) / 4), block(256);
  if (basis == BASIS_H0) {
    if (write) hex_matgen_kernel<BASIS_H0, true><<<grid, block, 0, s>>>(ha, counts, offsets, out);
    else hex_matgen_kernel<BASIS_H0, false><<<grid, block, 0, s>>>(ha, counts, offsets, out);
  } else if (basis == BASIS_HL) {
    if (write) hex_matgen_kernel<BASIS_HL, true><<<grid, block, 0, s>>>(ha, counts, offsets, out);
    else hex_matgen_kernel<BASIS_HL, false><<<grid, block, 0, s>>>(ha, counts, offsets, out);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_hex_count(const Proj2DArgs& g, double dt, unsigned long long* out, hipStream_t s) {
  HexArgs ha{g, dt};
  hex_count_kernel<<<dim3((g.nx + 15) / 16, (g.ny + 15) / 16), dim3(256), 0, s>>>(ha, out);
  return hipGetLastError();
}

}  // namespace sgdct
