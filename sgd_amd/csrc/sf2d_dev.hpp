// sf2d_dev.hpp -- device code of the 2-D separable-footprint projector,
// shared by sf2d.hip and the batched persistent kernels (batch.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "group2d_dev.hpp"
#include "projector.hpp"

namespace sgdct {

// min / max / clamp of finite values as v_med3_f32: exact, one instruction, and
// no NaN quieting of the operands (fminf / fmaxf add it)
__device__ __forceinline__ float min2f(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, -__builtin_inff()); }
__device__ __forceinline__ float max2f(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, __builtin_inff()); }
__device__ __forceinline__ float clamp3(float x, float lo, float hi) { return __builtin_amdgcn_fmed3f(x, lo, hi); }

// 1 / d for a normal double d: the approximation of v_rcp_f64 (relative error
// below 2^-23) refined by two Newton steps to an ulp, in place of the double
// division's longer sequence (scaling, three steps, fix-up)
__device__ __forceinline__ double recip(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
  return __builtin_fma(r, __builtin_fma(-d, r, 1.0), r);
}

// Unit-height trapezoid over sorted corners, 1 / (q1 - q0) and 1 / (q3 - q2)
// (finite for an empty ramp, whose terms are then zero).
struct Trap {
  float q0, q1, q2, q3, ir, iff;
};

__device__ __forceinline__ void sort2(float a, float b, float& lo, float& hi) {
  lo = min2f(a, b);
  hi = max2f(a, b);
}

// Trapezoid of two pairs of corners, each sorted.
__device__ __forceinline__ Trap make_trap(float a0, float a1, float b0, float b1) {
  Trap t;
  t.q0 = min2f(a0, b0);
  t.q3 = max2f(a1, b1);
  sort2(max2f(a0, b0), min2f(a1, b1), t.q1, t.q2);
  t.ir = __builtin_amdgcn_rcpf(max2f(t.q1 - t.q0, 1e-30f));
  t.iff = __builtin_amdgcn_rcpf(max2f(t.q3 - t.q2, 1e-30f));
  return t;
}

__device__ __forceinline__ Trap sorted_trap(float a, float b, float c, float d) {
  float a0, a1, b0, b1;
  sort2(a, b, a0, a1);
  sort2(c, d, b0, b1);
  return make_trap(a0, a1, b0, b1);
}

// Area of the trapezoid over [s1, s2] (layers/A_SF.cu:48-84), the ramps'
// squares differenced as products of sum and difference.  A walk over adjacent
// intervals passes what it holds of the last edge on: start() at the first
// edge, next() per further edge.
struct TrapWalk {
  float b, m, e;  // clamped distances into the rising ramp, flat top, falling ramp
  __device__ __forceinline__ void start(const Trap& t, float s) {
    b = clamp3(s, t.q0, t.q1) - t.q0;
    m = clamp3(s, t.q1, t.q2);
    e = t.q3 - clamp3(s, t.q2, t.q3);
  }
  __device__ __forceinline__ float next(const Trap& t, float s) {
    TrapWalk n;
    n.start(t, s);
    const float ramps =
        __builtin_fmaf((e - n.e) * (e + n.e), t.iff, (n.b - b) * (n.b + b) * t.ir);
    const float area = __builtin_fmaf(0.5f, ramps, n.m - m);
    *this = n;
    return area;
  }
};

__device__ __forceinline__ float trap_gamma(const Trap& t, float s1, float s2) {
  TrapWalk w;
  w.start(t, s1);
  return w.next(t, s2);
}

// dx / max(|cos t|, |sin t|) of the ray through (wx, wy) from the source;
// v_sqrt_f32 (1 ulp) instead of the correctly rounded square-root sequence
__device__ __forceinline__ float sf_weight(float dx, float wx, float wy) {
  float r2 = wx * wx + wy * wy;
  return dx * __builtin_amdgcn_sqrtf(r2) * __builtin_amdgcn_rcpf(fmaxf(fabsf(wx), fabsf(wy)));
}

// A: bin-driven gather (the strip walk of fwd_bin_lines, corner rule h = 1/2).
// One wave: bins [64 chunk, 64 chunk + 64) of view v, lines m = w0 mod wn of
// segment seg of nseg, sums into acc[G]; images as in fwd_bin_lines, by address
// where they hold 4 GiB or more (FAR).
template <int G, bool FAR = false>
__device__ __forceinline__ void sf_fwd_lines(const Proj2DArgs& g, int v, int chunk, const float* __restrict__ rows_img,
                                             const float* __restrict__ cols_img, int w0, int wn, int seg, int nseg,
                                             double (&acc)[G], int place = 0) {
  const bool inside = chunk * 64 + (int)(threadIdx.x & 63) < g.nu;
  const int u = inside ? chunk * 64 + (int)(threadIdx.x & 63) : g.nu - 1;
  const ViewGeo vg = g.views[v];
  const int umid = min(chunk * 64 + 32, g.nu - 1);
  const double mx = vg.e0x + (umid + 0.5) * vg.pux, my = vg.e0y + (umid + 0.5) * vg.puy;
  const bool rows = fabs(my) >= fabs(mx);

  const double eax = vg.e0x + u * vg.pux, eay = vg.e0y + u * vg.puy;
  const double ebx = eax + vg.pux, eby = eay + vg.puy;
  const double acx = -eay * g.dx, acy = eax * g.dy, ac0 = eax * vg.w0y - eay * vg.w0x;
  const double bcx = -eby * g.dx, bcy = ebx * g.dy, bc0 = ebx * vg.w0y - eby * vg.w0x;
  const double ra = 0.5 * (fabs(acx) + fabs(acy)), rb = 0.5 * (fabs(bcx) + fabs(bcy));
  const double sa = rows ? acx : acy, ma = rows ? acy : acx;
  const double sb = rows ? bcx : bcy, mb = rows ? bcy : bcx;
  const int nmin = rows ? g.nx : g.ny, nmaj = rows ? g.ny : g.nx;
  const bool strided = !rows && !cols_img;
  int base = 0, smin = strided ? g.nx : 1, smaj = strided ? 1 : nmin;
  if (G == 1 && place) {
    const SymOp::Steps st = SymOp::steps(place, g.nx, g.ny);
    base = st.base;
    smin = rows ? st.x : st.y;
    smaj = rows ? st.y : st.x;
  }
  // beta(ix, iy) = cross(pu, w): affine, steps (bcxx, bcyy) per index
  const double bcxx = -vg.puy * g.dx, bcyy = vg.pux * g.dy, bc00 = vg.pux * vg.w0y - vg.puy * vg.w0x;
  const double sB = rows ? bcxx : bcyy, mB = rows ? bcyy : bcxx;
  const float dN = (float)sa, dB = (float)sB;
  // source -> pixel centre, along the walk (moving) and across it (fixed)
  const double dmov = rows ? g.dx : g.dy, dfix = rows ? g.dy : g.dx;
  const double w0mov = rows ? vg.w0x : vg.w0y, w0fix = rows ? vg.w0y : vg.w0x;
  const float fdmov = (float)dmov, fdx = (float)g.dx;
  // offsets of N_u and beta from a pixel's centre to its corners across the
  // walk on the leading side (nl, bl) and the trailing side (-nl, -bl): the
  // leading corners of one pixel are the trailing ones of the next
  const float w_n = 0.5f * (float)sa, c_n = 0.5f * (float)ma, w_b = 0.5f * (float)sB, c_b = 0.5f * (float)mB;
  const float nl1 = w_n - c_n, nl2 = w_n + c_n, bl1 = w_b - c_b, bl2 = w_b + c_b;

  int m_lo, m_hi;
  strip_lines(sa, ma, -ra - ac0, sb, mb, rb - bc0, 0.0, (double)(nmin - 1), nmaj, &m_lo, &m_hi);
  if (nseg > 1) {
    const int len = (nmaj + nseg - 1) / nseg;
    m_lo = max(m_lo, seg * len);
    m_hi = min(m_hi, seg * len + len - 1);
  }
  if (!inside) m_hi = -1;
  const float* const img = (rows || strided) ? rows_img : cols_img;
  const __amdgpu_buffer_rsrc_t img_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(img), (short)0, (int)(4u * G * (unsigned)g.nx * (unsigned)g.ny), 0x00020000);
  using Off = std::conditional_t<FAR, size_t, unsigned>;  // modulo its range: steps may be negative
  const Off bstep = 4 * G * (Off)smin;
  // Pixel interval of line m, from N_u + R_u >= 0 and N_{u+1} - R_{u+1} < 0.
  const float lastn = (float)(nmin - 1);
  StripLines lines;
  lines.set(sa, ma, -ra - ac0, sb, mb, rb - bc0, (float)nmaj);
  // The weight's larger coordinate is the fixed one (reciprocal once per line)
  // if every lane's strip stays inside 45 degrees: at a line's end pixels the
  // moving coordinate exceeds the ray's by at most the strip's half width and a
  // pixel.
  const double f0 = __builtin_fma((double)m_lo, dfix, w0fix), f1 = __builtin_fma((double)m_hi, dfix, w0fix);
  const double slope = fmax(fabs(rows ? eax / eay : eay / eax), fabs(rows ? ebx / eby : eby / ebx));
  const bool own = __ballot(inside && !(f0 * f1 > 0.0 && fmin(fabs(f0), fabs(f1)) * (0.999 - slope) >
                                                             2.0 * (fabs(dmov) + fabs(dfix)))) == 0;
  auto walk = [&](auto own_c) {
    for (int m = m_lo + ((w0 - m_lo) & (wn - 1)); m <= m_hi; m += wn) {
      float flo, fhi;
      if (!lines.at((float)m, 0.0f, &flo, &fhi))
        lines.settle(sa, -ra - ma * m - ac0, sb, rb - mb * m - bc0, (double)lastn, &flo, &fhi);
      flo = fmaxf(ceilf(flo), 0.0f);
      fhi = fminf(floorf(fhi), lastn);
      if (!(flo <= fhi)) continue;
      const int n0 = (int)flo;
      const double dm = (double)m, dn = (double)flo;
      float nu_ = (float)__builtin_fma(dn, sa, __builtin_fma(dm, ma, ac0));
      float be = (float)__builtin_fma(dn, sB, __builtin_fma(dm, mB, bc00));
      float wm = (float)__builtin_fma(dn, dmov, w0mov);
      const float wf = (float)__builtin_fma(dm, dfix, w0fix);
      const float ifix = __builtin_amdgcn_rcpf(fabsf(wf)), wf2 = wf * wf;
      Off off = 4 * G * ((Off)base + (Off)m * (Off)smaj + (Off)n0 * (Off)smin);
      const Off end = off + (Off)((int)fhi - n0 + 1) * bstep;
      float accl[G];
#pragma unroll
      for (int k = 0; k < G; ++k) accl[k] = 0.0f;
      // corner projections relative to edge u, -N_u(c) / beta(c), of the
      // trailing corners of the line's first pixel
      float t1, t2;
      sort2((nl2 - nu_) * __builtin_amdgcn_rcpf(be - bl2), (nl1 - nu_) * __builtin_amdgcn_rcpf(be - bl1), t1, t2);
      do {
        float x[G];
        if constexpr (FAR) __builtin_memcpy(x, reinterpret_cast<const char*>(img) + off, sizeof(x));
        else buffer_load_n<G>(img_rsrc, off, x);
        float l1, l2;
        sort2(-(nu_ + nl1) * __builtin_amdgcn_rcpf(be + bl1), -(nu_ + nl2) * __builtin_amdgcn_rcpf(be + bl2), l1, l2);
        const Trap t = make_trap(t1, t2, l1, l2);
        t1 = l1;
        t2 = l2;
        const float gm = trap_gamma(t, 0.0f, 1.0f);
        // dx / max(|cos|, |sin|) of the ray through the pixel's centre
        const float il = decltype(own_c)::value ? ifix : __builtin_amdgcn_rcpf(fmaxf(fabsf(wm), fabsf(wf)));
        const float w = fdx * __builtin_amdgcn_sqrtf(__builtin_fmaf(wm, wm, wf2)) * il;
        const float val = (gm > 1e-7f) ? gm * w : 0.0f;
#pragma unroll
        for (int k = 0; k < G; ++k) accl[k] = __builtin_fmaf(val, x[k], accl[k]);
        off += bstep;
        nu_ += dN;
        be += dB;
        wm += fdmov;
      } while (off != end);
#pragma unroll
      for (int k = 0; k < G; ++k) acc[k] += (double)accl[k];
    }
  };
  if (own) walk(std::true_type{});
  else walk(std::false_type{});
}

// One wave of the batched work queue: item `wave` = chunk * np + view, every
// line, finished values to sino.
__device__ __forceinline__ void sf_fwd_wave(const Proj2DArgs& g, const float* __restrict__ img,
                                            float* __restrict__ sino, int wave) {
  const int chunk = wave / g.np;
  if (chunk >= g.nchunk) return;
  const int v = wave - chunk * g.np, u = chunk * 64 + (int)(threadIdx.x & 63);
  double acc[1] = {0.0};
  sf_fwd_lines<1>(g, v, chunk, img, nullptr, 0, 1, 0, 1, acc);
  if (u < g.nu) sino[(size_t)v * g.nu + u] = (float)acc[0];
}


// A^T: pixel-driven gather, one 16x16 tile per 256-thread block, views
// [v_begin, v_end); with `part` the FP64 sums go to part[iy * nx + ix].
__device__ __forceinline__ void sf_bwd_tile(const Proj2DArgs& g, const float* __restrict__ sino,
                                            float* __restrict__ img, int tile_x, int tile_y, int v_begin = 0,
                                            int v_end = -1, double* __restrict__ part = nullptr) {
  const int ix = tile_x * kTile + (threadIdx.x & (kTile - 1));
  const int iy = tile_y * kTile + threadIdx.x / kTile;
  if (ix >= g.nx || iy >= g.ny) return;
  if (v_end < 0) v_end = g.np;
  const float fdx = (float)g.dx;
  double acc = 0.0;
  for (int v = v_begin; v < v_end; ++v) {
    const ViewGeo& vg = g.views[v];
    const double wx = ix * g.dx + vg.w0x, wy = iy * g.dy + vg.w0y;
    const double n0 = vg.e0x * wy - vg.e0y * wx;
    const double be = vg.pux * wy - vg.puy * wx;
    const double kc = -n0 / be;
    const double kfl = floor(kc);
    const float kf = (float)(kc - kfl);
    const float kcf = (float)kc, bef = (float)be;
    const float gx = 0.5f * __builtin_fmaf(kcf, vg.gx1, vg.gx0), gy = 0.5f * __builtin_fmaf(kcf, vg.gy1, vg.gy0);
    const float bx = 0.5f * vg.gx1, by = 0.5f * vg.gy1;
    // corner c: k*(c) - kc = -(d.G) / (beta + d.grad beta)
    const Trap t = sorted_trap(kf + (gx + gy) * __builtin_amdgcn_rcpf(bef - bx - by),
                               kf + (gx - gy) * __builtin_amdgcn_rcpf(bef - bx + by),
                               kf - (gx - gy) * __builtin_amdgcn_rcpf(bef + bx - by),
                               kf - (gx + gy) * __builtin_amdgcn_rcpf(bef + bx + by));
    const int ki = (int)kfl;
    const int jlo = (int)floorf(t.q0), jhi = (int)floorf(t.q3);
    if (ki + jhi < 0 || ki + jlo > g.nu - 1) continue;
    const int ulo = max(ki + jlo, 0), uhi = min(ki + jhi, g.nu - 1);
    const float w = sf_weight(fdx, (float)wx, (float)wy);
    const float* row = sino + (size_t)v * g.nu;
    float accv = 0.0f, edge = (float)(ulo - ki);
    TrapWalk walk;
    walk.start(t, edge);
    for (int u = ulo; u <= uhi; ++u) {
      edge += 1.0f;
      const float gm = walk.next(t, edge);
      accv = __builtin_fmaf((gm > 1e-7f) ? gm : 0.0f, row[u], accv);
    }
    acc += (double)(accv * w);
  }
  if (part) part[(size_t)iy * g.nx + ix] = acc;
  else img[(size_t)iy * g.nx + ix] = (float)acc;
}

// A^T in the grouped frame (group2d_dev.hpp): no records, the sinogram values
// of a tile's bins staged in LDS.  sf_bwd_tile's arithmetic per view.
struct SfBwd {
  using Args = Proj2DArgs;
  static constexpr int kRec = 0;
  struct Pixel {
    double fx, fy;
  };
  __device__ static __forceinline__ const Proj2DArgs& geo(const Args& a) { return a; }
  __device__ static __forceinline__ void window(const Args& a, const ViewGeo& vg, int ix0, int iy0, int* lo, int* n,
                                                int cap) {
    tile_window(a, vg, ix0, iy0, lo, n, cap);
  }
  __device__ static __forceinline__ Pixel pixel(const Args& a, int ix, int iy) { return {ix * a.dx, iy * a.dy}; }
  __device__ static __forceinline__ bool active(const Args&, int, int) { return true; }
  __device__ static __forceinline__ void image(const Args& a, int op, int ix, int iy, int* qx, int* qy) {
    SymOp::pixel(op, a.nx, a.ny, ix, iy, qx, qy);
  }
  __device__ static __forceinline__ float value(const float4 (&)[1], float y) { return y; }
  __device__ static __forceinline__ double result(const Args&, double acc) { return acc; }

  template <int G>
  __device__ static __forceinline__ void view(const Args& g, const ViewGeo& vg, const Pixel& p, const Staged<kRec, G>& st,
                                              int base, int wlo, int wn, float (&accv)[G]) {
    const double wx = p.fx + vg.w0x, wy = p.fy + vg.w0y;
    const double n0 = vg.e0x * wy - vg.e0y * wx;
    const double be = vg.pux * wy - vg.puy * wx;
    const double kc = -n0 * recip(be);
    const double kfl = floor(kc);
    const float kf = (float)(kc - kfl);
    const float kcf = (float)kc, bef = (float)be;
    const float gx = 0.5f * __builtin_fmaf(kcf, vg.gx1, vg.gx0), gy = 0.5f * __builtin_fmaf(kcf, vg.gy1, vg.gy0);
    const float bx = 0.5f * vg.gx1, by = 0.5f * vg.gy1;
    // corner c: k*(c) - kc = -(d.G) / (beta + d.grad beta)
    const Trap t = sorted_trap(kf + (gx + gy) * __builtin_amdgcn_rcpf(bef - bx - by),
                               kf + (gx - gy) * __builtin_amdgcn_rcpf(bef - bx + by),
                               kf - (gx - gy) * __builtin_amdgcn_rcpf(bef + bx - by),
                               kf - (gx + gy) * __builtin_amdgcn_rcpf(bef + bx + by));
    const int ki = (int)kfl;
    // bins of the trapezoid, inside the detector and the tile's window
    const int ulo = max(ki + (int)floorf(t.q0), wlo), uhi = min(ki + (int)floorf(t.q3), wlo + wn - 1);
    const float w = sf_weight((float)g.dx, (float)wx, (float)wy);
    float edge = (float)(ulo - ki);
    TrapWalk walk;
    walk.start(t, edge);
    int at = base + ulo - wlo;
    for (int u = ulo; u <= uhi; ++u, ++at) {
      edge += 1.0f;
      const float gm = walk.next(t, edge);
      st.add(at, (gm > 1e-7f) ? gm : 0.0f, accv);
    }
#pragma unroll
    for (int s = 0; s < G; ++s) accv[s] *= w;
  }
};

}  // namespace sgdct
