// group2d_dev.hpp -- device code shared by the grouped 2-D projectors
// (group2d.hpp): wide and scalar loads, the sum over an A workgroup's waves,
// and the frame of A^T (tiles, staging, output) around each basis's footprint.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "group2d.hpp"

namespace sgdct {

// N consecutive floats of a buffer resource at a byte offset (reads past the
// resource's end return zero).
template <int N>
__device__ __forceinline__ void buffer_load_n(__amdgpu_buffer_rsrc_t r, unsigned off, float (&x)[N]) {
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  if constexpr (N == 1) {
    x[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
  } else if constexpr (N == 2) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0);
    x[0] = __uint_as_float(v.x);
    x[1] = __uint_as_float(v.y);
  } else {
    static_assert(N % 4 == 0, "whole 16-byte loads");
#pragma unroll
    for (int k = 0; k < N; k += 4) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 4 * k, 0);
      x[k] = __uint_as_float(v.x);
      x[k + 1] = __uint_as_float(v.y);
      x[k + 2] = __uint_as_float(v.z);
      x[k + 3] = __uint_as_float(v.w);
    }
  }
}

// Loads of tables that no kernel writes, at wave-uniform addresses, through
// the constant address space, so that they become scalar loads also after a
// workgroup barrier (where the compiler can no longer tell that the table has
// not changed; as vector loads the view record cost A^T a memory latency per
// view: 303 -> 265 us with cheaper tile windows, 200 us with these and with a
// bin's staged values loaded together).
template <class T>
__device__ __forceinline__ T const_load(const T* p, int i) {
  typedef const __attribute__((address_space(4))) T* const_ptr;
  return *((const_ptr)(uintptr_t)p + i);
}

__device__ __forceinline__ ViewGeo scalar_view(const ViewGeo* views, int v) {
  const double* d = reinterpret_cast<const double*>(views + __builtin_amdgcn_readfirstlane(v));
  ViewGeo r{};
  r.e0x = const_load(d, 0);
  r.e0y = const_load(d, 1);
  r.pux = const_load(d, 2);
  r.puy = const_load(d, 3);
  r.w0x = const_load(d, 4);
  r.w0y = const_load(d, 5);
  const float* f = reinterpret_cast<const float*>(d + 8);
  r.gx0 = const_load(f, 0);
  r.gy0 = const_load(f, 1);
  r.gx1 = const_load(f, 2);
  r.gy1 = const_load(f, 3);
  r.db = const_load(f, 4);
  return r;
}

// Bin window of one view for a pixel tile: bins touched by the tile's box
// widened by h, from the exact projection of its four corners, +-1 margin.
__host__ __device__ inline void tile_window(const Proj2DArgs& g, const ViewGeo& vg, int ix0, int iy0, int* lo,
                                            int* n, int cap = kMaxWindow) {
  double umin = 1e300, umax = -1e300;
#pragma unroll 1  // four divisions at once cost the gather kernels a wave per SIMD
  for (int c = 0; c < 4; ++c) {
    double fx = (c & 1) ? (ix0 + kTile - 1 + g.h) : (ix0 - g.h);
    double fy = (c & 2) ? (iy0 + kTile - 1 + g.h) : (iy0 - g.h);
    double wx = fx * g.dx + vg.w0x, wy = fy * g.dy + vg.w0y;
    double n0 = vg.e0x * wy - vg.e0y * wx;
    double be = vg.pux * wy - vg.puy * wx;
    double uu = -n0 / be;
    umin = fmin(umin, uu);
    umax = fmax(umax, uu);
  }
  double l = fmax(floor(umin) - 1.0, 0.0), hgh = fmin(floor(umax) + 1.0, (double)(g.nu - 1));
  int li = (int)l, hi = (int)hgh;
  *lo = li;
  *n = hi >= li ? min(hi - li + 1, cap) : 0;
}

// Sums of an A workgroup's W waves (red[wave][slot][lane]) in wave order,
// times the bin's factors, to the outputs of every slot: view h v, bin u
// (reversed where h mirrors).  All threads of the workgroup call this after
// writing red and a barrier.
template <int G, int W>
__device__ __forceinline__ void fwd_group_store(const Proj2DArgs& g, const SymPlan& sp, int rep, int v, int u, int m,
                                                int batch, const double (*red)[G][64], double f0, double f1, double f2,
                                                float* __restrict__ sino, double* __restrict__ part) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int img0 = blockIdx.y * m, nimg = min(m, batch - img0);
  const size_t nsino = (size_t)g.np * g.nu;
  for (int s = wv; s < sp.nh * nimg; s += W) {
    const int k = s >> sp.lg, h = s & (sp.nh - 1);
    const int vh = sp.rep_view ? sp.rep_view[rep * sp.row + sp.h0 + h] : v;
    if (vh < 0) continue;
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < W; ++w) t += red[w][s][lane];
    t = t * f0 * f1 * f2;
    const int uh = SymOp::reverses(sp.op[h]) ? g.nu - 1 - u : u;
    const size_t o = (img0 + k) * nsino + (size_t)vh * g.nu + uh;
    if (part) part[(size_t)blockIdx.z * batch * nsino + o] = t;
    else sino[o] = (float)t;
  }
}

// A lone run's sums of bin u over its segments, times the bin's factors one by
// one (each product rounded before the addition), added in segment order.  All threads of the workgroup call this after
// writing red and a barrier.
__device__ __forceinline__ void fwd_lone_store(int nseg, const double (*red)[64], double f0, double f1, double f2,
                                               float* out) {
  if (threadIdx.x >= 64) return;
  double t = 0.0;
  for (int k = 0; k < nseg; ++k) {
#pragma clang fp contract(off)
    const double p = red[k][threadIdx.x] * f0 * f1 * f2;
    t += p;
  }
  *out = (float)t;
}

// Points [flo, fhi] of line l of a strip, from the tests
//   q:  s_q n >= r1     and     r:  s_r n < r2,      r1 = q0 - m_q l, r2 = r0 - m_r l,
// on whole n.  Their ends are affine in l and formed in FP32; where one comes
// within its error of a whole number, `settle` tests that number in FP64, so that
// a line holds the points of the FP64 tests and no other (a point outside has
// no weight, but an infinite one would still turn the bin's sum into NaN).
struct StripLines {
  float lo0 = 0.0f, lo1 = 0.0f, hi0 = 0.0f, hi1 = 0.0f, tlo = -1.0f, thi = -1.0f;
  // lines |l| <= most; slopes that are not of one sign leave every line unsettled
  __device__ __forceinline__ void set(double s_q, double m_q, double q0, double s_r, double m_r, double r0, float most) {
    if (!((s_q > 0.0 && s_r > 0.0) || (s_q < 0.0 && s_r < 0.0))) return;
    const bool up = s_q > 0.0;
    const float a0 = (float)(q0 / s_q), a1 = (float)(-m_q / s_q), b0 = (float)(r0 / s_r), b1 = (float)(-m_r / s_r);
    lo0 = up ? a0 : b0;
    lo1 = up ? a1 : b1;
    hi0 = up ? b0 : a0;
    hi1 = up ? b1 : a1;
    // three roundings of at most 2^-24 of each term (at(): one more), and some
    tlo = 0.5f - 1e-6f - 2.4e-7f * __builtin_fmaf(fabsf(lo1), most, fabsf(lo0) + 1.0f);
    thi = 0.5f - 1e-6f - 2.4e-7f * __builtin_fmaf(fabsf(hi1), most, fabsf(hi0) + 1.0f);
  }
  // points n + shift; false: not settled
  __device__ __forceinline__ bool at(float l, float shift, float* lo, float* hi) const {
    *lo = __builtin_fmaf(l, lo1, lo0) - shift;
    *hi = __builtin_fmaf(l, hi1, hi0) - shift;
    return fabsf(__builtin_amdgcn_fractf(*lo) - 0.5f) <= tlo && fabsf(__builtin_amdgcn_fractf(*hi) - 0.5f) <= thi;
  }
  // at()'s ends, moved to the first and last point, within [0, last]
  __device__ __forceinline__ void settle(double s_q, double r1, double s_r, double r2, double last, float* lo,
                                         float* hi) const {
    if (tlo > 0.0f && thi > 0.0f) {  // off by less than a half: one of two whole numbers
      const double a = rint((double)*lo), b = rint((double)*hi);
      const bool up = s_q > 0.0;
      *lo = (float)((up ? s_q * a >= r1 : s_r * a < r2) ? a : a + 1.0);
      *hi = (float)((up ? s_r * b < r2 : s_q * b >= r1) ? b : b - 1.0);
      return;
    }
    double x = 0.0, y = last;
    if (s_q > 0.0) x = fmax(x, ceil(r1 / s_q));
    else if (s_q < 0.0) y = fmin(y, floor(r1 / s_q));
    else if (r1 > 0.0) y = -1.0;
    if (s_r > 0.0) y = fmin(y, ceil(r2 / s_r) - 1.0);
    else if (s_r < 0.0) x = fmax(x, floor(r2 / s_r) + 1.0);
    else if (r2 <= 0.0) y = -1.0;
    *lo = (float)x;
    *hi = (float)y;
  }
};

// Lines l of [0, n) on which some point x of [x0, x1] can pass both tests, s_q x
// + m_q l >= q0 and s_r x + m_r l < r0: each bounds l from one side at most,
// one line of margin.  (The rows at which the strip's two edges meet x0 and x1
// bound it only if the strip is narrower than they are far apart: a slab inside
// a wide bin's strip may lie to one side of all four.)
__device__ __forceinline__ void strip_lines(double s_q, double m_q, double q0, double s_r, double m_r, double r0,
                                            double x0, double x1, int n, int* lo, int* hi) {
  const double a = q0 - fmax(s_q * x0, s_q * x1), b = r0 - fmin(s_r * x0, s_r * x1);
  double l = 0.0, h = (double)(n - 1);
  if (m_q > 0.0) l = fmax(l, floor(a / m_q) - 1.0);
  else if (m_q < 0.0) h = fmin(h, ceil(a / m_q) + 1.0);
  if (m_r > 0.0) h = fmin(h, ceil(b / m_r) + 1.0);
  else if (m_r < 0.0) l = fmax(l, floor(b / m_r) - 1.0);
  *lo = (int)fmin(l, (double)n);
  *hi = (int)fmax(h, -1.0);
}

// A tile's staged bins in LDS: the records as REC float4 planes, then the G
// sinogram values of each bin as planes of up to 4, so that 16-byte reads of
// consecutive bins touch all banks.
template <int REC, int G> struct Staged {
  static constexpr int GV = G < 4 ? G : 4, GP = G / GV;  // values per vector, planes
  float4* rec;
  float* ys;
  int cap;
  __device__ __forceinline__ Staged(float4* lds, int cap_) : rec(lds), ys(reinterpret_cast<float*>(lds + REC * cap_)), cap(cap_) {}
  template <int N>
  __device__ __forceinline__ void record(int at, float4 (&r)[N]) const {
#pragma unroll
    for (int k = 0; k < N; ++k) r[k] = rec[k * cap + at];
  }
  __device__ __forceinline__ void put(int at, const float (&y)[G]) const {
#pragma unroll
    for (int p = 0; p < GP; ++p)
#pragma unroll
      for (int e = 0; e < GV; ++e) ys[(p * cap + at) * GV + e] = y[p * GV + e];
  }
  // acc += c * values of bin `at`
  __device__ __forceinline__ void add(int at, float c, float (&acc)[G]) const {
#pragma unroll
    for (int p = 0; p < GP; ++p) {
      float y[GV];
      __builtin_memcpy(y, __builtin_assume_aligned(ys + (p * cap + at) * GV, 4 * GV), sizeof(y));
#pragma unroll
      for (int e = 0; e < GV; ++e) acc[p * GV + e] = __builtin_fmaf(c, y[e], acc[p * GV + e]);
    }
  }
};

// A^T: pixel-driven gather for G = nh * m values per footprint.  One 16 x 16
// tile of the plan's fundamental domain per 256-thread block, views [v_begin,
// v_end).  `lds` holds nvc views x win bins (Staged).  Slot s = image * nh +
// symmetry; slots past nimg * nh repeat the last and write nothing.  Sums go
// to part[image * nx * ny + pixel] (FP64) or img.  P gives the basis: its bin
// window of a tile, records, and footprints of a pixel in one view.
constexpr int kWinViews = 64;  // views whose bin windows are computed at a time

template <class P, int G>
__device__ __forceinline__ void bwd_group_tile(const typename P::Args& a, const SymPlan& sp, int nimg,
                                               const float* __restrict__ sino, float* __restrict__ img, int tile,
                                               float4* lds, int nvc, int win, int* win_lo, int* win_n, int v_begin,
                                               int v_end, double* __restrict__ part) {
  const Proj2DArgs& g = P::geo(a);
  constexpr int REC = P::kRec;
  const int tiles_x = (g.nx + kTile - 1) / kTile;
  const int txy = sp.tile ? sp.tile[tile] : ((tile / tiles_x) << 16 | (tile % tiles_x));
  const int ix0 = (txy & 0xffff) * kTile, iy0 = (txy >> 16) * kTile;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ix = ix0 + (threadIdx.x & (kTile - 1)), iy = iy0 + threadIdx.x / kTile;
  const bool inside = ix < g.nx && iy < g.ny, valid = inside && P::active(a, ix, iy);
  const float4* bins = reinterpret_cast<const float4*>(g.bins);
  const size_t nsino = (size_t)g.np * g.nu, npix = (size_t)g.nx * g.ny;
  const int nslot = sp.nh * nimg;
  const Staged<REC, G> st(lds, nvc * win);
  const typename P::Pixel px = P::pixel(a, ix, iy);
  unsigned rev = 0;  // slots whose bins run backwards
#pragma unroll
  for (int s = 0; s < G; ++s) rev |= (unsigned)SymOp::reverses(sp.op[min(s, nslot - 1) & (sp.nh - 1)]) << s;

  double acc[G];
#pragma unroll
  for (int s = 0; s < G; ++s) acc[s] = 0.0;
  for (int w0 = v_begin; w0 < v_end; w0 += kWinViews) {
    const int nw = min(kWinViews, v_end - w0);
    __syncthreads();  // the previous views' windows and records are read
    if ((int)threadIdx.x < nw) {
      int lo, n;
      P::window(a, g.views[w0 + threadIdx.x], ix0, iy0, &lo, &n, win);
      win_lo[threadIdx.x] = lo;
      win_n[threadIdx.x] = n;
    }
    for (int c0 = 0; c0 < nw; c0 += nvc) {
      const int nv = min(nvc, nw - c0);
      __syncthreads();
      for (int j = wv; j < nv; j += 4) {
        const int v = w0 + c0 + j, lo = win_lo[c0 + j], n = win_n[c0 + j];
        int row[G];  // sinogram row of each slot
#pragma unroll
        for (int s = 0; s < G; ++s) {
          const int sl = min(s, nslot - 1), k = sl >> sp.lg, h = sl & (sp.nh - 1);
          row[s] = k * g.np + (sp.view ? const_load(sp.view, v * sp.nh + h) : v);
        }
        for (int i = lane; i < n; i += 64) {
          const int u = lo + i;
          float4 rd[REC > 0 ? REC : 1];
#pragma unroll
          for (int k = 0; k < REC; ++k) rd[k] = bins[((size_t)v * g.nu + u) * REC + k];
          float y[G];
#pragma unroll
          for (int s = 0; s < G; ++s)
            y[s] = sino[(size_t)row[s] * g.nu + ((rev >> s) & 1 ? g.nu - 1 - u : u)];
#pragma unroll
          for (int k = 0; k < REC; ++k) st.rec[k * st.cap + j * win + i] = rd[k];
#pragma unroll
          for (int s = 0; s < G; ++s) y[s] = P::value(rd, y[s]);
          st.put(j * win + i, y);
        }
      }
      __syncthreads();
      if (!valid) continue;
      for (int j = 0; j < nv; ++j) {
        const ViewGeo vg = scalar_view(g.views, w0 + c0 + j);
        float accv[G];
#pragma unroll
        for (int s = 0; s < G; ++s) accv[s] = 0.0f;
        P::template view<G>(a, vg, px, st, j * win, win_lo[c0 + j], win_n[c0 + j], accv);
#pragma unroll
        for (int s = 0; s < G; ++s) acc[s] += (double)accv[s];
      }
    }
  }
  if (!inside) return;
  const unsigned own = sp.owner ? sp.owner[(size_t)tile * (kTile * kTile) + threadIdx.x] : 1u;
#pragma unroll
  for (int s = 0; s < G; ++s) {
    if (s >= nslot) continue;
    const int k = s >> sp.lg, h = s & (sp.nh - 1);
    if (!((own >> h) & 1)) continue;
    int qx, qy;
    P::image(a, sp.op[h], ix, iy, &qx, &qy);
    const double val = P::result(a, acc[s]);
    const size_t q = k * npix + (size_t)qy * g.nx + qx;
    if (part) part[q] = val;
    else img[q] = (float)val;
  }
}

// grid (tiles, view groups, image groups): view group k covers views
// [k vpg, (k + 1) vpg); with more than one group it writes FP64 partial images
// to part[(k * batch + image) * nx * ny + ...] for sum_parts_kernel.
template <class P, int G>
__device__ __forceinline__ void bwd_group_block(const typename P::Args& a, const SymPlan& sp, int m, int batch,
                                                const float* __restrict__ sino, float* __restrict__ img, int vpg,
                                                int nvc, int win, double* __restrict__ part) {
  extern __shared__ float4 bwd_lds[];
  __shared__ int win_lo[kWinViews], win_n[kWinViews];
  const Proj2DArgs& g = P::geo(a);
  const int k = blockIdx.y, img0 = blockIdx.z * m;
  const size_t npix = (size_t)g.nx * g.ny;
  const int v0 = k * vpg, v1 = min(g.np, v0 + vpg);
  bwd_group_tile<P, G>(a, sp, min(m, batch - img0), sino + (size_t)img0 * g.np * g.nu, img + img0 * npix, blockIdx.x,
                       bwd_lds, nvc, win, win_lo, win_n, v0, v1,
                       gridDim.y > 1 ? part + ((size_t)k * batch + img0) * npix : nullptr);
}

}  // namespace sgdct
