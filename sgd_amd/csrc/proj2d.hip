// proj2d.hip -- gfx950 kernels of the 2-D fan-beam footprint projectors.
//
//   fwd_group_kernel A   (image -> sinogram).  One lane per (view, bin): the
//                    lane walks the pixels of its bin's strip line by line and
//                    gathers sum_pixel conv * x for the G values (symmetric
//                    views x images, group2d.hpp) that share the footprint.
//                    No atomics, deterministic.
//   bwd_group_kernel A^T (sinogram -> image).  One lane per pixel, 16x16
//                    pixel tiles per workgroup; per-bin constants and the
//                    sinogram values of the bins the tile sees are staged in
//                    LDS, a few views at a time.  Deterministic gather.
//   sum_parts_kernel adds the FP64 partial results of split launches in a
//                    fixed order: A may split every bin's walk into grid
//                    segments and A^T the views into groups, so that a single
//                    image fills the GPU; the split is chosen per projector
//                    from one image's launch size.
//   interleave_kernel  the G-fold image A reads, and its transpose.
//   count_kernel     number of footprint evaluations under the reference's
//                    corner rule (the value layers/A_B1.cu:50,643 returns).
//
// Footprint values follow layers/A_B1.cu:62-208 (B1), layers/A_B0.cu:123-229
// (B0), layers/A_SF.cu:48-225 (SF); see footprint.hpp for the form used.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "proj2d_dev.hpp"
#include "symmetry.hpp"

namespace sgdct {

hipError_t launch_sum_parts(const double* part, float* out, size_t n, int nparts, hipStream_t s);

// A for G = nh * m values per footprint (group2d.hpp).  grid (nrep * nchunk,
// image groups, nseg): a workgroup of kFwdWaves waves takes one
// representative view and 64-bin chunk; its waves walk interleaved lines, so
// they stay level, and their FP64 sums are added in wave order through LDS
// (no partial sums in HBM).  With nseg > 1 every segment writes FP64 partial
// sums for sum_parts_kernel.
// Bound by VALU issue (62 % of it at the size below) and the vector L1, which
// feeds 4 G bytes per lane and footprint.  B1 at 512 x 512, 720 views, 768
// bins, per call: 960 us with one value per footprint and 24 partial sums,
// 178 us with the scan's 8 symmetries; 2048 x 2048, 1440 views, 3072 bins
// 44.6 -> 4.7 ms.  Eight waves: four 214 us (too few waves per view), sixteen
// 202 us (one workgroup per CU).  Column walks read the transposed copy, so
// that both walks read consecutive pixels (512 x 512, 721 views without
// symmetries, read in place 947 us, with the copy 782 us).
template <int BASIS, int G, int W>
__global__ __launch_bounds__(64 * W) void fwd_group_kernel(Proj2DArgs g, SymPlan sp, int m, int batch,
                                                           const float* __restrict__ rows_img,
                                                           const float* __restrict__ cols_img,
                                                           float* __restrict__ sino, double* __restrict__ part) {
  __shared__ double red[W][G][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int rank = blockIdx.x / sp.nrep, rep = blockIdx.x - rank * sp.nrep;
  const int chunk = centre_out(rank, g.nchunk);
  const int v = sp.rep ? sp.rep[rep] : rep;
  const size_t gpix = (size_t)G * g.nx * g.ny;
  double acc[G];
#pragma unroll
  for (int s = 0; s < G; ++s) acc[s] = 0.0;
  fwd_bin_lines<BASIS, G>(g, v, chunk, rows_img + blockIdx.y * gpix, cols_img ? cols_img + blockIdx.y * gpix : nullptr,
                          wv, W, blockIdx.z, gridDim.z, acc, sp.place);
#pragma unroll
  for (int s = 0; s < G; ++s) red[wv][s][lane] = acc[s];
  __syncthreads();
  const int u = chunk * 64 + lane;
  if (u >= g.nu) return;
  const typename Traits<BASIS>::Bin* bins = reinterpret_cast<const typename Traits<BASIS>::Bin*>(g.bins);
  fwd_group_store<G, W>(g, sp, rep, v, u, m, batch, red, g.dx, g.dy,
                        Traits<BASIS>::scale(bins[(size_t)v * g.nu + u]), sino, gridDim.z > 1 ? part : nullptr);
}

// A of one image in nseg line segments per bin, each summed by itself in line
// order and the segments in theirs (GroupRun::lone).  Same bounds as
// fwd_group_kernel; a wave's set-up serves its segments, and their sums stay in
// LDS (one segment per wave, its sums through HBM: B0 at 256 x 256, 360 views,
// 512 bins 131 -> 112 us, B1 at 400 x 380, 500 views, 700 bins 422 -> 395 us).
// grid (np * nchunk), nseg rows of 64 doubles of LDS.
template <int BASIS>
__global__ __launch_bounds__(64 * kFwdWaves) void fwd_lone_kernel(Proj2DArgs g, int nseg,
                                                                  const float* __restrict__ img,
                                                                  const float* __restrict__ cols_img,
                                                                  float* __restrict__ sino) {
  extern __shared__ double lone_red[];
  double(*const red)[64] = reinterpret_cast<double(*)[64]>(lone_red);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int rank = blockIdx.x / g.np, v = blockIdx.x - rank * g.np;
  const int chunk = centre_out(rank, g.nchunk);
  for (int k = wv; k < nseg; k += kFwdWaves) {
    double acc[1] = {0.0};
    fwd_bin_lines<BASIS, 1>(g, v, chunk, img, cols_img, 0, 1, k, nseg, acc);
    red[k][lane] = acc[0];
  }
  __syncthreads();
  const int u = chunk * 64 + lane;
  if (u >= g.nu) return;
  const typename Traits<BASIS>::Bin* bins = reinterpret_cast<const typename Traits<BASIS>::Bin*>(g.bins);
  fwd_lone_store(nseg, red, g.dx, g.dy, Traits<BASIS>::scale(bins[(size_t)v * g.nu + u]), sino + (size_t)v * g.nu + u);
}

// Interleaved copies of the images of one launch: slot s = image * nh + h of
// pixel p holds the image at h p, rows[(iy nx + ix) G + s], and transposed,
// cols[(ix ny + iy) G + s] (either null: not wanted).  grid (tiles x, tiles y, image
// groups), 16 x 16 pixels per block; slots past the last image hold zeros.
template <int G>
__global__ __launch_bounds__(256) void interleave_kernel(SymPlan sp, int nx, int ny, int m, int batch,
                                                         const float* __restrict__ img, float* __restrict__ rows,
                                                         float* __restrict__ cols) {
  const size_t npix = (size_t)nx * ny;
  const int img0 = blockIdx.z * m, nslot = sp.nh * min(m, batch - img0);
  float x[G];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int ix = blockIdx.x * 16 + tx, iy = blockIdx.y * 16 + ty;
  if (ix >= nx || iy >= ny) return;
#pragma unroll
  for (int s = 0; s < G; ++s) {
    x[s] = 0.0f;
    if (s < nslot) {
      const int k = s >> sp.lg, h = s & (sp.nh - 1);
      int qx, qy;
      SymOp::pixel(sp.op[h], nx, ny, ix, iy, &qx, &qy);
      x[s] = img[(img0 + k) * npix + (size_t)qy * nx + qx];
    }
  }
  if (rows) {
    rows += blockIdx.z * npix * G;
    __builtin_memcpy(__builtin_assume_aligned(rows + ((size_t)iy * nx + ix) * G, G < 4 ? 4 * G : 16), x, sizeof(x));
  }
  if (cols) {
    cols += blockIdx.z * npix * G;
    __builtin_memcpy(__builtin_assume_aligned(cols + ((size_t)ix * ny + iy) * G, G < 4 ? 4 * G : 16), x, sizeof(x));
  }
}

// out[i] = sum_k part[k n + i], k ascending (deterministic).
__global__ __launch_bounds__(256) void sum_parts_kernel(const double* __restrict__ part, float* __restrict__ out,
                                                        size_t n, int nparts) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    double acc = 0.0;
    for (int k = 0; k < nparts; ++k) acc += part[(size_t)k * n + i];
    out[i] = (float)acc;
  }
}


// Bin window that holds every tile's window over all views (host-side, on the
// host copy of the view table): the bound from the corner tiles, or, where
// that is above `enough`, every tile looked at (kNoWindow: there is none).
int max_tile_window(const Proj2DArgs& g, const ViewGeo* views_host, int enough) {
  const double half = 0.5 * (kTile - 1), r = half + (double)g.h;
  int w = window_bound(g, views_host, half * g.dx, half * g.dy, r * g.dx, r * g.dy);
  if (w <= enough || w == kNoWindow) return w;
  w = 0;
  for (int v = 0; v < g.np; ++v)
    for (int iy0 = 0; iy0 < g.ny; iy0 += kTile)
      for (int ix0 = 0; ix0 < g.nx; ix0 += kTile) {
        int lo, n;
        tile_window(g, views_host[v], ix0, iy0, &lo, &n, 1 << 30);
        w = n > w ? n : w;
      }
  return w;
}

// grid (tiles, view groups, image groups), bwd_group_block.  Bound by VALU
// issue and the LDS reads of records and values (64 bytes per footprint at G =
// 8).  B1 at 512 x 512, 720 views, 768 bins, per call: 940 us with one value
// per footprint, 197 us with the scan's 8 symmetries; 2048 x 2048, 1440 views,
// 3072 bins 29.3 -> 5.5 ms.
template <int BASIS, int G>
__global__ __launch_bounds__(256) void bwd_group_kernel(Proj2DArgs g, SymPlan sp, int m, int batch,
                                                        const float* __restrict__ sino, float* __restrict__ img,
                                                        int vpg, int nvc, int win, double* __restrict__ part) {
  bwd_group_block<FanBwd<BASIS>, G>(g, sp, m, batch, sino, img, vpg, nvc, win, part);
}

// Tiles whose bin windows are too wide for LDS: records read from global
// memory (L2), one image and no symmetries.  grid (tiles x, tiles y, batch *
// ngroup).
template <int BASIS>
__global__ __launch_bounds__(256, 8) void bwd_pix_kernel(Proj2DArgs g, const float* __restrict__ sino,
                                                         float* __restrict__ img, int ngroup, int vpg,
                                                         double* __restrict__ part) {
  const int k = blockIdx.z % ngroup, b = blockIdx.z / ngroup, batch = gridDim.z / ngroup;
  const size_t nimg = (size_t)g.nx * g.ny;
  const int v0 = k * vpg, v1 = min(g.np, v0 + vpg);
  bwd_pix_tile<BASIS, false>(g, sino + (size_t)b * g.np * g.nu, img + b * nimg, blockIdx.x, blockIdx.y, nullptr,
                             nullptr, v0, v1, ngroup > 1 ? part + ((size_t)k * batch + b) * nimg : nullptr);
}

// ---------------------------------------------------------------------------
// Evaluation count under the reference's clamped corner rule.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void count_kernel(Proj2DArgs g, unsigned long long* out) {
  __shared__ unsigned long long part[256];
  const int ix = blockIdx.x * 16 + (threadIdx.x & 15), iy = blockIdx.y * 16 + (threadIdx.x >> 4);
  unsigned long long c = 0;
  if (ix < g.nx && iy < g.ny) {
    for (int v = 0; v < g.np; ++v) {
      const ViewGeo& vg = g.views[v];
      double umin = 1e300, umax = -1e300;
      for (int k = 0; k < 4; ++k) {
        double fx = ix + ((k & 1) ? g.h : -g.h), fy = iy + ((k & 2) ? g.h : -g.h);
        double wx = fx * g.dx + vg.w0x, wy = fy * g.dy + vg.w0y;
        double uu = -(vg.e0x * wy - vg.e0y * wx) / (vg.pux * wy - vg.puy * wx);
        umin = fmin(umin, uu);
        umax = fmax(umax, uu);
      }
      int lo = (int)fmin(fmax(floor(umin), 0.0), (double)(g.nu - 1));
      int hi = (int)fmin(fmax(floor(umax), 0.0), (double)(g.nu - 1));
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

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
hipError_t launch_sum_parts(const double* part, float* out, size_t n, int nparts, hipStream_t s) {
  sum_parts_kernel<<<(unsigned)std::min<size_t>((n + 255) / 256, 4096), 256, 0, s>>>(part, out, n, nparts);
  return hipGetLastError();
}

namespace {
dim3 grid3(int x, int y, int z) { return dim3((unsigned)x, (unsigned)y, (unsigned)z); }

template <int G>
hipError_t interleave_g(const Proj2DArgs& g, const GroupRun& r, const float* img, hipStream_t s) {
  interleave_kernel<G><<<grid3((g.nx + 15) / 16, (g.ny + 15) / 16, r.groups()), 256, 0, s>>>(
      r.sym, g.nx, g.ny, r.m, r.batch, img, r.rows, r.cols);
  return hipGetLastError();
}

template <int BASIS, int G, int W>
hipError_t forward_g(const Proj2DArgs& g, const GroupRun& r, const float* img, float* sino, hipStream_t s) {
  const float* rows = r.rows ? r.rows : img;
  fwd_group_kernel<BASIS, G, W><<<grid3(r.sym.nrep * g.nchunk, r.groups(), r.split), 64 * W, 0, s>>>(
      g, r.sym, r.m, r.batch, rows, r.cols, sino, r.part);
  return hipGetLastError();
}

template <int BASIS, int G>
hipError_t backward_g(const Proj2DArgs& g, const GroupRun& r, const float* sino, float* img, hipStream_t s) {
  const size_t lds = (size_t)r.nvc * r.win * (32 + 4 * G);
  bwd_group_kernel<BASIS, G><<<grid3(r.sym.ntile, r.split, r.groups()), 256, lds, s>>>(
      g, r.sym, r.m, r.batch, sino, img, r.vpg, r.nvc, r.win, r.part);
  return hipGetLastError();
}

template <int BASIS>
hipError_t forward_b(const Proj2DArgs& g, const GroupRun& r, const float* img, float* sino, hipStream_t s) {
  switch (r.g) {
    case 1:
      if (r.lone) {
        fwd_lone_kernel<BASIS><<<(unsigned)(g.np * g.nchunk), 64 * kFwdWaves, (size_t)r.split * 64 * sizeof(double), s>>>(
            g, r.split, img, r.cols, sino);
        return hipGetLastError();
      }
      return forward_g<BASIS, 1, kFwdWaves>(g, r, img, sino, s);
    case 2: return forward_g<BASIS, 2, kFwdWaves>(g, r, img, sino, s);
    case 4: return forward_g<BASIS, 4, kFwdWaves>(g, r, img, sino, s);
    case 8: return forward_g<BASIS, 8, kFwdWaves>(g, r, img, sino, s);
    default: return hipErrorInvalidValue;
  }
}

template <int BASIS>
hipError_t backward_b(const Proj2DArgs& g, const GroupRun& r, const float* sino, float* img, hipStream_t s) {
  switch (r.g) {
    case 1: return backward_g<BASIS, 1>(g, r, sino, img, s);
    case 2: return backward_g<BASIS, 2>(g, r, sino, img, s);
    case 4: return backward_g<BASIS, 4>(g, r, sino, img, s);
    case 8: return backward_g<BASIS, 8>(g, r, sino, img, s);
    default: return hipErrorInvalidValue;
  }
}
}  // namespace

// The interleaved copies of the images of one launch (r.rows; r.cols too
// where the caller wants the transposed one).
hipError_t launch_interleave(const Proj2DArgs& g, const GroupRun& r, const float* img, hipStream_t s) {
  switch (r.g) {
    case 1: return interleave_g<1>(g, r, img, s);
    case 2: return interleave_g<2>(g, r, img, s);
    case 4: return interleave_g<4>(g, r, img, s);
    case 8: return interleave_g<8>(g, r, img, s);
    default: return hipErrorInvalidValue;
  }
}

// r.split > 1 needs r.part with split * batch * np * nu doubles.
hipError_t launch_forward(int basis, const Proj2DArgs& g, const GroupRun& r, const float* img, float* sino,
                          hipStream_t s) {
  if (r.split < 1 || (r.split > 1 && !r.part && !r.lone)) return hipErrorInvalidValue;
  hipError_t e = r.rows || r.cols ? launch_interleave(g, r, img, s) : hipSuccess;
  if (e != hipSuccess) return e;
  if (basis == BASIS_B1) e = forward_b<BASIS_B1>(g, r, img, sino, s);
  else if (basis == BASIS_B0) e = forward_b<BASIS_B0>(g, r, img, sino, s);
  else return hipErrorInvalidValue;
  if (e == hipSuccess && r.split > 1 && r.sum && !r.lone)
    e = launch_sum_parts(r.part, sino, (size_t)r.batch * g.np * g.nu, r.split, s);
  return e;
}

// r.split > 1 needs r.part with split * batch * nx * ny doubles; r.win = 0
// reads the records from global memory.
hipError_t launch_backward(int basis, const Proj2DArgs& g, const GroupRun& r, const float* sino, float* img,
                           hipStream_t s) {
  if (r.split < 1 || (r.split > 1 && !r.part)) return hipErrorInvalidValue;
  if (basis != BASIS_B1 && basis != BASIS_B0) return hipErrorInvalidValue;
  hipError_t e;
  if (r.win > 0) {
    e = basis == BASIS_B1 ? backward_b<BASIS_B1>(g, r, sino, img, s) : backward_b<BASIS_B0>(g, r, sino, img, s);
  } else {
    if (r.sym.nh != 1) return hipErrorInvalidValue;
    const dim3 grid = grid3((g.nx + kTile - 1) / kTile, (g.ny + kTile - 1) / kTile, r.batch * r.split);
    if (basis == BASIS_B1) bwd_pix_kernel<BASIS_B1><<<grid, 256, 0, s>>>(g, sino, img, r.split, r.vpg, r.part);
    else bwd_pix_kernel<BASIS_B0><<<grid, 256, 0, s>>>(g, sino, img, r.split, r.vpg, r.part);
    e = hipGetLastError();
  }
  if (e == hipSuccess && r.split > 1) e = launch_sum_parts(r.part, img, (size_t)r.batch * g.nx * g.ny, r.split, s);
  return e;
}

hipError_t launch_count(const Proj2DArgs& g, unsigned long long* out, hipStream_t s) {
  dim3 grid((g.nx + 15) / 16, (g.ny + 15) / 16), block(256);
  count_kernel<<<grid, block, 0, s>>>(g, out);
  return hipGetLastError();
}

}  // namespace sgdct

