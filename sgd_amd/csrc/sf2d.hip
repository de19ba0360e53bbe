// sf2d.hip -- separable-footprint (SF) fan-beam projector kernels, gfx950.
//
// SF footprint of layers/A_SF.cu:87-225: the four pixel corners (ix +- 1/2,
// iy +- 1/2) are projected to continuous detector coordinates and sorted into
// a trapezoid of unit height; the value for bin u is the trapezoid's area over
// [u, u+1) (gamma, layers/A_SF.cu:48-84) times dx / max(|sin t|, |cos t|),
// t the angle of the source->pixel-centre ray (layers/A_SF.cu:174-177).
//
// Corner projections are formed relative to an integer bin (a nearby edge)
// from the edge functions N_k, so they carry ~1e-7 bin of error instead of
// the ~6e-5 bin that absolute FP32 detector coordinates (up to nu) carry.
#include <hip/hip_runtime.h>

#include <cmath>

#include "sf2d_dev.hpp"

namespace sgdct {

hipError_t launch_sum_parts(const double* part, float* out, size_t n, int nparts, hipStream_t s);
hipError_t launch_interleave(const Proj2DArgs& g, const GroupRun& r, const float* img, hipStream_t s);

// A, launched as fwd_group_kernel.  Bound by VALU issue: 57 instructions per
// footprint, five of them reciprocals and roots at a quarter of the rate (two
// new corner projections, the merge of two sorted pairs, the trapezoid's area),
// and about as many per line, beside one multiply-add per value.  512 x 512,
// 720 views, 768 bins, per call: one value per footprint 1456 us, the scan's 8
// symmetries 215 us; 1024 x 1024, 900 views 7.04 -> 0.91 ms; 256 x 256, 90
// views, batch 5 266 -> 74 us; one value, 721 views from another start angle
// 1455 -> 1170 us.  (Line ends by FP64 divisions throughout, a four-value sort,
// compared ramps and the weight's reciprocal per pixel: 260, 1130, 84, 1418 us.)
// FAR: an image of 4 GiB and more (G = 1).
template <int G, int W, bool FAR>
__global__ __launch_bounds__(64 * W) void sf_fwd_kernel(Proj2DArgs g, SymPlan sp, int m, int batch,
                                                        const float* __restrict__ rows_img,
                                                        const float* __restrict__ cols_img, float* __restrict__ sino,
                                                        double* __restrict__ part) {
  __shared__ double red[W][G][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int rank = blockIdx.x / sp.nrep, rep = blockIdx.x - rank * sp.nrep;
  const int chunk = centre_out(rank, g.nchunk);
  const int v = sp.rep ? sp.rep[rep] : rep;
  const size_t gpix = (size_t)G * g.nx * g.ny;
  double acc[G];
#pragma unroll
  for (int s = 0; s < G; ++s) acc[s] = 0.0;
  sf_fwd_lines<G, FAR>(g, v, chunk, rows_img + blockIdx.y * gpix, cols_img ? cols_img + blockIdx.y * gpix : nullptr,
                       wv, W, blockIdx.z, gridDim.z, acc, sp.place);
#pragma unroll
  for (int s = 0; s < G; ++s) red[wv][s][lane] = acc[s];
  __syncthreads();
  const int u = chunk * 64 + lane;
  if (u >= g.nu) return;
  fwd_group_store<G, W>(g, sp, rep, v, u, m, batch, red, 1.0, 1.0, 1.0, sino, gridDim.z > 1 ? part : nullptr);
}

// A of one image in nseg line segments per bin, as fwd_lone_kernel.
__global__ __launch_bounds__(64 * kFwdWaves) void sf_lone_kernel(Proj2DArgs g, int nseg, const float* __restrict__ img,
                                                                 const float* __restrict__ cols_img,
                                                                 float* __restrict__ sino) {
  extern __shared__ double lone_red[];
  double(*const red)[64] = reinterpret_cast<double(*)[64]>(lone_red);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int rank = blockIdx.x / g.np, v = blockIdx.x - rank * g.np;
  const int chunk = centre_out(rank, g.nchunk);
  for (int k = wv; k < nseg; k += kFwdWaves) {
    double acc[1] = {0.0};
    sf_fwd_lines<1>(g, v, chunk, img, cols_img, 0, 1, k, nseg, acc);
    red[k][lane] = acc[0];
  }
  __syncthreads();
  const int u = chunk * 64 + lane;
  if (u < g.nu) fwd_lone_store(nseg, red, 1.0, 1.0, 1.0, sino + (size_t)v * g.nu + u);
}

// A^T, launched as bwd_group_kernel; same cases as above: 841 -> 154 us, 4.13
// -> 0.65 ms, 146 -> 50 us, 869 -> 683 us.  The FP64 projection of the pixel's
// centre and its sorted corners are formed once per view for all values, and
// each bin's area from one new edge (both edges per bin, and a double division
// per view: 174 us in the first case).
template <int G>
__global__ __launch_bounds__(256) void sf_bwd_kernel(Proj2DArgs g, SymPlan sp, int m, int batch,
                                                     const float* __restrict__ sino, float* __restrict__ img, int vpg,
                                                     int nvc, int win, double* __restrict__ part) {
  bwd_group_block<SfBwd, G>(g, sp, m, batch, sino, img, vpg, nvc, win, part);
}

// Tiles whose bin windows are too wide for LDS: sinogram values from global
// memory, one image and no symmetries.  grid (tiles x, tiles y, batch *
// ngroup).
__global__ __launch_bounds__(256) void sf_bwd_wide_kernel(Proj2DArgs g, const float* __restrict__ sino,
                                                          float* __restrict__ img, int ngroup, int vpg,
                                                          double* __restrict__ part) {
  const int k = blockIdx.z % ngroup, b = blockIdx.z / ngroup, batch = gridDim.z / ngroup;
  const size_t nimg = (size_t)g.nx * g.ny;
  const int v0 = k * vpg, v1 = min(g.np, v0 + vpg);
  sf_bwd_tile(g, sino + (size_t)b * g.np * g.nu, img + b * nimg, blockIdx.x, blockIdx.y, v0, v1,
              ngroup > 1 ? part + ((size_t)k * batch + b) * nimg : nullptr);
}

namespace {
template <int G, int W>
hipError_t sf_forward_g(const Proj2DArgs& g, const GroupRun& r, const float* img, float* sino, hipStream_t s) {
  const dim3 grid((unsigned)(r.sym.nrep * g.nchunk), (unsigned)r.groups(), (unsigned)r.split);
  const float* const rows = r.rows ? r.rows : img;
  if (G == 1 && (size_t)g.nx * g.ny >= (size_t)1 << 30)
    sf_fwd_kernel<1, W, true><<<grid, 64 * W, 0, s>>>(g, r.sym, r.m, r.batch, rows, r.cols, sino, r.part);
  else
    sf_fwd_kernel<G, W, false><<<grid, 64 * W, 0, s>>>(g, r.sym, r.m, r.batch, rows, r.cols, sino, r.part);
  return hipGetLastError();
}

template <int G>
hipError_t sf_backward_g(const Proj2DArgs& g, const GroupRun& r, const float* sino, float* img, hipStream_t s) {
  const dim3 grid((unsigned)r.sym.ntile, (unsigned)r.split, (unsigned)r.groups());
  sf_bwd_kernel<G><<<grid, 256, (size_t)r.nvc * r.win * 4 * G, s>>>(g, r.sym, r.m, r.batch, sino, img, r.vpg, r.nvc,
                                                                   r.win, r.part);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_sf_forward(const Proj2DArgs& g, const GroupRun& r, const float* img, float* sino, hipStream_t s) {
  if (r.split < 1 || (r.split > 1 && !r.part && !r.lone)) return hipErrorInvalidValue;
  hipError_t e = r.rows || r.cols ? launch_interleave(g, r, img, s) : hipSuccess;
  if (e != hipSuccess) return e;
  if (r.g == 1 && r.lone) {
    sf_lone_kernel<<<(unsigned)(g.np * g.nchunk), 64 * kFwdWaves, (size_t)r.split * 64 * sizeof(double), s>>>(
        g, r.split, img, r.cols, sino);
    return hipGetLastError();
  }
  if (r.g == 1) e = sf_forward_g<1, kFwdWaves>(g, r, img, sino, s);
  else if (r.g == 2) e = sf_forward_g<2, kFwdWaves>(g, r, img, sino, s);
  else if (r.g == 4) e = sf_forward_g<4, kFwdWaves>(g, r, img, sino, s);
  else if (r.g == 8) e = sf_forward_g<8, kFwdWaves>(g, r, img, sino, s);
  else return hipErrorInvalidValue;
  if (e == hipSuccess && r.split > 1 && r.sum) e = launch_sum_parts(r.part, sino, (size_t)r.batch * g.np * g.nu, r.split, s);
  return e;
}

hipError_t launch_sf_backward(const Proj2DArgs& g, const GroupRun& r, const float* sino, float* img, hipStream_t s) {
  if (r.split < 1 || (r.split > 1 && !r.part)) return hipErrorInvalidValue;
  hipError_t e;
  if (r.win == 0) {
    if (r.sym.nh != 1) return hipErrorInvalidValue;
    const dim3 grid((g.nx + kTile - 1) / kTile, (g.ny + kTile - 1) / kTile, (unsigned)(r.batch * r.split));
    sf_bwd_wide_kernel<<<grid, 256, 0, s>>>(g, sino, img, r.split, r.vpg, r.part);
    e = hipGetLastError();
  } else if (r.g == 1) {
    e = sf_backward_g<1>(g, r, sino, img, s);
  } else if (r.g == 2) {
    e = sf_backward_g<2>(g, r, sino, img, s);
  } else if (r.g == 4) {
    e = sf_backward_g<4>(g, r, sino, img, s);
  } else if (r.g == 8) {
    e = sf_backward_g<8>(g, r, sino, img, s);
  } else {
    return hipErrorInvalidValue;
  }
  if (e == hipSuccess && r.split > 1) e = launch_sum_parts(r.part, img, (size_t)r.batch * g.nx * g.ny, r.split, s);
  return e;
}

}  // namespace sgdct
