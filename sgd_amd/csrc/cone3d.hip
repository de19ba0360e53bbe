// cone3d.hip -- gfx950 kernels of the cone-beam projectors: B1 (layers/A_B1_3D.cu)
// and separable footprints SF-TR / SF-TT (layers/SF_projector.cu).
//
// The reference's value of voxel (ix, iy, iz) in detector cell (u, j) of view p
// factors into an in-plane part and an axial part (A_B1_3D.cu:95-305):
//     conv_p(u; ix, iy)  *  x * cfac_p(ix, iy, iz) * gamma_p(j; ix, iy, iz)
// conv is the 2-D B1 footprint of the (ix, iy) column (it does not depend on
// iz: the detector's u axis is in-plane), cfac = dx dy dz * path-length weight
// * inverse area of the voxel's axial trapezoid, gamma its overlap with row j.
// So per view A = (sum over columns of conv * Y), with
//     Y_p[c][j] = sum_iz x[iz][c] * cfac * gamma_j      (column c = iy*nx + ix)
// and each Y value is shared by the ~4-5 bins that see the column.  A runs as
//   axial_fwd_kernel   Y for a chunk of views (wave per column and view:
//                      lanes stage every voxel's trapezoid in LDS, then
//                      gather by detector row; deterministic)
//   conv_fwd_kernel    proj[p][j][u] = sum_c conv(u, c) Y[c][j] (wave per
//                      bin: the bin's strip walk of the 2-D A kernel, lanes
//                      over rows, no atomics)
// and A^T, which the reference does not provide (its back-projector multiplies
// by the zeroed output volume, A_B1_3D.cu:408, 436), as the exact transpose:
//   conv_bwd_kernel    Yb[c][j] = sum_u conv(u, c) proj[p][j][u]
//   axial_bwd_kernel   x[iz][c] += cfac * sum_j gamma_j Yb[c][j]
// Volumes are kept column-major (xT[c][iz]) inside, transposed on the way in
// and out, so a wave's voxel reads are contiguous.
//
// The separable-footprint projector (layers/SF_projector.cu:81-234) has the
// same structure: its u trapezoid (corners ix +- 1/2, iy +- 1/2) does not
// depend on iz, and its amplitude factors into an in-plane part
// (2 / trapezoid width) and an axial part (lsd^2 dx dy dz / (du dv r^2) times
// the inverse v-footprint area).  The kernels are templated on the model:
//   CONE_B1     B1 in-plane, axial trapezoid from x +- 1, rows [j, j+1),
//               gamma <= 1e-7 skipped (A_B1_3D.cu:300)
//   CONE_SF_TR  SF trapezoid in-plane, axial rectangle of the centre column,
//               cells centred on integers ([j - 1/2, j + 1/2], :209-216)
//   CONE_SF_TT  as SF_TR with an axial trapezoid from x +- 1/2 at iy
// For SF the view table is built with edges at half-integer detector
// coordinates, so "bin u" of the in-plane machinery is cell [u - 1/2, u + 1/2].
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "footprint.hpp"
#include "group2d.hpp"
#include "projector.hpp"
#include "sf2d_dev.hpp"

namespace sgdct {

// Columns taller than kMaxNz voxels are processed in chunks of kMaxNz (the
// axial forward stages a chunk's voxel records in LDS, the axial transpose
// holds a chunk's voxel sums in registers); detector rows are staged for the
// axial transpose in windows of kMaxNv.  Neither bounds nz or nv.
constexpr int kMaxNz = 512;
constexpr int kMaxNv = 512;
// The in-plane kernels give each wave RCW chunks of 64 detector rows, at most
// kAllRows (a grid dimension runs over the chunk groups).
constexpr int kAllRows = 8;
constexpr float kGammaEps = 1e-7f; // A_B1_3D.cu:300 skips gamma <= eps

enum ConeModel : int { CONE_B1 = 0, CONE_SF_TR = 1, CONE_SF_TT = 2 };

// Axial footprint of voxel iz in a column: sorted rows of its corners (B1:
// x index +- 1 at the column's iy, A_B1_3D.cu:133-137, 188-202; SF-TT:
// x +- 1/2, SF_projector.cu:136-141, 160-168; SF-TR: the centre column, a
// rectangle stored as v0 = v1, v2 = v3, :151-158) and the axial factor cf
// (B1: dx dy dz * path-length weight * 2 / widths, A_B1_3D.cu:209-210;
// SF: lsd^2 dx dy dz / (du dv r^2) / area, SF_projector.cu:193-198, 364).
struct AxialTrap {
  float v0, v1, v2, v3, cf;
  float i01, i23;  // 1 / (2 (v1 - v0)), 1 / (2 (v3 - v2)); 0 on a flat side
};

__device__ __forceinline__ float inv_or_zero(float w) { return w > 0.0f ? 0.5f * __builtin_amdgcn_rcpf(w) : 0.0f; }

struct ColumnAxial {
  float ka, kb;        // ldz / depth at the two x corners (SF-TR: both the centre)
  float ka_lo, kb_lo;  // their FP32 remainders: ka + ka_lo is the FP64 value
  float r2;            // |in-plane source -> centre|^2
};

template <int M>
__device__ __forceinline__ ColumnAxial column_axial(const Cone3DArgs& a, const ViewGeo& vg, int ix, int iy) {
  const double off = (M == CONE_B1) ? 1.0 : (M == CONE_SF_TT ? 0.5 : 0.0);
  const double wy = iy * a.g.dy + vg.w0y;
  const double wxa = (ix - off) * a.g.dx + vg.w0x, wxb = (ix + off) * a.g.dx + vg.w0x;
  const double wx = ix * a.g.dx + vg.w0x;
  // depth along the central axis = -cross(pu, X - p) / |pu|, so
  // ldz / depth = ldz |pu| / cross(p - X, pu) with |pu| = du
  const double num = a.ldz * a.du;
  const double ka = num * recip(vg.puy * wxa - vg.pux * wy);
  const double kb = num * recip(vg.puy * wxb - vg.pux * wy);
  ColumnAxial c;
  c.ka = (float)ka;
  c.kb = (float)kb;
  c.ka_lo = (float)(ka - (double)c.ka);
  c.kb_lo = (float)(kb - (double)c.kb);
  c.r2 = (float)(wx * wx + wy * wy);
  return c;
}

// Trapezoid of voxel zc (index offset from the column's middle) from the rows
// of its corners: a1, a2 at x corner a and z -+ 1/2, b1, b2 at corner b.
template <int M>
__device__ __forceinline__ AxialTrap trap_from_corners(const Cone3DArgs& a, const ColumnAxial& c, float zc, float a1,
                                                       float a2, float b1, float b2) {
  AxialTrap t;
  t.v0 = fminf(a1, b1);
  t.v3 = fmaxf(a2, b2);
  const float h1 = fmaxf(a1, b1), l2 = fminf(a2, b2);
  t.v1 = fminf(h1, l2);
  t.v2 = fmaxf(h1, l2);
  const float oz = zc * a.dz;
  if (M == CONE_B1) {
    // correctly rounded: with v_sqrt_f32 and v_rcp_f32 A^T's error grows by 3 to 5 %
    const float w = __builtin_sqrtf(__builtin_fmaf(oz * oz, 1.0f / c.r2, 1.0f));
    t.cf = a.cvol * w * 2.0f * __builtin_amdgcn_rcpf((t.v3 - t.v0) + (t.v2 - t.v1));
  } else {
    if (M == CONE_SF_TR) {  // a1 == b1, a2 == b2: a rectangle
      t.v1 = t.v0;
      t.v2 = t.v3;
    }
    const float area = (M == CONE_SF_TR) ? (t.v3 - t.v0) : 0.5f * ((t.v3 - t.v0) + (t.v2 - t.v1));
    t.cf = a.fac * __builtin_amdgcn_rcpf((c.r2 + oz * oz) * area);
  }
  t.i01 = inv_or_zero(t.v1 - t.v0);
  t.i23 = inv_or_zero(t.v3 - t.v2);
  return t;
}

// Corners as detector rows (A's staged records).
template <int M>
__device__ __forceinline__ AxialTrap voxel_trap(const Cone3DArgs& a, const ColumnAxial& c, int iz) {
  const float zc = (float)iz - 0.5f * (float)(a.nz - 1);
  const float a1 = __builtin_fmaf(c.ka, zc - 0.5f, a.vc), a2 = __builtin_fmaf(c.ka, zc + 0.5f, a.vc);
  const float b1 = __builtin_fmaf(c.kb, zc - 0.5f, a.vc), b2 = __builtin_fmaf(c.kb, zc + 0.5f, a.vc);
  return trap_from_corners<M>(a, c, zc, a1, a2, b1, b2);
}

// The same trapezoid with its corners relative to the integer row *k0 next
// to it.  As FP32 detector rows in the hundreds, corners carry up to ~6e-5
// rows of rounding, which A^T of white-noise rows reads (~8e-6 relative at
// 512^3 voxels / 768 rows); relative to k0, each corner is one fused
// multiply-add of the exact vc - k0 plus the slope's FP32 remainder, ~1e-7
// rows from exact.
template <int M>
__device__ __forceinline__ AxialTrap voxel_trap_rel(const Cone3DArgs& a, const ColumnAxial& c, int iz, int* k0) {
  const float zc = (float)iz - 0.5f * (float)(a.nz - 1);
  const float zl = zc - 0.5f;
  const int k = (int)floorf(__builtin_fmaf(c.ka, zl, a.vc));
  const float vk = a.vc - (float)k;  // exact: both are multiples of 1/2 below 2^23
  const float a1 = __builtin_fmaf(c.ka_lo, zl, __builtin_fmaf(c.ka, zl, vk));
  const float b1 = __builtin_fmaf(c.kb_lo, zl, __builtin_fmaf(c.kb, zl, vk));
  // the far corners are one slope further (zc + 1/2 = zl + 1)
  const float a2 = a1 + c.ka, b2 = b1 + c.kb;
  *k0 = k;
  return trap_from_corners<M>(a, c, zc, a1, a2, b1, b2);
}

// detector row j spans [j + row_off, j + row_off + 1)
template <int M>
__device__ __forceinline__ float row_off() {
  return M == CONE_B1 ? 0.0f : -0.5f;
}

// Overlap of [s, s+1) with the unit-height trapezoid (A_SF.cu:48-84 /
// A_B1_3D.cu:30-66), segment by segment: [s, s+1) clamped into each segment
// gives the overlap's ends (equal when they do not meet).  The sloped sides
// divide by their widths through the voxel's precomputed reciprocals, zero
// for a side of zero width, which never overlaps.
// A walk over adjacent rows carries the last upper edge on.
struct AxialWalk {
  float c0, c1, c2;  // the edge clamped into the three segments
  __device__ __forceinline__ void start(const AxialTrap& t, float s) {
    c0 = clamp3(s, t.v0, t.v1);
    c1 = clamp3(s, t.v1, t.v2);
    c2 = clamp3(s, t.v2, t.v3);
  }
  __device__ __forceinline__ float next(const AxialTrap& t, float e) {
    AxialWalk n;
    n.start(t, e);
    const float g0 = (n.c0 - c0) * (n.c0 + c0 - 2.0f * t.v0) * t.i01;
    const float g2 = (n.c2 - c2) * (2.0f * t.v3 - c2 - n.c2) * t.i23;
    const float g = g0 + (n.c1 - c1) + g2;
    *this = n;
    return g;
  }
};

__device__ __forceinline__ float trap_gamma(float s, const AxialTrap& t) {
  AxialWalk w;
  w.start(t, s);
  return w.next(t, s + 1.0f);
}

template <int M>
__device__ __forceinline__ bool keep_gamma(float gm) {
  return M == CONE_B1 ? gm > kGammaEps : gm == gm;
}

// Orders a wave's LDS accesses across lanes: LDS operations of one wave are
// performed in program order, so a compiler barrier at wavefront scope suffices.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// Y[pl][c][j] = sum_iz xT[c][iz] * cfac * gamma_j.  Block: 4 waves, one
// column each (each wave uses only its own LDS records); grid
// (ceil(ncol / 4), views in the chunk).  BIG (nz > kMaxNz): the column runs
// in chunks of kMaxNz voxels, the rows' sums added chunk by chunk.
// ---------------------------------------------------------------------------
// Dynamic LDS: per wave and voxel a record of kAxialFields floats (v0, v1,
// v2, v3, i01, i23, x * cf).  The odd stride puts the records of 64
// consecutive voxels on distinct banks, so a wave's rows (which read
// neighbouring voxels) do not conflict.
constexpr int kAxialFields = 7;

template <int M, bool BIG>
__global__ __launch_bounds__(256) void axial_fwd_kernel(Cone3DArgs a, int p0, const float* __restrict__ xT,
                                                        float* __restrict__ Y) {
  extern __shared__ float axial_lds[];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int zcap = BIG ? kMaxNz : a.nz;
  float* const R = axial_lds + (size_t)wv * kAxialFields * zcap;  // this wave's records
  const int ncol = a.g.nx * a.g.ny;
  const int c = blockIdx.x * 4 + wv, pl = blockIdx.y;
  const bool live = c < ncol;
  ColumnAxial ca{};
  if (live) ca = column_axial<M>(a, a.g.views[p0 + pl], c % a.g.nx, c / a.g.nx);
  float* yrow = Y + ((size_t)pl * ncol + c) * a.nv;
  // v3(iz) = vc + k (zc + 1/2), zc = iz - (nz - 1) / 2, with k = max(ka, kb)
  // above vc and min(ka, kb) below; it grows with iz (ka, kb > 0: voxels in
  // front of the source), so the first voxel reaching a row follows from that
  // line up to rounding, and the staged values settle it exactly
  const float ikhi = __builtin_amdgcn_rcpf(fmaxf(ca.ka, ca.kb)), iklo = __builtin_amdgcn_rcpf(fminf(ca.ka, ca.kb));
  const float zoff = 0.5f * (float)(a.nz - 1) - 0.5f;
  // voxels [z0, z1): stage their records, then add their share to every row
  auto chunk = [&](int z0, int z1, bool first) {
    if (live) {
      for (int iz = z0 + lane; iz < z1; iz += 64) {
        const AxialTrap t = voxel_trap<M>(a, ca, iz);
        float* const r = R + kAxialFields * (iz - z0);
        r[0] = t.v0;
        r[1] = t.v1;
        r[2] = t.v2;
        r[3] = t.v3;
        r[4] = t.i01;
        r[5] = t.i23;
        r[6] = xT[(size_t)c * a.nz + iz] * t.cf;
      }
    }
    __syncthreads();
    if (!live) return;
    for (int j = lane; j < a.nv; j += 64) {
      const float fj = (float)j + row_off<M>();
      // first voxel of the chunk whose footprint reaches row j
      const float est = __builtin_fmaf(fj - a.vc, fj >= a.vc ? ikhi : iklo, zoff);
      int lo = (int)fminf(fmaxf(ceilf(est), (float)z0), (float)z1);
      while (lo > z0 && R[kAxialFields * (lo - 1 - z0) + 3] >= fj) --lo;
      while (lo < z1 && R[kAxialFields * (lo - z0) + 3] < fj) ++lo;
      float acc = 0.0f;
      for (int iz = lo; iz < z1; ++iz) {
        const float* const r = R + kAxialFields * (iz - z0);
        if (!(r[0] < fj + 1.0f)) break;
        AxialTrap t;
        t.v0 = r[0];
        t.v1 = r[1];
        t.v2 = r[2];
        t.v3 = r[3];
        t.i01 = r[4];
        t.i23 = r[5];
        const float gm = trap_gamma(fj, t);
        if (keep_gamma<M>(gm)) acc = __builtin_fmaf(r[6], gm, acc);
      }
      if (first) yrow[j] = acc;
      else yrow[j] += acc;
    }
  };
  if (!BIG) {
    chunk(0, a.nz, true);
    return;
  }
  // every wave of the block reaches both barriers of every chunk
  for (int z0 = 0; z0 < a.nz; z0 += kMaxNz) {
    if (z0 > 0) __syncthreads();  // the previous chunk's reads come first
    chunk(z0, min(a.nz, z0 + kMaxNz), z0 == 0);
  }
}

// Column c under symmetry op.
__device__ __forceinline__ int image_column(const Proj2DArgs& g, int op, int c) {
  int qx, qy;
  SymOp::pixel(op, g.nx, g.ny, c % g.nx, c / g.nx, &qx, &qy);
  return qy * g.nx + qx;
}

// The same for the G views of a class at once: the trapezoids of (view, c) are
// staged once, with the voxel values of the G columns h c, and every overlap is
// formed once for G row sums.  Block: two columns of the class's first view,
// 128 threads each; grid (ceil(ncol / 2), classes in the pass).  nz <= kMaxNz.
// Dynamic LDS: per column and voxel 6 + G floats and one of padding to an odd
// stride.  Bound by the LDS reads of the records and, at G = 4, by the stores
// of Y.  256^3 voxels, 360 views, 512 x 384, classes of 4: A as a whole 40.0 ->
// 20.5 ms against one view at a time.
template <int M, int G>
__global__ __launch_bounds__(256) void axial_fwd_group_kernel(Cone3DArgs a, int p0, const float* __restrict__ xT,
                                                              float* __restrict__ Y) {
  extern __shared__ float axial_lds[];
  constexpr int F = (6 + G) | 1;
  const int t = threadIdx.x & 127, half = threadIdx.x >> 7;
  float* const R = axial_lds + (size_t)half * F * a.nz;
  const int ncol = a.g.nx * a.g.ny;
  const int c = blockIdx.x * 2 + half, s0 = blockIdx.y * G;
  const bool live = c < ncol;
  ColumnAxial ca{};
  int col[G];
  if (live) {
    ca = column_axial<M>(a, a.g.views[a.slot_view[p0 + s0]], c % a.g.nx, c / a.g.nx);
#pragma unroll
    for (int h = 0; h < G; ++h) col[h] = image_column(a.g, a.op[h], c);
    for (int iz = t; iz < a.nz; iz += 128) {
      const AxialTrap tr = voxel_trap<M>(a, ca, iz);
      float* const r = R + F * iz;
      r[0] = tr.v0;
      r[1] = tr.v1;
      r[2] = tr.v2;
      r[3] = tr.v3;
      r[4] = tr.i01;
      r[5] = tr.i23;
#pragma unroll
      for (int h = 0; h < G; ++h) r[6 + h] = xT[(size_t)col[h] * a.nz + iz] * tr.cf;
    }
  }
  __syncthreads();
  if (!live) return;
  // first voxel that reaches a row, as in axial_fwd_kernel
  const float ikhi = __builtin_amdgcn_rcpf(fmaxf(ca.ka, ca.kb)), iklo = __builtin_amdgcn_rcpf(fminf(ca.ka, ca.kb));
  const float zoff = 0.5f * (float)(a.nz - 1) - 0.5f;
  for (int j = t; j < a.nv; j += 128) {
    const float fj = (float)j + row_off<M>();
    const float est = __builtin_fmaf(fj - a.vc, fj >= a.vc ? ikhi : iklo, zoff);
    int lo = (int)fminf(fmaxf(ceilf(est), 0.0f), (float)a.nz);
    while (lo > 0 && R[F * (lo - 1) + 3] >= fj) --lo;
    while (lo < a.nz && R[F * lo + 3] < fj) ++lo;
    float acc[G];
#pragma unroll
    for (int h = 0; h < G; ++h) acc[h] = 0.0f;
    for (int iz = lo; iz < a.nz; ++iz) {
      const float* const r = R + F * iz;
      if (!(r[0] < fj + 1.0f)) break;
      AxialTrap tr;
      tr.v0 = r[0];
      tr.v1 = r[1];
      tr.v2 = r[2];
      tr.v3 = r[3];
      tr.i01 = r[4];
      tr.i23 = r[5];
      const float gm = trap_gamma(fj, tr);
      if (keep_gamma<M>(gm)) {
#pragma unroll
        for (int h = 0; h < G; ++h) acc[h] = __builtin_fmaf(r[6 + h], gm, acc[h]);
      }
    }
#pragma unroll
    for (int h = 0; h < G; ++h)
      if (a.slot_view[p0 + s0 + h] >= 0) Y[((size_t)(s0 + h) * ncol + col[h]) * a.nv + j] = acc[h];
  }
}

// ---------------------------------------------------------------------------
// In-plane kernels.  Their weights do not depend on the detector row, so lanes
// cover the rows (RCW chunks of 64 per wave) where row profiles are read and
// added up, and pairs (column, bin) where the weights are evaluated: one
// evaluation gives up to 64 weights, which the row loop then reads lane by
// lane into scalar registers.
// ---------------------------------------------------------------------------
// SF in-plane weight of cell u for pixel (ix, iy): area of the pixel's unit
// trapezoid over the cell times 2 / (sum of its widths), from the corner
// projections relative to edge u, -N_u(c) / beta(c) (SF_projector.cu:123-133,
// 175-190, 193-198, 209-214).
__device__ __forceinline__ float sf_cell_weight(const ViewGeo& vg, const Proj2DArgs& g, int u, int ix, int iy) {
  const double wx = ix * g.dx + vg.w0x, wy = iy * g.dy + vg.w0y;
  const double ex = vg.e0x + u * vg.pux, ey = vg.e0y + u * vg.puy;
  const float nc = (float)(ex * wy - ey * wx);
  const float bc = (float)(vg.pux * wy - vg.puy * wx);
  const float hx = (float)(-0.5 * ey * g.dx), hy = (float)(0.5 * ex * g.dy);      // N_u steps
  const float bx = (float)(-0.5 * vg.puy * g.dx), by = (float)(0.5 * vg.pux * g.dy);  // beta steps
  const float q0 = -(nc - hx - hy) / (bc - bx - by);
  const float q1 = -(nc - hx + hy) / (bc - bx + by);
  const float q2 = -(nc + hx - hy) / (bc + bx - by);
  const float q3 = -(nc + hx + hy) / (bc + bx + by);
  const Trap t = sorted_trap(q0, q1, q2, q3);
  const float width = (t.q3 - t.q0) + (t.q2 - t.q1);
  const float gm = trap_gamma(t, 0.0f, 1.0f);
  return width > 0.0f ? gm * 2.0f / width : 0.0f;
}

// Lane `l`'s value, wave-uniform (l too).
__device__ __forceinline__ float lane_value(float x, int l) {
  return __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(x), l));
}

// min / max over each group of four lanes
__device__ __forceinline__ int quad_min(int x) {
  x = min(x, __builtin_amdgcn_mov_dpp(x, 0xB1, 0xf, 0xf, true));   // lanes 1 0 3 2
  return min(x, __builtin_amdgcn_mov_dpp(x, 0x4E, 0xf, 0xf, true));  // lanes 2 3 0 1
}
__device__ __forceinline__ int quad_max(int x) {
  x = max(x, __builtin_amdgcn_mov_dpp(x, 0xB1, 0xf, 0xf, true));
  return max(x, __builtin_amdgcn_mov_dpp(x, 0x4E, 0xf, 0xf, true));
}

// proj[p][j][u] = sum over the columns c of bin u's strip of conv(u, c) Y[c][j].
// A workgroup of four waves takes kFwdBins adjacent bins of one view; wave w
// walks the lines m = w mod 4 of their strips (the 2-D A's walk), and the
// waves' FP64 sums are added in wave order through LDS.  Per line the wave
// finds the columns that its four strips cover together, requests the row
// profiles of the first kFwdCols of them, and evaluates the weights meanwhile
// (lane = 4 column + bin); a column's profile is read once for the bins it
// touches, and a bin takes only columns of its own strip.  Grid: ceil(nu / 4) *
// nview blocks, view = blockIdx % nview (consecutive blocks, which the
// dispatcher spreads over the XCDs, take different views; the blocks of one
// view share an XCD's L2 when nview is 8).
constexpr int kFwdBins = 4, kFwdCols = 4;

template <int M, int RCW>
__global__ __launch_bounds__(256) void conv_fwd_kernel(Cone3DArgs a, int p0, int nview, const float* __restrict__ Y,
                                                       float* __restrict__ proj) {
  __shared__ double red[2][kFwdBins][RCW][64];
  const Proj2DArgs& g = a.g;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kc0 = blockIdx.y * RCW;  // this wave's detector-row chunks
  const int pl = blockIdx.x % nview, u0 = (blockIdx.x / nview) * kFwdBins;
  const int lb = lane & (kFwdBins - 1), lt = lane / kFwdBins;  // this lane's bin and column of a weight evaluation
  const bool live = u0 + lb < g.nu;
  const int u = live ? u0 + lb : g.nu - 1;
  const int v = slot_view(a, p0 + pl);
  if (v < 0) return;  // the whole workgroup
  const int ncol = g.nx * g.ny;
  const ViewGeo vg = g.views[v];
  B1Bin rec{};
  if (M == CONE_B1) rec = reinterpret_cast<const B1Bin*>(g.bins)[(size_t)v * g.nu + u];

  const double eax = vg.e0x + u * vg.pux, eay = vg.e0y + u * vg.puy;
  const double ebx = eax + vg.pux, eby = eay + vg.puy;
  // walk direction from the bins' middle ray (uniform over the workgroup)
  const double um = u0 + 0.5 * min(kFwdBins, g.nu - u0);
  const double mx = vg.e0x + um * vg.pux, my = vg.e0y + um * vg.puy;
  const bool rows = fabs(my) >= fabs(mx);
  const double acx = -eay * g.dx, acy = eax * g.dy, ac0 = eax * vg.w0y - eay * vg.w0x;
  const double bcx = -eby * g.dx, bcy = ebx * g.dy, bc0 = ebx * vg.w0y - eby * vg.w0x;
  // clamped end bins (A_B1_3D.cu:150-151, as in the 2-D kernel); SF drops
  // cells outside the detector instead
  const bool clamp = M == CONE_B1;
  const double lax = (clamp && u == 0) ? eax - vg.pux : eax, lay = (clamp && u == 0) ? eay - vg.puy : eay;
  const double lbx = (clamp && u == g.nu - 1) ? ebx + vg.pux : ebx;
  const double lby = (clamp && u == g.nu - 1) ? eby + vg.puy : eby;
  const double qcx = -lay * g.dx, qcy = lax * g.dy, qc0 = lax * vg.w0y - lay * vg.w0x;
  const double rcx = -lby * g.dx, rcy = lbx * g.dy, rc0 = lbx * vg.w0y - lby * vg.w0x;
  const double ra = g.h * (fabs(qcx) + fabs(qcy)), rb = g.h * (fabs(rcx) + fabs(rcy));
  const double sa = rows ? acx : acy, ma = rows ? acy : acx;
  const double sb = rows ? bcx : bcy, mb = rows ? bcy : bcx;
  const double sq = rows ? qcx : qcy, mq = rows ? qcy : qcx;
  const double sr = rows ? rcx : rcy, mr = rows ? rcy : rcx;
  const int nmin = rows ? g.nx : g.ny, nmaj = rows ? g.ny : g.nx;
  const int smin = rows ? 1 : g.nx, smaj = rows ? g.nx : 1;

  int m_lo, m_hi;
  strip_lines(sq, mq, -ra - qc0, sr, mr, rb - rc0, 0.0, (double)(nmin - 1), nmaj, &m_lo, &m_hi);
  if (!live) m_lo = nmaj, m_hi = -1;
  double lo0 = 0.0, lo1 = 0.0, hi0 = nmin - 1, hi1 = 0.0;
  if (sq > 0.0 && sr > 0.0) {
    lo0 = (-ra - qc0) / sq; lo1 = -mq / sq; hi0 = (rb - rc0) / sr; hi1 = -mr / sr;
  } else if (sq < 0.0 && sr < 0.0) {
    hi0 = (-ra - qc0) / sq; hi1 = -mq / sq; lo0 = (rb - rc0) / sr; lo1 = -mr / sr;
  }
  const double an = (double)rec.ka * sa, am = (double)rec.ka * ma, a0 = (double)rec.ka * ac0;
  const double bn = (double)rec.kb * sb, bm = (double)rec.kb * mb, b0 = (double)rec.kb * bc0;
  const int b_lo = __builtin_amdgcn_readfirstlane(quad_min(m_lo)), b_hi = __builtin_amdgcn_readfirstlane(quad_max(m_hi));

  double acc[kFwdBins][RCW];
#pragma unroll
  for (int b = 0; b < kFwdBins; ++b)
#pragma unroll
    for (int k = 0; k < RCW; ++k) acc[b][k] = 0.0;
  // Row-profile reads of a column: every lane loads (rows past nv read the
  // last row and are never stored), so the loads need no per-lane branch.
  const float* ybase = Y + (size_t)pl * ncol * a.nv;
  int joff[RCW];
#pragma unroll
  for (int k = 0; k < RCW; ++k) joff[k] = min((kc0 + k) * 64 + lane, a.nv - 1);
  for (int m = b_lo + ((wv - b_lo) & 3); m <= b_hi; m += 4) {
    // this lane's bin: columns [n0, n1] of line m
    int n0 = (int)fmax(ceil(fma((double)m, lo1, lo0)), 0.0);
    int n1 = (int)fmin(floor(fma((double)m, hi1, hi0)), (double)(nmin - 1));
    if (m < m_lo || m > m_hi || n0 > n1) n0 = 0x7fffffff, n1 = -1;
    const int c_lo = __builtin_amdgcn_readfirstlane(quad_min(n0)), c_hi = __builtin_amdgcn_readfirstlane(quad_max(n1));
    if (c_lo > c_hi) continue;
    float accl[kFwdBins][RCW];
#pragma unroll
    for (int b = 0; b < kFwdBins; ++b)
#pragma unroll
      for (int k = 0; k < RCW; ++k) accl[b][k] = 0.0f;
    float w = 0.0f;
    for (int c0 = c_lo; c0 <= c_hi; c0 += kFwdCols) {
      float y[kFwdCols][RCW];
#pragma unroll
      for (int i = 0; i < kFwdCols; ++i) {
        const float* yc = ybase + (size_t)(m * smaj + min(c0 + i, c_hi) * smin) * a.nv;
#pragma unroll
        for (int k = 0; k < RCW; ++k) y[i][k] = yc[joff[k]];
      }
      if (((c0 - c_lo) & (64 / kFwdBins - 1)) == 0) {  // weights of the next 16 columns
        const int n = c0 + lt;
        w = 0.0f;
        if (n >= n0 && n <= n1) {
          if (M == CONE_B1) {
            const float ta = (float)fma((double)n, an, fma((double)m, am, a0));
            const float tb = (float)fma((double)n, bn, fma((double)m, bm, b0));
            w = b1_mean(rec, ta, tb) * rec.scale;
          } else {
            w = sf_cell_weight(vg, g, u, rows ? n : m, rows ? m : n);
          }
        }
      }
      const int l0 = ((c0 - c_lo) & (64 / kFwdBins - 1)) * kFwdBins;
#pragma unroll
      for (int i = 0; i < kFwdCols; ++i) {
        if (c0 + i > c_hi) break;
#pragma unroll
        for (int b = 0; b < kFwdBins; ++b) {
          const float wb = lane_value(w, l0 + i * kFwdBins + b);
          if (wb != 0.0f) {
#pragma unroll
            for (int k = 0; k < RCW; ++k) accl[b][k] = __builtin_fmaf(wb, y[i][k], accl[b][k]);
          }
        }
      }
    }
#pragma unroll
    for (int b = 0; b < kFwdBins; ++b)
#pragma unroll
      for (int k = 0; k < RCW; ++k) acc[b][k] += (double)accl[b][k];
  }
  // waves 2, 3 onto 0, 1, then 1 onto 0
#pragma unroll
  for (int half = 2; half >= 1; half >>= 1) {
    if (wv >= half && wv < 2 * half) {
#pragma unroll
      for (int b = 0; b < kFwdBins; ++b)
#pragma unroll
        for (int k = 0; k < RCW; ++k) red[wv - half][b][k][lane] = acc[b][k];
    }
    __syncthreads();
    if (wv < half) {
#pragma unroll
      for (int b = 0; b < kFwdBins; ++b)
#pragma unroll
        for (int k = 0; k < RCW; ++k) acc[b][k] += red[wv][b][k][lane];
    }
    __syncthreads();
  }
  if (wv != 0) return;
  float* out = proj + (size_t)v * a.nv * g.nu + u0;
#pragma unroll
  for (int k = 0; k < RCW; ++k) {
    const int j = (kc0 + k) * 64 + lane;
    if (j >= a.nv) continue;
#pragma unroll
    for (int b = 0; b < kFwdBins; ++b)
      if (u0 + b < g.nu) out[(size_t)j * g.nu + b] = (float)acc[b][k];
  }
}

// Yb[pl][c][j] = sum_u conv(u, c) projT[pl][u][j], u over the column's clamped
// corner range (A_B1_3D.cu:117-151).  Wave per kBwdCols adjacent columns of a
// view: lane = 8 column + bin evaluates the weights of the first 8 bins of
// every column at once (further ones as the column's loop reaches them), then
// the columns take their bins' detector rows in turn, kBwdBins at a time.
constexpr int kBwdCols = 8, kBwdBins = 6;

template <int M, int RCW>
__global__ __launch_bounds__(256) void conv_bwd_kernel(Cone3DArgs a, int p0, const float* __restrict__ projT,
                                                       float* __restrict__ Yb) {
  const Proj2DArgs& g = a.g;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int ncol = g.nx * g.ny;
  const int col0 = __builtin_amdgcn_readfirstlane((blockIdx.x * 4 + wv) * kBwdCols), pl = blockIdx.y;
  const int kc0 = blockIdx.z * RCW;  // this wave's detector-row chunks
  const int v = slot_view(a, p0 + pl);
  if (col0 >= ncol || v < 0) return;
  const int lt = lane & 7, lc = min(col0 + lane / 8, ncol - 1);  // this lane's bin slot and column
  const int ix = lc % g.nx, iy = lc / g.nx;
  const ViewGeo& vg = g.views[v];
  const B1Bin* bins = M == CONE_B1 ? reinterpret_cast<const B1Bin*>(g.bins) + (size_t)v * g.nu : nullptr;
  const double wx = ix * g.dx + vg.w0x, wy = iy * g.dy + vg.w0y;
  const double n0 = vg.e0x * wy - vg.e0y * wx;
  const double be = vg.pux * wy - vg.puy * wx;
  const float bef = (float)be;
  const float kc = -(float)n0 * __builtin_amdgcn_rcpf(bef);
  const float gx = __builtin_fmaf(kc, vg.gx1, vg.gx0), gy = __builtin_fmaf(kc, vg.gy1, vg.gy0);
  const float hw = g.h * (__builtin_fabsf(gx) + __builtin_fabsf(gy)) * __builtin_amdgcn_rcpf(__builtin_fabsf(bef) - vg.db);
  const float last = (float)(g.nu - 1);
  const int ulo = (int)fminf(fmaxf(floorf(kc - hw), 0.0f), last);
  const int uhi = (int)fminf(fmaxf(floorf(kc + hw), 0.0f), last);
  auto weight = [&](int u) {
    float w = 0.0f;
    if (u <= uhi) {
      if (M == CONE_B1) {
        const B1Bin rec = bins[u];
        const float ta = rec.ka * (float)fma((double)u, be, n0), tb = rec.kb * (float)fma((double)(u + 1), be, n0);
        w = b1_mean(rec, ta, tb) * rec.scale;
      } else {
        w = sf_cell_weight(vg, g, u, ix, iy);
      }
    }
    return w;
  };
  const float w_first = weight(ulo + lt);
  // every lane loads (rows past nv read the last row and are never stored)
  const float* rows0 = projT + (size_t)pl * g.nu * a.nv;
  int joff[RCW];
#pragma unroll
  for (int k = 0; k < RCW; ++k) joff[k] = min((kc0 + k) * 64 + lane, a.nv - 1);
  const int ncols = min(kBwdCols, ncol - col0);
  for (int c = 0; c < ncols; ++c) {
    const int u0 = __builtin_amdgcn_readlane(ulo, 8 * c), u1 = __builtin_amdgcn_readlane(uhi, 8 * c);
    float acc[RCW];
#pragma unroll
    for (int k = 0; k < RCW; ++k) acc[k] = 0.0f;
    float w = w_first;
    int w0 = u0;  // bin of slot 0 of w
    for (int ub = u0; ub <= u1; ub += kBwdBins) {
      float y[kBwdBins][RCW];
#pragma unroll
      for (int i = 0; i < kBwdBins; ++i) {
        const float* row = rows0 + (size_t)min(ub + i, u1) * a.nv;
#pragma unroll
        for (int k = 0; k < RCW; ++k) y[i][k] = row[joff[k]];
      }
      if (ub > u0) {  // slots of this column's further bins
        w = weight(ub + lt);
        w0 = ub;
      }
#pragma unroll
      for (int i = 0; i < kBwdBins; ++i) {
        if (ub + i > u1) break;
        const float wi = lane_value(w, 8 * c + ub + i - w0);
#pragma unroll
        for (int k = 0; k < RCW; ++k) acc[k] = __builtin_fmaf(wi, y[i][k], acc[k]);
      }
    }
    float* out = Yb + ((size_t)pl * ncol + col0 + c) * a.nv;
#pragma unroll
    for (int k = 0; k < RCW; ++k)
      if ((kc0 + k) * 64 + lane < a.nv) out[(kc0 + k) * 64 + lane] = acc[k];
  }
}

// ---------------------------------------------------------------------------
// xT[c][iz] (+)= sum over the chunk's views of cfac * sum_j gamma_j Yb[c][j].
// Wave per column, lanes over voxels; grid ceil(ncol / 4).  Each view's row
// profile Yb[c][*] is copied into the wave's LDS with coalesced loads (the
// next view's loads are in flight meanwhile); the voxels then gather their
// rows from LDS.  BIG (nz > kMaxNz or nv > kMaxNv): the grid's y dimension
// takes the column's voxels in chunks of kMaxNz, and each view's profile is
// staged kMaxNv rows at a time.
// ---------------------------------------------------------------------------
template <int M, bool BIG>
__global__ __launch_bounds__(256) void axial_bwd_kernel(Cone3DArgs a, int p0, int nview, const float* __restrict__ Yb,
                                                        float* __restrict__ xT, int accumulate) {
  __shared__ float prof_lds[4][kMaxNv];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int ncol = a.g.nx * a.g.ny;
  const int c = blockIdx.x * 4 + wv;
  if (c >= ncol) return;  // waves share no LDS and meet at no block barrier
  float* const yl = prof_lds[wv];
  const int ix = c % a.g.nx, iy = c / a.g.nx;
  constexpr int kSlots = kMaxNz / 64, kRowSlots = kMaxNv / 64;
  const int z0 = BIG ? blockIdx.y * kMaxNz : 0;
  const int nwin = BIG ? (a.nv + kMaxNv - 1) / kMaxNv : 1;
  double acc[kSlots];
#pragma unroll
  for (int s = 0; s < kSlots; ++s) acc[s] = 0.0;
  float pre[kRowSlots];
  // window q = pl * nwin + w: rows [w kMaxNv, min(nv, (w + 1) kMaxNv)) of view pl
  auto fetch = [&](int q) {
    const int pl = BIG ? q / nwin : q, r0 = BIG ? (q - pl * nwin) * kMaxNv : 0;
    const float* yrow = Yb + ((size_t)pl * ncol + c) * a.nv + r0;
    const int nr = BIG ? min(kMaxNv, a.nv - r0) : a.nv;
#pragma unroll
    for (int k = 0; k < kRowSlots; ++k)
      if (k * 64 < nr) pre[k] = (k * 64 + lane < nr) ? yrow[k * 64 + lane] : 0.0f;
  };
  fetch(0);
  const float lastj = (float)(a.nv - 1);
  const int nq = nview * nwin;
  for (int q = 0; q < nq; ++q) {
    const int pl = BIG ? q / nwin : q, r0 = BIG ? (q - pl * nwin) * kMaxNv : 0;
    const int nr = BIG ? min(kMaxNv, a.nv - r0) : a.nv;
    wave_lds_sync();  // the previous window's reads come first
#pragma unroll
    for (int k = 0; k < kRowSlots; ++k)
      if (k * 64 + lane < nr) yl[k * 64 + lane] = pre[k];
    wave_lds_sync();
    if (q + 1 < nq) fetch(q + 1);
    const ColumnAxial ca = column_axial<M>(a, a.g.views[p0 + pl], ix, iy);
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      const int iz = z0 + s * 64 + lane;
      if (iz >= a.nz) continue;
      int k0;
      const AxialTrap t = voxel_trap_rel<M>(a, ca, iz, &k0);
      const float ro = row_off<M>();
      // rows relative to k0 (small integers plus ro: exact)
      int jlo = (int)fminf(fmaxf(floorf(t.v0 - ro) + (float)k0, 0.0f), lastj);
      int jhi = (int)fminf(fmaxf(floorf(t.v3 - ro) + (float)k0, 0.0f), lastj);
      if (BIG) {
        jlo = max(jlo, r0);
        jhi = min(jhi, r0 + nr - 1);
      }
      float sum = 0.0f;
      float sj = (float)(jlo - k0) + ro;
      AxialWalk walk;
      walk.start(t, sj);
      for (int j = jlo; j <= jhi; ++j) {
        sj += 1.0f;
        const float gm = walk.next(t, sj);
        if (keep_gamma<M>(gm)) sum = __builtin_fmaf(gm, yl[j - r0], sum);
      }
      acc[s] += (double)(t.cf * sum);
    }
  }
  float* out = xT + (size_t)c * a.nz;
#pragma unroll
  for (int s = 0; s < kSlots; ++s) {
    const int iz = z0 + s * 64 + lane;
    if (iz < a.nz) out[iz] = (float)((accumulate ? (double)out[iz] : 0.0) + acc[s]);
  }
}

// The same for the G columns h c of a column c of the fundamental domain: the
// trapezoid of (view, voxel) serves voxel h c of the views h v, whose row
// profiles are staged side by side (one 16-byte LDS read per row at G = 4).
// Block: 256 voxels of one column; grid (ndom, ceil(nz / 256)).  The next
// view's profiles are requested before the current view's rows are gathered.
// nv <= kGroupRows.  Bound by the reads of the profiles (1.6 GB per 16 views of
// the case above); A^T as a whole 34.3 -> 21.2 ms.
constexpr int kGroupRows = 512;

template <int M, int G>
__global__ __launch_bounds__(256) void axial_bwd_group_kernel(Cone3DArgs a, int p0, int nview,
                                                              const float* __restrict__ Yb, float* __restrict__ xT,
                                                              int accumulate) {
  extern __shared__ __attribute__((aligned(16))) float prof[];  // [nv][G]
  constexpr int kPre = (kGroupRows * G + 255) / 256;
  const int ncol = a.g.nx * a.g.ny;
  const int xy = a.dom[blockIdx.x], ix = xy & 0xffff, iy = xy >> 16;
  const unsigned own = a.own[blockIdx.x];
  const int iz = blockIdx.y * 256 + threadIdx.x;
  int col[G];
#pragma unroll
  for (int h = 0; h < G; ++h) col[h] = image_column(a.g, a.op[h], iy * a.g.nx + ix);
  double acc[G];
#pragma unroll
  for (int h = 0; h < G; ++h) acc[h] = 0.0;
  const int rows = a.nv;
  float pre[kPre];
  auto fetch = [&](int s) {
#pragma unroll
    for (int h = 0; h < G; ++h) {
      const int cls = s / G * G;
      const float* src = Yb + ((size_t)(cls + a.peer[(size_t)(p0 + s) * G + h]) * ncol + col[h]) * rows;
#pragma unroll
      for (int k = 0; k < kPre / G; ++k) {
        const int j = k * 256 + (int)threadIdx.x;
        pre[h * (kPre / G) + k] = j < rows ? src[j] : 0.0f;
      }
    }
  };
  auto next_slot = [&](int s) {
    while (s < nview && a.slot_view[p0 + s] < 0) ++s;
    return s;
  };
  const float lastj = (float)(rows - 1), ro = row_off<M>();
  int s = next_slot(0);
  if (s < nview) fetch(s);
  while (s < nview) {
    __syncthreads();  // the previous view's reads come first
#pragma unroll
    for (int k = 0; k < kPre / G; ++k) {
      const int j = k * 256 + (int)threadIdx.x;
      if (j < rows) {
#pragma unroll
        for (int h = 0; h < G; ++h) prof[j * G + h] = pre[h * (kPre / G) + k];
      }
    }
    __syncthreads();
    const int sn = next_slot(s + 1);
    if (sn < nview) fetch(sn);
    if (iz < a.nz) {
      const ColumnAxial ca = column_axial<M>(a, a.g.views[a.slot_view[p0 + s]], ix, iy);
      int k0;
      const AxialTrap tr = voxel_trap_rel<M>(a, ca, iz, &k0);
      // rows relative to k0 (small integers plus ro: exact)
      const int jlo = (int)fminf(fmaxf(floorf(tr.v0 - ro) + (float)k0, 0.0f), lastj);
      const int jhi = (int)fminf(fmaxf(floorf(tr.v3 - ro) + (float)k0, 0.0f), lastj);
      float sum[G];
#pragma unroll
      for (int h = 0; h < G; ++h) sum[h] = 0.0f;
      float sj = (float)(jlo - k0) + ro;
      AxialWalk walk;
      walk.start(tr, sj);
      for (int j = jlo; j <= jhi; ++j) {
        sj += 1.0f;
        const float gm = walk.next(tr, sj);
        if (keep_gamma<M>(gm)) {
          float y[G];
          __builtin_memcpy(y, __builtin_assume_aligned(prof + j * G, G < 4 ? 4 * G : 16), sizeof(y));
#pragma unroll
          for (int h = 0; h < G; ++h) sum[h] = __builtin_fmaf(gm, y[h], sum[h]);
        }
      }
#pragma unroll
      for (int h = 0; h < G; ++h) acc[h] += (double)(tr.cf * sum[h]);
    }
    s = sn;
  }
  if (iz >= a.nz) return;
#pragma unroll
  for (int h = 0; h < G; ++h) {
    if (!((own >> h) & 1)) continue;
    float* const out = xT + (size_t)col[h] * a.nz + iz;
    *out = (float)((accumulate ? (double)*out : 0.0) + acc[h]);
  }
}

// ---------------------------------------------------------------------------
// out[b][c][r] = in[map(b)][r][c] for a batch of rows x cols matrices (map null:
// the identity; an entry -1: nothing).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void transpose_kernel(const float* __restrict__ in, float* __restrict__ out,
                                                        int rows, int cols, const int* __restrict__ map) {
  __shared__ float tile[32][33];
  const int src = map ? map[blockIdx.z] : (int)blockIdx.z;
  if (src < 0) return;
  const size_t off = (size_t)blockIdx.z * rows * cols, in_off = (size_t)src * rows * cols;
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int k = ty; k < 32; k += 8) {
    const int r = r0 + k, c = c0 + tx;
    if (r < rows && c < cols) tile[k][tx] = in[in_off + (size_t)r * cols + c];
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const int c = c0 + k, r = r0 + tx;
    if (r < rows && c < cols) out[off + (size_t)c * rows + r] = tile[tx][k];
  }
}

hipError_t launch_transpose(const float* in, float* out, int rows, int cols, int batch, const int* map,
                            hipStream_t s) {
  dim3 grid((cols + 31) / 32, (rows + 31) / 32, batch);
  transpose_kernel<<<grid, dim3(256), 0, s>>>(in, out, rows, cols, map);
  return hipGetLastError();
}

// Chunks of 64 detector rows per wave of the in-plane kernels: at most
// kAllRows, as few as hold the rows of a group.
static int row_chunks(const Cone3DArgs& a) {
  const int groups = (a.nrc + kAllRows - 1) / kAllRows, per = (a.nrc + groups - 1) / groups;
  return (per + 1) / 2 * 2;
}

template <int M>
static void cone_forward_chunk(const Cone3DArgs& a, int p0, int nview, const float* xT, float* Y, float* proj,
                               hipStream_t s) {
  const int ncol = a.g.nx * a.g.ny;
  if (a.nh > 1) {
    const dim3 grid((ncol + 1) / 2, nview / a.nh);
    const size_t lds = sizeof(float) * 2 * ((6 + a.nh) | 1) * a.nz;
    if (a.nh == 2) axial_fwd_group_kernel<M, 2><<<grid, dim3(256), lds, s>>>(a, p0, xT, Y);
    else if (a.nh == 4) axial_fwd_group_kernel<M, 4><<<grid, dim3(256), lds, s>>>(a, p0, xT, Y);
    else if (M == CONE_SF_TR) axial_fwd_group_kernel<M, 8><<<grid, dim3(256), lds, s>>>(a, p0, xT, Y);
  } else {
    const size_t lds = sizeof(float) * 4 * kAxialFields * std::min(a.nz, kMaxNz);  // 4 waves
    if (a.nz > kMaxNz) axial_fwd_kernel<M, true><<<dim3((ncol + 3) / 4, nview), dim3(256), lds, s>>>(a, p0, xT, Y);
    else axial_fwd_kernel<M, false><<<dim3((ncol + 3) / 4, nview), dim3(256), lds, s>>>(a, p0, xT, Y);
  }
  const int groups = (a.nrc + kAllRows - 1) / kAllRows;
  const dim3 grid(((a.g.nu + kFwdBins - 1) / kFwdBins) * nview, groups);
  switch (row_chunks(a)) {
    case 2: conv_fwd_kernel<M, 2><<<grid, dim3(256), 0, s>>>(a, p0, nview, Y, proj); break;
    case 4: conv_fwd_kernel<M, 4><<<grid, dim3(256), 0, s>>>(a, p0, nview, Y, proj); break;
    case 6: conv_fwd_kernel<M, 6><<<grid, dim3(256), 0, s>>>(a, p0, nview, Y, proj); break;
    default: conv_fwd_kernel<M, 8><<<grid, dim3(256), 0, s>>>(a, p0, nview, Y, proj); break;
  }
}

template <int M>
static void cone_backward_chunk(const Cone3DArgs& a, int p0, int nview, const float* projT, float* Yb, float* xT,
                                int accumulate, hipStream_t s) {
  const int ncol = a.g.nx * a.g.ny;
  const int groups = (a.nrc + kAllRows - 1) / kAllRows;
  const dim3 cgrid((ncol + 4 * kBwdCols - 1) / (4 * kBwdCols), nview, groups);
  switch (row_chunks(a)) {
    case 2: conv_bwd_kernel<M, 2><<<cgrid, dim3(256), 0, s>>>(a, p0, projT, Yb); break;
    case 4: conv_bwd_kernel<M, 4><<<cgrid, dim3(256), 0, s>>>(a, p0, projT, Yb); break;
    case 6: conv_bwd_kernel<M, 6><<<cgrid, dim3(256), 0, s>>>(a, p0, projT, Yb); break;
    default: conv_bwd_kernel<M, 8><<<cgrid, dim3(256), 0, s>>>(a, p0, projT, Yb); break;
  }
  if (a.nh > 1) {
    const dim3 dgrid(a.ndom, (a.nz + 255) / 256);
    const size_t lds = sizeof(float) * a.nh * a.nv;
    if (a.nh == 2) axial_bwd_group_kernel<M, 2><<<dgrid, dim3(256), lds, s>>>(a, p0, nview, Yb, xT, accumulate);
    else if (a.nh == 4) axial_bwd_group_kernel<M, 4><<<dgrid, dim3(256), lds, s>>>(a, p0, nview, Yb, xT, accumulate);
    else if (M == CONE_SF_TR) axial_bwd_group_kernel<M, 8><<<dgrid, dim3(256), lds, s>>>(a, p0, nview, Yb, xT, accumulate);
    return;
  }
  const dim3 grid((ncol + 3) / 4, (a.nz + kMaxNz - 1) / kMaxNz);
  if (a.nv > kMaxNv || a.nz > kMaxNz)
    axial_bwd_kernel<M, true><<<grid, dim3(256), 0, s>>>(a, p0, nview, Yb, xT, accumulate);
  else
    axial_bwd_kernel<M, false><<<grid, dim3(256), 0, s>>>(a, p0, nview, Yb, xT, accumulate);
}

// Sizes the grouped axial kernels take.
bool cone_groups_fit(int nz, int nv) { return nz <= kMaxNz && nv <= kGroupRows; }

hipError_t launch_cone_forward_chunk(int model, const Cone3DArgs& a, int p0, int nview, const float* xT, float* Y,
                                     float* proj, hipStream_t s) {
  if (model == CONE_B1) cone_forward_chunk<CONE_B1>(a, p0, nview, xT, Y, proj, s);
  else if (model == CONE_SF_TR) cone_forward_chunk<CONE_SF_TR>(a, p0, nview, xT, Y, proj, s);
  else if (model == CONE_SF_TT) cone_forward_chunk<CONE_SF_TT>(a, p0, nview, xT, Y, proj, s);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_cone_backward_chunk(int model, const Cone3DArgs& a, int p0, int nview, const float* projT,
                                      float* Yb, float* xT, int accumulate, hipStream_t s) {
  if (model == CONE_B1) cone_backward_chunk<CONE_B1>(a, p0, nview, projT, Yb, xT, accumulate, s);
  else if (model == CONE_SF_TR) cone_backward_chunk<CONE_SF_TR>(a, p0, nview, projT, Yb, xT, accumulate, s);
  else if (model == CONE_SF_TT) cone_backward_chunk<CONE_SF_TT>(a, p0, nview, projT, Yb, xT, accumulate, s);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace sgdct
