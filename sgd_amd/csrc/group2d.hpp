// group2d.hpp -- plans and device helpers that let one footprint evaluation
// serve several images and several views of a 2-D projector.
//
// The footprint w(pixel, view, bin) does not depend on the image, and it is
// the same for congruent (pixel, view, bin): a symmetry h of the image grid
// (quarter turns and mirrors) that maps the set of views onto itself gives
//     w(h pixel, h view, h bin) = w(pixel, view, bin).
// A scan of np views over a full turn from angle 0 on a square image has 8
// such symmetries when 4 divides np, 4 when np is even, 2 when it is odd; a
// scan from any other start angle keeps its turns.  The kernels evaluate w
// once per (pixel, view, bin) class and apply it to G = nh * m values: nh
// symmetries and m images of a batch.  The footprint takes ~40 VALU
// instructions, each value one more multiply-add.
//   A    runs over one representative view per class and all pixels, on an
//        interleaved image xi[pixel][G] whose slot (h, k) holds image k at
//        h pixel; slot (h, k) of a lane's sums is output (h view, h bin).
//   A^T  runs over all views and the pixel tiles of a fundamental domain;
//        slot (h, k) of a bin's staged sinogram values is (h view, h bin) of
//        image k, and slot (h, k) of a lane's sums is pixel h pixel.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "projector.hpp"

namespace sgdct {

constexpr int kMaxSym = 8;   // symmetries of a square grid
constexpr int kMaxGroup = 8; // values per footprint evaluation

// A symmetry of the image grid: swap the axes (bit 0), then mirror x (bit 1)
// and y (bit 2).  An odd number of set bits reverses the detector's bins.
struct SymOp {
  enum : int { kSwap = 1, kFlipX = 2, kFlipY = 4 };
  __host__ __device__ static __forceinline__ bool reverses(int op) {
    return ((op ^ (op >> 1) ^ (op >> 2)) & 1) != 0;
  }
  // pixel (ix, iy) of an nx x ny grid (nx == ny where op swaps)
  __host__ __device__ static __forceinline__ void pixel(int op, int nx, int ny, int ix, int iy, int* ox, int* oy) {
    int x = (op & kSwap) ? iy : ix, y = (op & kSwap) ? ix : iy;
    if (op & kFlipX) x = nx - 1 - x;
    if (op & kFlipY) y = ny - 1 - y;
    *ox = x;
    *oy = y;
  }
  // pixel offset (iy nx + ix) of op (ix, iy): base + ix step_x + iy step_y
  struct Steps {
    int base, x, y;
  };
  __host__ __device__ static __forceinline__ Steps steps(int op, int nx, int ny) {
    const int sx = (op & kFlipX) ? -1 : 1, sy = (op & kFlipY) ? -nx : nx;
    return {((op & kFlipX) ? nx - 1 : 0) + ((op & kFlipY) ? (ny - 1) * nx : 0), (op & kSwap) ? sy : sx,
            (op & kSwap) ? sx : sy};
  }
  // point (ic, il) of a hexagonal lattice (odd rows hold nx - 1 points, half a
  // column on; their slot nx - 1 is no point and maps to such a slot).  A
  // vertical mirror keeps a row's parity only when ny is odd.
  __host__ __device__ static __forceinline__ void hex_point(int op, int nx, int ny, int ix, int iy, int* ox, int* oy) {
    const int n = nx - (iy & 1);
    *ox = (op & kFlipX) && ix < n ? n - 1 - ix : ix;
    *oy = (op & kFlipY) ? ny - 1 - iy : iy;
  }
  __host__ __device__ static __forceinline__ void point(int op, double x, double y, double* ox, double* oy) {
    const double a = (op & kSwap) ? y : x, b = (op & kSwap) ? x : y;
    *ox = (op & kFlipX) ? -a : a;
    *oy = (op & kFlipY) ? -b : b;
  }
};

// The symmetries a launch uses (device pointers; nh = 1 has the identity
// only and may leave every table null).  A launch of A may take some of the
// plan's symmetries only, nh of `row` from h0 on, where there is no room for
// the copies of all: a value's footprints and sums are the same in any launch.
struct SymPlan {
  int nh;                      // symmetries used (1, 2, 4 or 8)
  int lg;                      // log2(nh)
  int op[kMaxSym];             // op[0] = 0 where h0 = 0
  int h0, row;                 // A: first symmetry of the launch, symmetries of the plan
  int place;                   // A, one value per footprint: the symmetry at which the image is read in place
  int nrep;                    // A: representative views
  const int* rep;              // [nrep]
  const int* rep_view;         // [nrep][row] view h rep, -1 where an earlier h gives the same view
  const int* view;             // [np][nh] view h v (A^T)
  int ntile;                   // A^T: tiles of the fundamental domain
  const int* tile;             // [ntile] tile_y << 16 | tile_x
  const unsigned char* owner;  // [ntile][kTile * kTile] bit h: this lane writes pixel h p
};

// One launch of a grouped A or A^T on `batch` images, m images per group.
struct GroupRun {
  SymPlan sym;
  int g = 1;              // values per footprint, >= sym.nh * m (1, 2, 4 or 8)
  int m = 1, batch = 1;
  int split = 1;          // A: grid segments, A^T: view groups
  bool lone = false;      // A (g = 1): `split` line segments per bin, added within a workgroup
  double* part = nullptr; // FP64 partial sums (split > 1)
  bool sum = true;        // A: add the partial sums (false: a later launch writes more of them)
  float* rows = nullptr;  // A: interleaved images (null: g = 1, read in place)
  float* cols = nullptr;  // A: their transposes (null: column walks read strided)
  int vpg = 0;            // A^T: views per group
  int nvc = 0, win = 0;   // A^T: views and bins per view staged in LDS
  int groups() const { return (batch + m - 1) / m; }
};

// Waves of an A workgroup share one (view, 64-bin chunk): wave w walks the
// lines m = w mod kFwdWaves of every bin's strip, and the FP64 sums of the
// waves are added in wave order through LDS.
// In a lone run the waves walk whole segments line by line (wave w the segments
// w mod kFwdWaves) and the segments' sums are added in segment order.
constexpr int kFwdWaves = 8;

// The chunk a workgroup takes: centre chunks (whose strips are longest) first,
// so that the short edge strips fill the launch's tail.
__device__ __forceinline__ int centre_out(int rank, int n) {
  return (rank & 1) ? n / 2 - (rank + 1) / 2 : n / 2 + rank / 2;
}

}  // namespace sgdct
