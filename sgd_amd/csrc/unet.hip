// unet.hip -- gfx950 training and inference kernels of the warm-start U-Net.
//
// No reference counterpart (the reference's network code is a cuBLAS MLP,
// network.cu / layers/linear.cu; its Layer::forward/back_prop pattern,
// layers/layer.hh:15-16, is the closest precedent).  Activations are NHWC
// bfloat16, gradients of activations FP32, weights bfloat16 W[cout][9 cin]
// (tap-major: k = (3 ky + kx) cin + c) with an FP32 master copy.
//
//   conv3x3_halo_kernel  3x3 zero-padded convolution as an implicit GEMM on the
//                    matrix cores: v_mfma_f32_16x16x32_bf16, FP32 accumulate;
//                    a tile's pixel halo and weights staged in LDS for all nine
//                    taps.  Bias + ReLU fused; stores bf16, or FP32 for the
//                    input-gradient pass (which runs the same kernel on the
//                    output gradient with the flipped, transposed weights).
//                    conv3x3_lds_kernel and conv3x3_kernel (operands gathered
//                    per K step, from LDS or straight from L2) take the channel
//                    counts it does not.
//   wgrad_halo_kernel  dW[co][k] = sum_m dY[m][co] X[m + tap(k)][c(k)]: the
//                    pixel sum is the GEMM's K; a tile of dY and its halo of X
//                    are staged in LDS and read transposed; each block reduces a
//                    range of tiles into an FP32 partial, and a second kernel
//                    adds the partials in a fixed order.  wgrad_kernel gathers X
//                    per tap for other channel counts.
//   small kernels    input padding, 2x2 average pool, nearest upsample +
//                    concatenation and their adjoints, the 1x1 output head,
//                    MSE gradient, ReLU-mask + bf16 conversion, weight
//                    transpose, Adam.
#include <hip/hip_runtime.h>

#include <cstdint>

namespace sgdct {

typedef __bf16 bf16;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

struct ConvArgs {
  const bf16* in;      // [B][H][W][cin] (with in2: [B][H/2][W/2][c0])
  const bf16* w;       // [cout][9 cin]
  const float* bias;   // [cout] or null
  void* out;           // [B][H][W][cout], bf16 or FP32
  int B, H, W, cin, cout;
  int relu, out_f32;
  const bf16* mask;    // [B][H][W][cout] or null: out = value * (mask > 0)
  const bf16* in2;     // [B][H][W][cin - c0] or null (see conv_in)
  int c0;
  // Output as the gradient of a concatenation [upsample2(low), skip] (halo
  // kernel; null low_out: the plain output): channels [0, low_c) are summed
  // over 2 x 2 blocks, masked and stored in bf16, the others go to skip_out.
  bf16* low_out;          // [B][H/2][W/2][low_c]
  const bf16* low_mask;
  float* skip_out;        // [B][H][W][cout - low_c]
  int low_c;
};

// Address of the 8 input channels c .. c + 7 at pixel (b, y, x).  With in2 the
// input is the decoder's concatenation, read in place: channels [0, c0) are
// the half-resolution tensor `in` upsampled by nearest neighbour, channels
// [c0, cin) the full-resolution skip tensor in2 (c0 % 8 == 0, so a group of
// 8 never straddles the two).
__device__ __forceinline__ const bf16* conv_in(const bf16* in, const bf16* in2, int c0, int H, int W, int cin, int b,
                                               int y, int x, int c) {
  if (!in2) return in + (((size_t)b * H + y) * W + x) * cin + c;
  if (c < c0) return in + (((size_t)b * (H >> 1) + (y >> 1)) * (W >> 1) + (x >> 1)) * c0 + c;
  return in2 + (((size_t)b * H + y) * W + x) * (cin - c0) + (c - c0);
}

__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = (bf16)0.0f;
  return z;
}

// One 32-pixel x 32-channel wave tile per (wm, wn); block tile WM*32 x WN*32.
template <int WM, int WN>
__global__ __launch_bounds__(256) void conv3x3_kernel(ConvArgs a) {
  static_assert(WM * WN == 4, "four waves per block");
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int wm = wv % WM, wn = wv / WM;
  const long long M = (long long)a.B * a.H * a.W;
  const long long m_base = (long long)blockIdx.x * (WM * 32) + wm * 32;
  const int n_base = blockIdx.y * (WN * 32) + wn * 32;
  const int K = 9 * a.cin;
  const int r16 = lane & 15, g = lane >> 4;

  // pixel coordinates of the two A rows this lane loads
  int py[2], px[2], pb[2];
  bool pv[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const long long m = m_base + 16 * i + r16;
    pv[i] = m < M;
    const long long mm = pv[i] ? m : 0;
    px[i] = (int)(mm % a.W);
    const long long t = mm / a.W;
    py[i] = (int)(t % a.H);
    pb[i] = (int)(t / a.H);
  }
  int co[2];
  bool cv[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    co[j] = n_base + 16 * j + r16;
    cv[j] = co[j] < a.cout;
  }

  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  for (int k0 = 0; k0 < K; k0 += 32) {
    const int k = k0 + 8 * g;  // this lane's 8 consecutive k: one tap, 8 channels
    const bool kv = k < K;
    const int t = kv ? k / a.cin : 0, c = kv ? k - t * a.cin : 0;
    const int dy = t / 3 - 1, dx = t % 3 - 1;
    bf16x8 av[2], bv[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int yy = py[i] + dy, xx = px[i] + dx;
      if (kv && pv[i] && yy >= 0 && yy < a.H && xx >= 0 && xx < a.W)
        av[i] = *reinterpret_cast<const bf16x8*>(conv_in(a.in, a.in2, a.c0, a.H, a.W, a.cin, pb[i], yy, xx, c));
      else
        av[i] = zero8();
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (kv && cv[j])
        bv[j] = *reinterpret_cast<const bf16x8*>(a.w + (size_t)co[j] * K + k);
      else
        bv[j] = zero8();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], bv[j], acc[i][j], 0, 0, 0);
  }

  // D layout: lane holds rows 4 g + r (r = 0..3) of column r16
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (!cv[j]) continue;
    const float bias = a.bias ? a.bias[co[j]] : 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const long long m = m_base + 16 * i + 4 * g + r;
        if (m >= M) continue;
        float v = acc[i][j][r] + bias;
        if (a.relu) v = fmaxf(v, 0.0f);
        if (a.mask && !((float)a.mask[m * a.cout + co[j]] > 0.0f)) v = 0.0f;
        if (a.out_f32) static_cast<float*>(a.out)[m * a.cout + co[j]] = v;
        else static_cast<bf16*>(a.out)[m * a.cout + co[j]] = (bf16)v;
      }
  }
}

// ---------------------------------------------------------------------------
// LDS-tiled implicit GEMM for the same convolution (cout a multiple of 32).
// Block tile BM pixels x BN output channels, K in steps of 32 (k = tap-major,
// each 8-element group one tap and 8 channels since cin % 8 == 0).  Every
// K step the block stages A (BM x 32) and B (BN x 32) in LDS with 80-byte
// rows (16 bytes of padding: the 16-byte fragment reads of 8 consecutive rows
// then fall in distinct banks), double-buffered: the next step's global loads
// are in flight while the waves run their MFMAs on the current one, and one
// barrier per step separates the two buffers' uses.  Waves WM x WN, each
// (BM / WM) x (BN / WN) of MFMA 16x16x32 tiles.
// ---------------------------------------------------------------------------
constexpr int kLdsRow = 40;  // bf16 per LDS row: 32 + 8 padding

template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(256) void conv3x3_lds_kernel(ConvArgs a) {
  static_assert(WM * WN == 4, "four waves per block");
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;  // MFMA tiles per wave
  constexpr int AC = BM * 4 / 256;                     // A chunks (16 B) per thread
  constexpr int BC = (BN * 4 + 255) / 256;             // B chunks per thread (some idle if BN = 32)
  __shared__ __attribute__((aligned(16))) bf16 As[2][BM * kLdsRow];
  __shared__ __attribute__((aligned(16))) bf16 Bs[2][BN * kLdsRow];

  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int wm = wv % WM, wn = wv / WM;
  const long long M = (long long)a.B * a.H * a.W;
  const long long m_base = (long long)blockIdx.x * BM;
  const int n_base = blockIdx.y * BN;
  const int K = 9 * a.cin, nk = (K + 31) / 32;
  const int r16 = lane & 15, g = lane >> 4;

  // this thread's A chunks: row = q / 4, k group = q % 4, q = tid + 256 i
  int ay[AC], ax[AC], ab[AC];
  bool av_ok[AC];
#pragma unroll
  for (int i = 0; i < AC; ++i) {
    const int q = tid + 256 * i;
    const long long m = m_base + q / 4;
    av_ok[i] = m < M;
    const long long mm = av_ok[i] ? m : 0;
    ax[i] = (int)(mm % a.W);
    const long long t = mm / a.W;
    ay[i] = (int)(t % a.H);
    ab[i] = (int)(t / a.H);
  }

  bf16x8 ra[AC], rb[BC];
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < AC; ++i) {
      const int q = tid + 256 * i;
      const int k = k0 + 8 * (q & 3);
      bf16x8 v = zero8();
      if (av_ok[i] && k < K) {
        const int t = k / a.cin, c = k - t * a.cin;
        const int yy = ay[i] + t / 3 - 1, xx = ax[i] + t % 3 - 1;
        if (yy >= 0 && yy < a.H && xx >= 0 && xx < a.W)
          v = *reinterpret_cast<const bf16x8*>(conv_in(a.in, a.in2, a.c0, a.H, a.W, a.cin, ab[i], yy, xx, c));
      }
      ra[i] = v;
    }
#pragma unroll
    for (int i = 0; i < BC; ++i) {
      const int q = tid + 256 * i;
      const int n = q / 4, k = k0 + 8 * (q & 3);
      bf16x8 v = zero8();
      if (q < BN * 4 && n_base + n < a.cout && k < K)
        v = *reinterpret_cast<const bf16x8*>(a.w + (size_t)(n_base + n) * K + k);
      rb[i] = v;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < AC; ++i) {
      const int q = tid + 256 * i;
      *reinterpret_cast<bf16x8*>(&As[buf][(q / 4) * kLdsRow + 8 * (q & 3)]) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < BC; ++i) {
      const int q = tid + 256 * i;
      if (q < BN * 4) *reinterpret_cast<bf16x8*>(&Bs[buf][(q / 4) * kLdsRow + 8 * (q & 3)]) = rb[i];
    }
  };

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  load(0);
  store(0);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < nk) load((kt + 1) * 32);
    bf16x8 fa[TM], fb[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
      fa[i] = *reinterpret_cast<const bf16x8*>(&As[buf][(wm * (BM / WM) + 16 * i + r16) * kLdsRow + 8 * g]);
#pragma unroll
    for (int j = 0; j < TN; ++j)
      fb[j] = *reinterpret_cast<const bf16x8*>(&Bs[buf][(wn * (BN / WN) + 16 * j + r16) * kLdsRow + 8 * g]);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    if (kt + 1 < nk) store(buf ^ 1);
    __syncthreads();
  }

  // D layout: lane holds rows 4 g + r (r = 0..3) of column r16
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int co = n_base + wn * (BN / WN) + 16 * j + r16;
    if (co >= a.cout) continue;
    const float bias = a.bias ? a.bias[co] : 0.0f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const long long m = m_base + wm * (BM / WM) + 16 * i + 4 * g + r;
        if (m >= M) continue;
        float v = acc[i][j][r] + bias;
        if (a.relu) v = fmaxf(v, 0.0f);
        if (a.mask && !((float)a.mask[m * a.cout + co] > 0.0f)) v = 0.0f;
        if (a.out_f32) static_cast<float*>(a.out)[m * a.cout + co] = v;
        else static_cast<bf16*>(a.out)[m * a.cout + co] = (bf16)v;
      }
  }
}

// A block's run in conv3x3_halo_kernel: of items whose weights stay in LDS (one
// chunk, one block of output channels), of tiles whose halos stay for all blocks
// of output channels (one chunk), any.
enum HaloRun { kWeightsStay, kHaloStays, kAnyRun };

// v, with 0 where the activation is not positive
__device__ __forceinline__ bf16x8 relu_masked(const bf16* v, const bf16* act) {
  bf16x8 x = *reinterpret_cast<const bf16x8*>(v);
  const i16x8 m = __builtin_bit_cast(i16x8, *reinterpret_cast<const bf16x8*>(act));
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (!(__uint_as_float((unsigned)(unsigned short)m[e] << 16) > 0.0f)) x[e] = (bf16)0.0f;
  return x;
}

// ---------------------------------------------------------------------------
// Halo-tiled 3x3 convolution, the same implicit GEMM with its operands staged
// once per tile and input-channel chunk: a tile is TH x 16 output pixels x BN
// channels, and for each chunk of CC input channels the block stages in LDS the
// (TH + 2) x 18 pixel halo of the tile (80-byte pixel rows for CC = 32) and the
// chunk's BN x 9 x CC weights (rows of 9 CC + 8 bf16), from which every tap's A
// and B fragments are read.  Nine taps thus reuse one staged slab instead of
// re-gathering the tile's pixels per tap.  CC = 32 (cin % 32 == 0): a K step is
// one tap x 32 channels; CC = 16, 8 (cin == CC): a K step is 32 / CC taps (lane
// group g takes tap (32 / CC) s + 8 g / CC).  Wave (wm, wn) computes TM tile
// rows x TN 16-channel tiles.
//
// A block walks a run of items, tiles x blocks of output channels (run_halo).
// The next chunk's operands, or the next item's, are loaded into registers
// during the MFMAs, and the weights of a single chunk stay in LDS; each wave
// finishes its own rows through LDS of its own without a block barrier.  With
// an item per block the first chunk's load and the epilogue were not
// overlapped, as much as two chunks' work.  The K steps are unrolled, so that a
// step's fragments are read during the one before (one step at a time: the
// second figure).  8 x 512 x 512, 32 -> 32 channels: 93 -> 73 -> 65 us (268 MB),
// 96 -> 32: 167 -> 178 -> 163 us; 8 x 256 x 256, 64 -> 64: 86 -> 69 -> 61 us (630
// TF/s); 8 x 64 x 64, 256 -> 256: 62 -> 59 -> 50 us.  Bound by memory at 32
// channels, by the loads' latency and the barriers of a chunk beyond.
// ---------------------------------------------------------------------------
template <int TH, int BN, int WM, int WN, int CC, HaloRun RUN>
__global__ __launch_bounds__(256, 2) void conv3x3_halo_kernel(ConvArgs a) {
  static_assert(WM * WN == 4 && TH % (2 * WM) == 0, "four waves, whole pairs of tile rows per wave");
  constexpr int TW = 16, HH = TH + 2, HWD = TW + 2;
  constexpr int PS = CC == 32 ? 40 : CC;          // LDS pixel stride (bf16)
  constexpr int WR = 9 * CC + 8;                  // LDS weight row (bf16)
  constexpr int TM = TH / WM, TN = BN / WN / 16;  // MFMA tiles per wave
  constexpr int CW = 16 * TN, CG = CW / 8;        // a wave's channels; 16-byte groups of them
  constexpr int GP = CC / 8;                      // 16-byte groups per halo pixel / weight tap
  constexpr int NG = HH * HWD * GP;               // groups per halo
  constexpr int NW = BN * 9 * GP;                 // groups per weight slab
  constexpr int HC = (NG + 255) / 256, WC = (NW + 255) / 256;  // groups per thread
  constexpr int TPS = 32 / CC;                    // taps per K step
  constexpr int NKS = (9 + TPS - 1) / TPS;        // K steps per chunk
  constexpr int ES = CW + 8, FS = CW + 4;         // a wave's epilogue pixel rows (bf16, FP32)
  constexpr int EB = TW * FS * 2;                 // and tile row of them (bf16 units)
  static_assert(TM / 2 * 8 * ES <= EB && TW * ES <= EB, "the epilogue's tiles fit");
  __shared__ __attribute__((aligned(16))) bf16 halo[HH * HWD * PS];
  __shared__ __attribute__((aligned(16))) bf16 wts[BN * WR];
  __shared__ __attribute__((aligned(16))) bf16 etiles[4 * EB];

  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int wm = wv % WM, wn = wv / WM;
  const int r16 = lane & 15, g = lane >> 4;
  const int tiles_x = (a.W + TW - 1) / TW, tiles_y = (a.H + TH - 1) / TH;
  const int K = 9 * a.cin, nchunk = a.cin / CC, nblk = a.cout / BN;
  const int nitem = tiles_x * tiles_y * a.B * nblk, G = (int)gridDim.x;
  // tile * nblk + block of output channels; the blocks of an XCD (every 8th)
  // take neighbouring items
  int item = G % 8 == 0 ? blockIdx.x % 8 * (G / 8) + blockIdx.x / 8 : blockIdx.x;
  if (RUN == kHaloStays) item *= nblk;

  bf16x8 rh[HC], rw[WC];
  auto load_halo = [&](int it, int cc) {
    const int t = it / nblk, tx = t % tiles_x, rest = t / tiles_x, ty = rest % tiles_y, b = rest / tiles_y;
#pragma unroll
    for (int i = 0; i < HC; ++i) {
      const int q = tid + 256 * i, p = q / GP, cg = (q % GP) * 8;
      const int hy = p / HWD, hx = p - hy * HWD;
      const int iy = ty * TH + hy - 1, ix = tx * TW + hx - 1;
      bf16x8 v = zero8();
      if (q < NG && iy >= 0 && iy < a.H && ix >= 0 && ix < a.W)
        v = *reinterpret_cast<const bf16x8*>(conv_in(a.in, a.in2, a.c0, a.H, a.W, a.cin, b, iy, ix, cc * CC + cg));
      rh[i] = v;
    }
  };
  auto load_weights = [&](int it, int cc) {
    const int nb = it % nblk * BN;
#pragma unroll
    for (int i = 0; i < WC; ++i) {
      const int q = tid + 256 * i, n = q / (9 * GP), rem = q - n * (9 * GP);
      const int tp = rem / GP, cg = (rem - tp * GP) * 8;
      bf16x8 v = zero8();
      if (q < NW) v = *reinterpret_cast<const bf16x8*>(a.w + (size_t)(nb + n) * K + tp * a.cin + cc * CC + cg);
      rw[i] = v;
    }
  };

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // per-lane fragment bases: A at tile row wm TM, pixel r16, channels
  // (8 g) % CC; B at weight row wn CW + r16
  const bf16* const abase = &halo[((wm * TM) * HWD + r16) * PS + (8 * g) % CC];
  const bf16* const bbase = &wts[(wn * CW + r16) * WR + (8 * g) % CC];
  bf16* const etile = etiles + wv * EB;
  load_halo(item, 0);
  load_weights(item, 0);
  auto store_weights = [&]() {
#pragma unroll
    for (int i = 0; i < WC; ++i) {
      const int q = tid + 256 * i, n = q / (9 * GP), rem = q - n * (9 * GP);
      if (q < NW) *reinterpret_cast<bf16x8*>(&wts[n * WR + rem * 8]) = rw[i];
    }
  };
  if (RUN == kWeightsStay) store_weights();
  for (int next; item < nitem; item = next) {
    next = item + G;
    if (RUN == kHaloStays) next = item + 1 + (item % nblk + 1 < nblk ? 0 : (G - 1) * nblk);
    const bool new_halo = RUN != kHaloStays || item % nblk == 0;
    const int nb = item % nblk * BN;
    float bv[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) bv[j] = a.bias ? a.bias[nb + wn * CW + 16 * j + r16] : 0.0f;
    for (int cc = 0; cc < (RUN == kWeightsStay || RUN == kHaloStays ? 1 : nchunk); ++cc) {
      __syncthreads();  // the previous chunk's reads come first
      if (new_halo)
#pragma unroll
        for (int i = 0; i < HC; ++i) {
          const int q = tid + 256 * i, p = q / GP, cg = (q % GP) * 8;
          if (q < NG) *reinterpret_cast<bf16x8*>(&halo[p * PS + cg]) = rh[i];
        }
      if (RUN != kWeightsStay) store_weights();
      __syncthreads();
      const bool last = RUN == kWeightsStay || RUN == kHaloStays || cc + 1 == nchunk;
      if (!last || next < nitem) {
        const int it = last ? next : item, c = last ? 0 : cc + 1;
        if (RUN != kHaloStays || it % nblk == 0) load_halo(it, c);
        if (RUN != kWeightsStay) load_weights(it, c);
      }
#pragma unroll NKS
      for (int ks = 0; ks < NKS; ++ks) {
        // this lane's tap in K step ks and its halo offsets (0..2)
        const int tg = ks * TPS + (8 * g) / CC;
        const int dy = tg / 3, dx = tg - 3 * dy;
        const bool tv = tg < 9;
        const bf16* const ap = abase + (dy * HWD + dx) * PS;
        const bf16* const bp = bbase + tg * CC;
        bf16x8 fa[TM], fb[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[i] = tv ? *reinterpret_cast<const bf16x8*>(ap + i * HWD * PS) : zero8();
#pragma unroll
        for (int j = 0; j < TN; ++j) fb[j] = tv ? *reinterpret_cast<const bf16x8*>(bp + 16 * j * WR) : zero8();
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
      }
    }
    // D layout: lane holds pixels 4 g + r of tile row wm TM + i, channel r16
    const int tile = item / nblk, tx = tile % tiles_x, rest = tile / tiles_x, ty = rest % tiles_y, b = rest / tiles_y;
    const int x0 = tx * TW, y0 = ty * TH + wm * TM, co = nb + wn * CW;
    if (a.low_out && nb < a.low_c) {
      // 2 x 2 sums (low_c is a multiple of BN; tiles start at even pixels)
      const int H2 = a.H >> 1, W2 = a.W >> 1;
#pragma unroll
      for (int i = 0; i < TM; i += 2)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 4; r += 2)
            etile[(i / 2 * 8 + 2 * g + r / 2) * ES + 16 * j + r16] =
                (bf16)(acc[i][j][r] + acc[i][j][r + 1] + acc[i + 1][j][r] + acc[i + 1][j][r + 1]);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      for (int q = lane; q < TM / 2 * 8 * CG; q += 64) {
        const int p = q / CG, c8 = (q - p * CG) * 8;
        const int oy = (y0 >> 1) + p / 8, ox = (x0 >> 1) + p % 8;
        if (oy >= H2 || ox >= W2) continue;
        const long long o = (((long long)b * H2 + oy) * W2 + ox) * a.low_c + co + c8;
        *reinterpret_cast<bf16x8*>(a.low_out + o) = relu_masked(&etile[p * ES + c8], a.low_mask + o);
      }
    } else if (a.low_out || a.out_f32) {
      // FP32 output, a tile row at a time
      float* const out = a.low_out ? a.skip_out : static_cast<float*>(a.out);
      float* const ftile = reinterpret_cast<float*>(etile);
      const int c0 = a.low_out ? a.low_c : 0, C = a.cout - c0;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float v = acc[i][j][r] + bv[j];
            if (a.relu) v = fmaxf(v, 0.0f);
            ftile[(4 * g + r) * FS + 16 * j + r16] = v;
          }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int q = lane; q < TW * CW / 4; q += 64) {
          const int p = q / (CW / 4), c4 = (q - p * (CW / 4)) * 4;
          const int oy = y0 + i, ox = x0 + p;
          if (oy >= a.H || ox >= a.W) continue;
          const long long o = (((long long)b * a.H + oy) * a.W + ox) * C + co - c0 + c4;
          f32x4 v = *reinterpret_cast<const f32x4*>(&ftile[p * FS + c4]);
          if (a.mask)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (!((float)a.mask[o + e] > 0.0f)) v[e] = 0.0f;
          *reinterpret_cast<f32x4*>(out + o) = v;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
    } else {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float v = acc[i][j][r] + bv[j];
            if (a.relu) v = fmaxf(v, 0.0f);
            etile[(4 * g + r) * ES + 16 * j + r16] = (bf16)v;
          }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (lane < TW * CG) {
          const int p = lane / CG, c8 = (lane - p * CG) * 8;
          const int oy = y0 + i, ox = x0 + p;
          const long long o = (((long long)b * a.H + oy) * a.W + ox) * a.cout + co + c8;
          if (oy < a.H && ox < a.W)
            *reinterpret_cast<bf16x8*>(static_cast<bf16*>(a.out) + o) =
                a.mask ? relu_masked(&etile[p * ES + c8], a.mask + o)
                       : *reinterpret_cast<const bf16x8*>(&etile[p * ES + c8]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
}

// ---------------------------------------------------------------------------
// Weight gradient dW[co][k] = sum_m dY[m][co] X[m + tap(k)][c(k)]: a GEMM
// whose reduction runs over pixels m.  Block tile CO_T (co) x KT (k) with
// KT = 256 / CO_T * 16 ... 4 waves, each a 16-row co strip x 64 k (4 MFMA
// tiles).  The block walks its pixel range in chunks of 64.  The chunk's dY
// and X tiles are staged in LDS in their natural pixel-major layout
// ([pixel][channel], one 16-byte write per 8 channels), and gfx950's
// transposing LDS read (ds_read_b64_tr_b16) hands each lane the 8
// consecutive pixels of one channel that an MFMA fragment needs, as two
// 8-byte reads.  Within each 16-lane group that read gives lane i, value k,
// the 16-bit element i % 4 of the 8 bytes addressed by lane 4k + i / 4; so
// lane j addresses pixel row p0 + j / 4, channels c0 + 4 (j % 4) .. + 3.
// Row strides of 80 / 48 / 144 bf16 (160 / 96 / 288 bytes, 32 or 96 mod 128)
// put the 4 rows a 16-lane group reads in distinct banks.  Result ->
// partial[blockIdx.z] (pixel-range splits, added in a fixed order by
// reduce_partials_kernel).
// ---------------------------------------------------------------------------
struct WgradArgs {
  const bf16* x;    // [B][H][W][cin] (with x2: the concatenation, as ConvArgs::in2)
  const bf16* dy;   // [B][H][W][cout]
  float* partial;   // [nsplit][cout][9 cin]
  int B, H, W, cin, cout;
  long long pix_per_split;  // multiple of 64
  const bf16* x2;
  int c0;
  float* bias_partial;      // [nsplit][cout] column sums of dy, or null
};


// An MFMA fragment of 8 consecutive pixels of one channel from a
// pixel-major LDS tile: the transposing reads of pixel rows [p, p + 4) and
// [p + 4, p + 8) (p, c as addressed by this lane, see above).
__device__ __forceinline__ bf16x8 tr_fragment(const bf16* tile, int row, int col, int stride) {
  const lds_i16x4* p0 = (const lds_i16x4*)((__attribute__((address_space(3))) char*)tile +
                                           2 * (row * stride + col));
  const lds_i16x4* p1 = (const lds_i16x4*)((__attribute__((address_space(3))) char*)tile +
                                           2 * ((row + 4) * stride + col));
  const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(const_cast<lds_i16x4*>(p0));
  const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(const_cast<lds_i16x4*>(p1));
  const i16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8, v);
}

template <int CO_T>
__global__ __launch_bounds__(256) void wgrad_kernel(WgradArgs a) {
  static_assert(CO_T == 64 || CO_T == 32, "co tile 64 or 32");
  constexpr int WK = 64 / CO_T * 1;       // waves along k: 1 (CO_T 64) or 2 (CO_T 32)
  constexpr int KT = 64 * WK;             // k tile
  constexpr int SD = CO_T + 16, SX = KT + 16;  // LDS row strides (bf16)
  constexpr int DG = CO_T / 8, XG = KT / 8;    // 16-byte groups per pixel row
  constexpr int DC = 64 * DG / 256;       // dY groups per thread: 2 or 1
  constexpr int XC = 64 * XG / 256;       // X groups per thread: 2 or 4
  __shared__ __attribute__((aligned(16))) bf16 s_dy[64 * SD];  // [m][co]
  __shared__ __attribute__((aligned(16))) bf16 s_x[64 * SX];   // [m][k]
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int r16 = lane & 15, g = lane >> 4;
  const int wco = wv % (4 / WK), wk = wv / (4 / WK);  // this wave's co strip and k half
  const int K = 9 * a.cin;
  const int co0 = blockIdx.x * CO_T, k0 = blockIdx.y * KT;
  const long long M = (long long)a.B * a.H * a.W;
  const long long m_begin = (long long)blockIdx.z * a.pix_per_split;
  const long long m_end = m_begin + a.pix_per_split < M ? m_begin + a.pix_per_split : M;

  f32x4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // Each thread stages the same 8 k values (one tap t, channels c .. c + 7)
  // of X for XC pixels, pm = tid / XG + i (256 / XG), in every chunk; the
  // chunk's first pixel (b, y, x0) advances by 64 pixels per chunk.
  const int kx = k0 + (int)(threadIdx.x % XG) * 8;
  const int tap = kx / a.cin, cx = kx - tap * a.cin;
  const int oy = tap / 3 - 1, ox = tap % 3 - 1;
  const bool kin = kx < K;
  const int pmx = (int)threadIdx.x / XG;
  const long long hw = (long long)a.H * a.W;
  int cb = (int)(m_begin / hw);
  int cy = (int)((m_begin - cb * hw) / a.W);
  int cx0 = (int)(m_begin - cb * hw - (long long)cy * a.W);
  // Operands of one chunk in registers: the next chunk's loads are issued
  // before the current chunk's MFMAs and land in LDS after them.
  bf16x8 rd[DC], rx[XC];
  auto load = [&](long long m0) {
#pragma unroll
    for (int i = 0; i < DC; ++i) {
      const int q = threadIdx.x + 256 * i, pm = q / DG, cg = (q % DG) * 8;
      const long long m = m0 + pm;
      rd[i] = zero8();
      if (m < m_end && co0 + cg < a.cout) rd[i] = *reinterpret_cast<const bf16x8*>(a.dy + m * a.cout + co0 + cg);
    }
#pragma unroll
    for (int i = 0; i < XC; ++i) {
      const int pm = pmx + i * (256 / XG);
      rx[i] = zero8();
      if (kin && m0 + pm < m_end) {
        int x = cx0 + pm, y = cy, b = cb;
        while (x >= a.W) {
          x -= a.W;
          if (++y == a.H) {
            y = 0;
            ++b;
          }
        }
        const int yy = y + oy, xx = x + ox;
        if (yy >= 0 && yy < a.H && xx >= 0 && xx < a.W)
          rx[i] = *reinterpret_cast<const bf16x8*>(conv_in(a.x, a.x2, a.c0, a.H, a.W, a.cin, b, yy, xx, cx));
      }
    }
    // the chunk's first pixel moves on by 64
    cx0 += 64;
    while (cx0 >= a.W) {
      cx0 -= a.W;
      if (++cy == a.H) {
        cy = 0;
        ++cb;
      }
    }
  };
  // Bias gradient (the blocks of the first k tile): each thread sums the dY
  // values it stages, channels (tid % DG) * 8 .. + 7, in FP32.
  const bool bias = a.bias_partial && blockIdx.y == 0;
  float bs[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  if (m_begin < m_end) load(m_begin);
  for (long long m0 = m_begin; m0 < m_end; m0 += 64) {
    // stage: group q -> pixel pm = q / G, channels cg .. cg + 7, cg = (q % G) * 8
#pragma unroll
    for (int i = 0; i < DC; ++i) {
      const int q = threadIdx.x + 256 * i, pm = q / DG, cg = (q % DG) * 8;
      *reinterpret_cast<bf16x8*>(&s_dy[pm * SD + cg]) = rd[i];
      if (bias) {
        const i16x8 u = __builtin_bit_cast(i16x8, rd[i]);
#pragma unroll
        for (int e = 0; e < 8; ++e) bs[e] += __uint_as_float((unsigned)(unsigned short)u[e] << 16);
      }
    }
#pragma unroll
    for (int i = 0; i < XC; ++i) {
      const int pm = pmx + i * (256 / XG);
      *reinterpret_cast<bf16x8*>(&s_x[pm * SX + (threadIdx.x % XG) * 8]) = rx[i];
    }
    __syncthreads();
    if (m0 + 64 < m_end) load(m0 + 64);
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // two 32-pixel MFMA steps
      const int row = 32 * h + 8 * g + (r16 >> 2), col = 4 * (r16 & 3);
      const bf16x8 av = tr_fragment(s_dy, row, 16 * wco + col, SD);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bf16x8 bv = tr_fragment(s_x, row, 64 * wk + 16 * j + col, SX);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc[j], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  float* out = a.partial + (size_t)blockIdx.z * a.cout * K;
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int co = co0 + 16 * wco + 4 * g + r, k = k0 + 64 * wk + 16 * j + r16;
      if (co < a.cout && k < K) out[(size_t)co * K + k] = acc[j][r];
    }
  if (bias) {
    // the 256 / DG threads of a channel group, added in thread order through
    // the (now idle) X tile
    float* red = reinterpret_cast<float*>(s_x);
#pragma unroll
    for (int e = 0; e < 8; ++e) red[threadIdx.x * 8 + e] = bs[e];
    __syncthreads();
    if ((int)threadIdx.x < CO_T) {
      const int grp = threadIdx.x / 8, e = threadIdx.x % 8;
      float t = 0.0f;
      for (int j = grp; j < 256; j += DG) t += red[j * 8 + e];
      if (co0 + (int)threadIdx.x < a.cout)
        a.bias_partial[(size_t)blockIdx.z * a.cout + co0 + threadIdx.x] = t;
    }
  }
}

// ---------------------------------------------------------------------------
// The same gradient with its operands staged once per spatial tile and input-
// channel chunk, for cin and cout multiples of 16 (or cin 8): the block walks tiles of 4 x
// 32 pixels, stages a tile's dY [128 pixels][CO_T] and the (6 x 34)-pixel halo
// of CC input channels of X in LDS, and forms all nine taps' products from
// them, where wgrad_kernel gathers X once per tap.  Each wave holds up to 32 co
// x 9 taps x 16 channels (18 MFMA tiles).  CC = 32: CO_T 64: waves = co halves
// x channel halves; CO_T 32: channel halves x row pairs of the tile, added
// through LDS at the end; CC = 16: one tile row per wave.  One MFMA step is one row of 32 pixels, so the
// three fragments (kx) of a halo row serve the three taps ky whose tile rows
// lie at it: 26 fragment reads per 72 MFMAs, where a step of two 16-pixel rows
// needs 88 and is bound by them.  Double-buffered LDS, the next tile's loads in
// flight during the MFMAs, one barrier per tile; pixels outside the image stage
// dY = 0.  CC = 8 (the network's first layer, bound by reading dY): 32 co x 9
// taps x 8 channels per wave as five tiles of two taps each (the tenth is
// dropped), one tile row per wave.
// EDGE (images that are no whole tiles): beyond the image a cut tile's dY is 0,
// and so is X but for the pixel on the edge, which the first pixel beyond meets
// at kx = 0 (ky = 0).  An infinite X must not meet it, and is left out there.
// At 8 x 512 x 512: 32 -> 32 channels 211 -> 77 us (268 MB; 500 TF/s), 96 -> 32
// 476 -> 204 us, 8 -> 32 180 -> 48 us; at 8 x 256 x 256 64 -> 64 167 -> 57 us
// (680 TF/s), 192 -> 64 339 -> 143 us.
// ---------------------------------------------------------------------------
constexpr int kWgTH = 4, kWgTW = 32;

template <int CO_T, int CC, bool EDGE>
__global__ __launch_bounds__(256, 2) void wgrad_halo_kernel(WgradArgs a, int tiles_per_split) {
  static_assert(CC == 32 ? CO_T == 64 || CO_T == 32 : (CC == 8 || CC == 16) && CO_T <= 32, "tile");
  constexpr int PW = CC < 32 ? 4 : CO_T == 32 ? 2 : 1, TR = kWgTH / PW;  // waves along the rows; rows per wave
  constexpr int NP = kWgTH * kWgTW, HH = kWgTH + 2, HW = kWgTW + 2;
  constexpr int SD = CO_T + 16, SX = CC < 32 ? CC : 48;  // LDS row strides (bf16)
  constexpr int XG = CC / 8, NB = CC == 8 ? 5 : 9, NI = CO_T == 16 ? 1 : 2;  // groups per halo pixel; tiles per wave
  constexpr int DG = CO_T / 8, DC = NP * DG / 256, NX = HH * HW * XG, XC = (NX + 255) / 256;  // 16-byte groups
  constexpr int BUF = NP * SD + HH * HW * SX;
  static_assert(2 * BUF * (int)sizeof(bf16) >= (CC < 32 ? 1 : 2) * 4 * NI * NB * 64 * (int)sizeof(float), "the final sums fit the tiles");
  __shared__ __attribute__((aligned(16))) bf16 smem[2 * BUF];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int r16 = lane & 15, g = lane >> 4;
  const int wa = wv & 1, wb = wv >> 1;
  const int wco = CO_T == 64 ? wa * 32 : 0;     // this wave's first co
  const int wch = CC < 32 ? 0 : (CO_T == 64 ? wb : wa) * 16;  // and input channel
  const int part = PW == 4 ? wv : PW == 2 ? wb : 0, wr = part * TR;  // and tile row
  const int K = 9 * a.cin;
  const int co0 = blockIdx.x * CO_T, ch0 = blockIdx.y * CC;
  const int tiles_x = (a.W + kWgTW - 1) / kWgTW, tiles_y = (a.H + kWgTH - 1) / kWgTH;
  const int ntile = tiles_x * tiles_y * a.B;
  const int t_begin = blockIdx.z * tiles_per_split, t_end = min(ntile, t_begin + tiles_per_split);

  f32x4 acc[NI][NB];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const bool bias = a.bias_partial && blockIdx.y == 0;
  float bs[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};

  bf16x8 rd[DC], rx[XC];
  auto load = [&](int t) {
    const int tx = t % tiles_x, r = t / tiles_x, ty = r % tiles_y, b = r / tiles_y;
    const int x0 = tx * kWgTW, y0 = ty * kWgTH;
#pragma unroll
    for (int i = 0; i < DC; ++i) {
      const int q = tid + 256 * i, p = q / DG, cg = (q % DG) * 8;
      const int y = y0 + p / kWgTW, x = x0 + p % kWgTW;
      rd[i] = zero8();
      if (y < a.H && x < a.W)
        rd[i] = *reinterpret_cast<const bf16x8*>(a.dy + (((size_t)b * a.H + y) * a.W + x) * a.cout + co0 + cg);
    }
#pragma unroll
    for (int i = 0; i < XC; ++i) {
      const int q = tid + 256 * i, p = q / XG, cg = (q % XG) * 8;
      const int hy = p / HW, y = y0 + hy - 1, x = x0 + p - hy * HW - 1;
      rx[i] = zero8();
      if (q < NX && y >= 0 && y < a.H && x >= 0 && x < a.W)
        rx[i] = *reinterpret_cast<const bf16x8*>(conv_in(a.x, a.x2, a.c0, a.H, a.W, a.cin, b, y, x, ch0 + cg));
    }
  };
  if (t_begin < t_end) load(t_begin);
  for (int t = t_begin; t < t_end; ++t) {
    bf16* const sd = smem + ((t - t_begin) & 1) * BUF;
    bf16* const sx = sd + NP * SD;
#pragma unroll
    for (int i = 0; i < DC; ++i) {
      const int q = tid + 256 * i;
      *reinterpret_cast<bf16x8*>(&sd[(q / DG) * SD + (q % DG) * 8]) = rd[i];
      if (bias) {
        const i16x8 u = __builtin_bit_cast(i16x8, rd[i]);
#pragma unroll
        for (int e = 0; e < 8; ++e) bs[e] += __uint_as_float((unsigned)(unsigned short)u[e] << 16);
      }
    }
#pragma unroll
    for (int i = 0; i < XC; ++i) {
      const int q = tid + 256 * i;
      if (q < NX) *reinterpret_cast<bf16x8*>(&sx[(q / XG) * SX + (q % XG) * 8]) = rx[i];
    }
    __syncthreads();
    if (t + 1 < t_end) load(t + 1);
    const int row = 8 * g + (r16 >> 2), col = 4 * (r16 & 3);
    bf16x8 fa[TR][NI];
    // EDGE: a fragment (this lane's pixels 8 g .. 8 g + 7) without pixel edge_x
    const int edge_x = a.W - t % tiles_x * kWgTW, rows_in = a.H - t / tiles_x % tiles_y * kWgTH - wr;
    auto off_edge = [&](bf16x8 fb) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (8 * g + e == edge_x) fb[e] = (bf16)0.0f;
      return fb;
    };
    if constexpr (CC == 8) {
#pragma unroll
      for (int i = 0; i < NI; ++i) fa[0][i] = tr_fragment(sd, wr * kWgTW + row, 16 * i + col, SD);
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int tap = min(2 * j + ((r16 & 3) >> 1), 8);
        bf16x8 fb = tr_fragment(sx, (wr + tap / 3) * HW + row + tap % 3, 4 * (r16 & 1), SX);
        if constexpr (EDGE) {
          const int mine = min(2 * j + (r16 >> 3), 8);  // the tap of this lane's column
          if (mine % 3 == 0) fb = off_edge(fb);
          if (mine < 3 && rows_in <= 0) fb = zero8();
        }
#pragma unroll
        for (int i = 0; i < NI; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[0][i], fb, acc[i][j], 0, 0, 0);
      }
      continue;
    }
#pragma unroll
    for (int hr = 0; hr < TR + 2; ++hr) {  // halo rows wr + hr; tile rows wr + hr - ky
      if (hr < TR)
#pragma unroll
        for (int i = 0; i < NI; ++i)
          fa[hr][i] = tr_fragment(sd, (wr + hr) * kWgTW + row, wco + 16 * i + col, SD);
#pragma unroll
      for (int kx = 0; kx < 3; ++kx) {
        bf16x8 fb = tr_fragment(sx, (wr + hr) * HW + row + kx, wch + col, SX);
        if (EDGE && kx == 0) fb = off_edge(fb);
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) {
          const int r = hr - ky, j = (3 * ky + kx) % NB;
          if (r < 0 || r >= TR) continue;
          const bf16x8 fk = EDGE && ky == 0 && r >= rows_in ? zero8() : fb;
#pragma unroll
          for (int i = 0; i < NI; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[r][i], fk, acc[i][j], 0, 0, 0);
        }
      }
    }
  }
  float* const red = reinterpret_cast<float*>(smem);
  float* const mine = red + (PW == 2 ? wa : 0) * 4 * NI * NB * 64 + lane;
#pragma unroll
  for (int k = 1; k < PW; ++k) {  // the waves' sums, in the order of their rows
    __syncthreads();
    if (part == k)
#pragma unroll
      for (int i = 0; i < NI * NB; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) mine[(4 * i + r) * 64] = acc[i / NB][i % NB][r];
    __syncthreads();
    if (part == 0)
#pragma unroll
      for (int i = 0; i < NI * NB; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i / NB][i % NB][r] += mine[(4 * i + r) * 64];
  }
  if (part == 0) {
    float* const out = a.partial + (size_t)blockIdx.z * a.cout * K;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int co = co0 + wco + 16 * i + 4 * g + r, k = CC == 8 ? 16 * j + r16 : j * a.cin + ch0 + wch + r16;
          if (CC != 8 || k < K) out[(size_t)co * K + k] = acc[i][j][r];
        }
  }
  if (bias) {
    // the threads of a channel group, added in thread order through LDS
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 8; ++e) red[tid * 8 + e] = bs[e];
    __syncthreads();
    if (tid < CO_T) {
      const int grp = tid / 8, e = tid % 8;
      float t = 0.0f;
      for (int j = grp; j < 256; j += DG) t += red[j * 8 + e];
      a.bias_partial[(size_t)blockIdx.z * a.cout + co0 + tid] = t;
    }
  }
}

// out[i] = sum_s partial[s][i] in a fixed order: 64 columns per block, four per
// thread (16-byte loads), 16 threads per column with every 16th partial each,
// added in thread order.  Two arrays (the weights' n, the bias's n2) in one
// launch.  Bound by reading the partials: 10.5 -> 7.2 us a launch on average
// over a gradient step at 8 x 512 x 512, against one thread per column.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

__global__ __launch_bounds__(256) void reduce_partials_kernel(const float* __restrict__ partial,
                                                              float* __restrict__ out, long long n,
                                                              const float* __restrict__ partial2,
                                                              float* __restrict__ out2, int n2, int nsplit) {
  __shared__ f32x4 red[16][16];
  const int c = threadIdx.x & 15, s = threadIdx.x >> 4;
  const long long nb = (n + 63) / 64;
  const bool second = blockIdx.x >= nb;
  const long long i = ((long long)blockIdx.x - (second ? nb : 0)) * 64 + 4 * c, m = second ? n2 : n;
  const float* const p = second ? partial2 : partial;
  f32x4 t = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  if (i + 4 <= m) {
    f32x4 u = t;
    int k = s;
    for (; k + 48 < nsplit; k += 64) {
      const f32x4 v0 = *reinterpret_cast<const f32x4u*>(p + (size_t)k * m + i);
      const f32x4 v1 = *reinterpret_cast<const f32x4u*>(p + (size_t)(k + 16) * m + i);
      const f32x4 v2 = *reinterpret_cast<const f32x4u*>(p + (size_t)(k + 32) * m + i);
      const f32x4 v3 = *reinterpret_cast<const f32x4u*>(p + (size_t)(k + 48) * m + i);
      t += v0 + v1;
      u += v2 + v3;
    }
    for (; k < nsplit; k += 16) t += *reinterpret_cast<const f32x4u*>(p + (size_t)k * m + i);
    t += u;
  } else {
    for (int k = s; k < nsplit; k += 16)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i + e < m) t[e] += p[(size_t)k * m + i + e];
  }
  red[s][c] = t;
  __syncthreads();
  if (s == 0) {
    f32x4 u = red[0][c];
#pragma unroll
    for (int k = 1; k < 16; ++k) u += red[k][c];
    float* const o = second ? out2 : out;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (i + e < m) o[i + e] = u[e];
  }
}

// Column sums of an [M][C] bf16 or FP32 matrix into partial[split][C]: block
// `split` reduces rows [split rpb, split rpb + rpb).  Up to 256 columns per
// pass; the 256 threads are (256 / cw) row lanes x cw columns, so a row's
// columns are read by consecutive threads, and the row lanes are added in a
// fixed order through LDS.  blockDim.x = 256.
template <typename T>
__global__ __launch_bounds__(256) void colsum_kernel(const T* __restrict__ a, float* __restrict__ partial, long long M,
                                                     int C, long long rows_per_split) {
  __shared__ float red[256];
  const long long r0 = (long long)blockIdx.x * rows_per_split;
  const long long r1 = r0 + rows_per_split < M ? r0 + rows_per_split : M;
  for (int c0 = 0; c0 < C; c0 += 256) {
    const int cw = C - c0 < 256 ? C - c0 : 256, nrl = 256 / cw;
    const int rl = threadIdx.x / cw, c = c0 + (int)threadIdx.x % cw;
    // eight independent partial sums keep eight loads in flight
    float p8[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (rl < nrl) {
      long long r = r0 + rl;
      for (; r + 7LL * nrl < r1; r += 8LL * nrl) {
#pragma unroll
        for (int j = 0; j < 8; ++j) p8[j] += (float)a[(r + (long long)j * nrl) * C + c];
      }
      for (int j = 0; r < r1; r += nrl, ++j) p8[j & 7] += (float)a[r * C + c];
    }
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) s += p8[j];
    red[threadIdx.x] = s;
    __syncthreads();
    if ((int)threadIdx.x < cw) {
      float t = 0.0f;
      for (int k = 0; k < nrl; ++k) t += red[k * cw + threadIdx.x];
      partial[(size_t)blockIdx.x * C + c0 + threadIdx.x] = t;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Elementwise kernels.
// ---------------------------------------------------------------------------
__global__ void pad_input_kernel(const float* __restrict__ x, bf16* __restrict__ out8, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  bf16x8 v = zero8();
  v[0] = (bf16)x[i];
  *reinterpret_cast<bf16x8*>(out8 + i * 8) = v;
}

// dst[b][y][x][c] = mean of src[b][2y+i][2x+j][c]
__global__ void pool2_kernel(const bf16* __restrict__ src, bf16* __restrict__ dst, int B, int H, int W, int C) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long n = (long long)B * H * W * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  long long q = i / C;
  const int x = (int)(q % W);
  q /= W;
  const int y = (int)(q % H);
  const int b = (int)(q / H);
  const size_t row = (size_t)2 * W * C;
  const size_t o = (((size_t)b * 2 * H + 2 * y) * 2 * W + 2 * x) * C + c;
  const float s = (float)src[o] + (float)src[o + C] + (float)src[o + row] + (float)src[o + row + C];
  dst[i] = (bf16)(0.25f * s);
}

// 8 bf16 of one 16-byte vector as floats
__device__ __forceinline__ void unpack8(const bf16* p, float (&x)[8]) {
  const i16x8 u = __builtin_bit_cast(i16x8, *reinterpret_cast<const bf16x8*>(p));
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = __uint_as_float((unsigned)(unsigned short)u[e] << 16);
}

// pool2_kernel for C % 8 == 0, one thread per 8 channels of a pixel (16-byte
// accesses; element-wise it issued four 2-byte loads and two 64-bit divisions
// per value: 92 -> 43 us for the three levels of 8 x 512 x 512 x 32).  grid.y = b.
__global__ __launch_bounds__(256) void pool2_vec_kernel(const bf16* __restrict__ src, bf16* __restrict__ dst, int H,
                                                        int W, int C8) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= H * W * C8) return;
  const int p = i / C8, c = (i - p * C8) * 8, y = p / W, x = p - y * W, C = C8 * 8;
  const size_t row = (size_t)2 * W * C;
  const bf16* const s = src + (((size_t)blockIdx.y * 2 * H + 2 * y) * 2 * W + 2 * x) * C + c;
  float v0[8], v1[8], v2[8], v3[8];
  unpack8(s, v0);
  unpack8(s + C, v1);
  unpack8(s + row, v2);
  unpack8(s + row + C, v3);
  bf16x8 h;
#pragma unroll
  for (int e = 0; e < 8; ++e) h[e] = (bf16)(0.25f * (v0[e] + v1[e] + v2[e] + v3[e]));
  *reinterpret_cast<bf16x8*>(dst + (size_t)blockIdx.y * H * W * C + (size_t)i * 8) = h;
}

// pool2_back_kernel with out for C % 8 == 0, one thread per 8 channels of a
// source pixel: bound by its 9 bytes per value (455 -> 173 us for the three
// levels of 8 x 512 x 512 x 32; 99 us, 6.1 TB/s, at the largest).  grid.y = b.
__global__ __launch_bounds__(256) void pool2_back_vec_kernel(const float* __restrict__ dv,
                                                             const float* __restrict__ gsrc, bf16* __restrict__ out,
                                                             const bf16* __restrict__ mask, int H, int W, int C8) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= 4 * H * W * C8) return;
  const int p = i / C8, c = (i - p * C8) * 8, y = p / (2 * W), x = p - y * 2 * W, C = C8 * 8;
  const size_t o = (size_t)blockIdx.y * 4 * H * W * C + (size_t)i * 8;
  const f32x4* const d = reinterpret_cast<const f32x4*>(dv + (((size_t)blockIdx.y * H + y / 2) * W + x / 2) * C + c);
  const f32x4* const s = reinterpret_cast<const f32x4*>(gsrc + o);
  const f32x4 d0 = d[0], d1 = d[1], s0 = s[0], s1 = s[1];
  float m[8];
  unpack8(mask + o, m);
  bf16x8 h;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float v = (e < 4 ? s0[e & 3] : s1[e & 3]) + 0.25f * (e < 4 ? d0[e & 3] : d1[e & 3]);
    h[e] = (bf16)(m[e] > 0.0f ? v : 0.0f);
  }
  *reinterpret_cast<bf16x8*>(out + o) = h;
}

// g_src[b][2y+i][2x+j][c] += dv[b][y][x][c] / 4   (one thread per source element)
// gsrc += dv / 4 over each 2x2 block; with out (bf16) the sum, masked by
// mask > 0, goes to out instead (the last contribution to that gradient)
__global__ void pool2_back_kernel(const float* __restrict__ dv, float* __restrict__ gsrc, bf16* __restrict__ out,
                                  const bf16* __restrict__ mask, int B, int H, int W, int C) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long n = (long long)B * 2 * H * 2 * W * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  long long q = i / C;
  const int x = (int)(q % (2 * W));
  q /= 2 * W;
  const int y = (int)(q % (2 * H));
  const int b = (int)(q / (2 * H));
  const float v = gsrc[i] + 0.25f * dv[(((size_t)b * H + y / 2) * W + x / 2) * C + c];
  if (out) out[i] = (bf16)((float)mask[i] > 0.0f ? v : 0.0f);
  else gsrc[i] = v;
}

// dst[b][y][x][0:C0] = low[b][y/2][x/2][:], dst[..][C0:C0+C1] = skip[b][y][x][:]
__global__ void upcat_kernel(const bf16* __restrict__ low, const bf16* __restrict__ skip, bf16* __restrict__ dst,
                             int B, int H, int W, int C0, int C1) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int C = C0 + C1;
  const long long n = (long long)B * H * W * C;
  if (i >= n) return;
  const int c = (int)(i % C);
  long long q = i / C;
  const int x = (int)(q % W);
  q /= W;
  const int y = (int)(q % H);
  const int b = (int)(q / H);
  dst[i] = c < C0 ? low[(((size_t)b * (H / 2) + y / 2) * (W / 2) + x / 2) * C0 + c]
                  : skip[(((size_t)b * H + y) * W + x) * C1 + (c - C0)];
}

// g_low[b][y'][x'][c] = sum of the four children (c < C0); g_skip += rest
// glow = sum over each 2x2 block of dv[..., :C0]; with out (bf16), masked by
// mask > 0, into out instead
__global__ void upcat_back_low_kernel(const float* __restrict__ dv, float* __restrict__ glow, bf16* __restrict__ out,
                                      const bf16* __restrict__ mask, int B, int H, int W, int C0, int C1) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int Hl = H / 2, Wl = W / 2, C = C0 + C1;
  const long long n = (long long)B * Hl * Wl * C0;
  if (i >= n) return;
  const int c = (int)(i % C0);
  long long q = i / C0;
  const int x = (int)(q % Wl);
  q /= Wl;
  const int y = (int)(q % Hl);
  const int b = (int)(q / Hl);
  const size_t o = (((size_t)b * H + 2 * y) * W + 2 * x) * C + c;
  const size_t row = (size_t)W * C;
  const float v = dv[o] + dv[o + C] + dv[o + row] + dv[o + row + C];
  if (out) out[i] = (bf16)((float)mask[i] > 0.0f ? v : 0.0f);
  else glow[i] = v;
}

// gskip (+)= dv[..., C0:]
__global__ void upcat_back_skip_kernel(const float* __restrict__ dv, float* __restrict__ gskip, int B, int H, int W,
                                       int C0, int C1, int accumulate) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long n = (long long)B * H * W * C1;
  if (i >= n) return;
  const int c = (int)(i % C1);
  const long long p = i / C1;
  const float v = dv[p * (C0 + C1) + C0 + c];
  gskip[i] = accumulate ? gskip[i] + v : v;
}

// y[m] = x[m] + sum_c d0[m][c] w[c] + b
__global__ void head_kernel(const bf16* __restrict__ d0, const float* __restrict__ w, const float* __restrict__ b,
                            const float* __restrict__ x, float* __restrict__ y, long long M, int C) {
  const long long m = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  float s = b[0];
  if (C % 8 == 0) {
    // 16-byte loads of 8 channels
    for (int c = 0; c < C; c += 8) {
      const i16x8 u = __builtin_bit_cast(i16x8, *reinterpret_cast<const bf16x8*>(d0 + m * C + c));
#pragma unroll
      for (int e = 0; e < 8; ++e) s = __builtin_fmaf(__uint_as_float((unsigned)(unsigned short)u[e] << 16), w[c + e], s);
    }
  } else {
    for (int c = 0; c < C; ++c) s = __builtin_fmaf((float)d0[m * C + c], w[c], s);
  }
  y[m] = x[m] + s;
}

// dy = 2 (y - target) / n
// gd0 = dy w (FP32), or with out: bf16(dy w * (mask > 0)) into out.  One
// thread per (pixel, channel), so the gradient stores are coalesced; the
// channel-0 thread of a pixel also stores dy.
__global__ void head_back_kernel(const float* __restrict__ y, const float* __restrict__ target,
                                 const float* __restrict__ w, float* __restrict__ dy, float* __restrict__ gd0,
                                 bf16* __restrict__ out, const bf16* __restrict__ mask, long long M, int C,
                                 float scale) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M * C) return;
  const long long m = i / C;
  const int c = (int)(i - m * C);
  const float d = scale * (y[m] - target[m]);
  if (c == 0) dy[m] = d;
  const float v = d * w[c];
  if (out) out[i] = (bf16)((float)mask[i] > 0.0f ? v : 0.0f);
  else gd0[i] = v;
}

// head weight gradient partials: part[s][c] = sum_m dy[m] d0[m][c], part[s][C] = sum_m dy[m]
// partial[split][c] = sum over the split's rows of dy[r] * d0[r][c] (c < C)
// or dy[r] (c = C, the bias); C + 1 <= 256 columns, row lanes as in
// colsum_kernel.  blockDim.x = 256.
__global__ __launch_bounds__(256) void head_wgrad_kernel(const float* __restrict__ dy, const bf16* __restrict__ d0,
                                                         float* __restrict__ part, long long M, int C,
                                                         long long rows_per_split) {
  __shared__ float red[256];
  const int cw = C + 1, nrl = 256 / cw;
  const int rl = threadIdx.x / cw, c = (int)threadIdx.x % cw;
  const long long r0 = (long long)blockIdx.x * rows_per_split;
  const long long r1 = r0 + rows_per_split < M ? r0 + rows_per_split : M;
  float p8[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  if (rl < nrl) {
    long long r = r0 + rl;
    for (; r + 7LL * nrl < r1; r += 8LL * nrl) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const long long rr = r + (long long)j * nrl;
        p8[j] += dy[rr] * (c < C ? (float)d0[rr * C + c] : 1.0f);
      }
    }
    for (int j = 0; r < r1; r += nrl, ++j) p8[j & 7] += dy[r] * (c < C ? (float)d0[r * C + c] : 1.0f);
  }
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) s += p8[j];
  red[threadIdx.x] = s;
  __syncthreads();
  if ((int)threadIdx.x < cw) {
    float t = 0.0f;
    for (int k = 0; k < nrl; ++k) t += red[k * cw + threadIdx.x];
    part[(size_t)blockIdx.x * cw + threadIdx.x] = t;
  }
}

// head_back_kernel with out and head_wgrad_kernel in one pass over d0, for C =
// 8 C8 with C8 a power of two up to 16: block `split` takes 4096 rows, C8
// threads per row with 8 channels each.  Bound by its 4 C + 12 bytes per row
// (mask and d0 being the same tensor, as in the network, 6 C bytes less than
// the two kernels moved): 443 -> 69 us at 8 x 512 x 512 x 32.
__global__ __launch_bounds__(256) void head_back_vec_kernel(const float* __restrict__ y,
                                                            const float* __restrict__ target,
                                                            const float* __restrict__ w, const bf16* __restrict__ d0,
                                                            float* __restrict__ dy, bf16* __restrict__ out,
                                                            const bf16* __restrict__ mask, float* __restrict__ part,
                                                            long long M, int C8, float scale) {
  __shared__ float red[256][9];
  const int lg = threadIdx.x & (C8 - 1), rl = threadIdx.x / C8, nrl = 256 / C8, C = C8 * 8;
  const long long r0 = (long long)blockIdx.x * 4096, r1 = r0 + 4096 < M ? r0 + 4096 : M;
  const bool same = mask == d0;
  float wc[8], acc[9];
#pragma unroll
  for (int e = 0; e < 8; ++e) wc[e] = w[lg * 8 + e];
#pragma unroll
  for (int e = 0; e < 9; ++e) acc[e] = 0.0f;
  for (long long r = r0 + rl; r < r1; r += nrl) {
    const float d = scale * (y[r] - target[r]);
    const long long o = r * C + lg * 8;
    float v[8], m[8];
    unpack8(d0 + o, v);
    if (same) {
#pragma unroll
      for (int e = 0; e < 8; ++e) m[e] = v[e];
    } else {
      unpack8(mask + o, m);
    }
    bf16x8 h;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float g = d * wc[e];
      h[e] = (bf16)(m[e] > 0.0f ? g : 0.0f);
      acc[e] = __builtin_fmaf(d, v[e], acc[e]);
    }
    *reinterpret_cast<bf16x8*>(out + o) = h;
    if (lg == 0) dy[r] = d;
    acc[8] += d;
  }
#pragma unroll
  for (int e = 0; e < 9; ++e) red[threadIdx.x][e] = acc[e];
  __syncthreads();
  // column c: the row lanes of its channel group, in order; column C: dy
  for (int c = threadIdx.x; c <= C; c += 256) {
    const int e = c < C ? c & 7 : 8, g = c < C ? c >> 3 : 0;
    float t = 0.0f;
    for (int k = 0; k < nrl; ++k) t += red[k * C8 + g][e];
    part[(size_t)blockIdx.x * (C + 1) + c] = t;
  }
}

// out = bf16(g * (act > 0))
__global__ void relu_mask_kernel(const float* __restrict__ g, const bf16* __restrict__ act, bf16* __restrict__ out,
                                 long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] = (bf16)((float)act[i] > 0.0f ? g[i] : 0.0f);
}

// wt[c][t][o] = w[o][8 - t][c]  (input-gradient weights)
__global__ void flip_weights_kernel(const bf16* __restrict__ w, bf16* __restrict__ wt, int cin, int cout) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long n = (long long)cin * 9 * cout;
  if (i >= n) return;
  const int o = (int)(i % cout);
  const long long q = i / cout;
  const int t = (int)(q % 9);
  const int c = (int)(q / 9);
  wt[i] = w[((size_t)o * 9 + (8 - t)) * cin + c];
}

// Adam on an FP32 master tensor, with its bf16 copy (nullable)
__global__ void adam_kernel(float* __restrict__ w32, bf16* __restrict__ w16, const float* __restrict__ g,
                            float* __restrict__ m, float* __restrict__ v, long long n, float lr, float b1, float b2,
                            float eps, float c1, float c2) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w32[i] - lr * (mi * c1) / (__builtin_sqrtf(vi * c2) + eps);
  w32[i] = wi;
  if (w16) w16[i] = (bf16)wi;
}

__global__ void fill_kernel(float* __restrict__ p, long long n, float value) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = value;
}

__global__ void to_bf16_kernel(const float* __restrict__ src, bf16* __restrict__ dst, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = (bf16)src[i];
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
static inline unsigned blocks_for(long long n, int t = 256) { return (unsigned)((n + t - 1) / t); }

static bool aligned16(const void* a, const void* b = nullptr, const void* c = nullptr, const void* d = nullptr) {
  return (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c | (uintptr_t)d) & 15) == 0;
}

// 3x3 convolutions with cin % 32 == 0 (or cin 16 or 8) and cout % 16 == 0 run
// the halo-tiled kernel; the others the K-step-staged ones.
static bool halo_conv(int cin, int cout) { return (cin % 32 == 0 || cin == 16 || cin == 8) && cout % 16 == 0; }

// 8-row tiles and 64-channel blocks where cout allows, else 16-row tiles.
static int halo_block(int cout) { return cout % 64 == 0 ? 64 : cout % 32 == 0 ? 32 : 16; }

// Blocks walk runs of items, two per CU (three with registers and LDS for it
// were slower: 73 -> 89 us for 32 -> 32 channels at 8 x 512 x 512).  With one
// chunk and several blocks of output channels a run is of tiles, each halo
// loaded once for all of them (32 -> 96 channels, split: 260 us where every item
// loads its own, 181), where that leaves a tile for every block.
template <int TH, int BN, int WM, int WN, int CC, HaloRun RUN>
static hipError_t run_halo(const ConvArgs& a, hipStream_t s) {
  const long long nitem = (long long)((a.W + 15) / 16) * ((a.H + TH - 1) / TH) * a.B * (a.cout / BN);
  if (nitem >= 1LL << 30) return hipErrorInvalidValue;
  const long long units = RUN == kHaloStays ? nitem / (a.cout / BN) : nitem;
  const long long blocks = units < 512 ? units : 512;
  conv3x3_halo_kernel<TH, BN, WM, WN, CC, RUN><<<(unsigned)blocks, 256, 0, s>>>(a);
  return hipGetLastError();
}

template <int CC>
static hipError_t run_halo_cc(const ConvArgs& a, hipStream_t s) {
  const int bn = halo_block(a.cout);
  const long long tiles = (long long)((a.W + 15) / 16) * ((a.H + (bn == 64 ? 7 : 15)) / (bn == 64 ? 8 : 16)) * a.B;
  const bool weights = a.cin == CC && a.cout == bn, halos = a.cin == CC && a.cout > bn && tiles >= 512;
  if (bn == 64) return halos ? run_halo<8, 64, 2, 2, CC, kHaloStays>(a, s) : run_halo<8, 64, 2, 2, CC, kAnyRun>(a, s);
  if (bn == 32)
    return weights ? run_halo<16, 32, 4, 1, CC, kWeightsStay>(a, s)
           : halos ? run_halo<16, 32, 4, 1, CC, kHaloStays>(a, s)
                   : run_halo<16, 32, 4, 1, CC, kAnyRun>(a, s);
  return weights ? run_halo<16, 16, 4, 1, CC, kWeightsStay>(a, s)
         : halos ? run_halo<16, 16, 4, 1, CC, kHaloStays>(a, s)
                 : run_halo<16, 16, 4, 1, CC, kAnyRun>(a, s);
}

static hipError_t launch_halo(const ConvArgs& a, hipStream_t s) {
  return a.cin == 8 ? run_halo_cc<8>(a, s) : a.cin == 16 ? run_halo_cc<16>(a, s) : run_halo_cc<32>(a, s);
}

// Whether nn_conv3x3_upback runs in one kernel: whole blocks of output
// channels on either side of the concatenation.
bool nn_upback_fused(int cin, int cout, int c0) { return halo_conv(cin, cout) && c0 % halo_block(cout) == 0; }

// Input gradient of a convolution of [upsample2(low), skip], low's part summed
// over 2 x 2 blocks and masked, in the convolution's epilogue: the FP32
// gradient of the concatenation, written and read again, is 1.6 GB at 8 x 512 x
// 512 x (64 + 32), and the two passes that split it took 614 us over the three
// levels; the convolution itself is no slower for it (the largest 231 -> 181 us
// with the halo kept for its three blocks of output channels).
hipError_t nn_conv3x3_upback(const void* in, const void* w, void* low_out, const void* low_mask, float* skip_out, int B,
                             int H, int W, int cin, int cout, int c0, hipStream_t s) {
  if (!nn_upback_fused(cin, cout, c0) || !aligned16(low_out, low_mask, skip_out)) return hipErrorInvalidValue;
  ConvArgs a{static_cast<const bf16*>(in), static_cast<const bf16*>(w), nullptr, nullptr, B, H, W, cin, cout, 0, 1,
             nullptr, nullptr, 0, static_cast<bf16*>(low_out), static_cast<const bf16*>(low_mask), skip_out, c0};
  return launch_halo(a, s);
}

hipError_t nn_conv3x3(const void* in, const void* in2, int c0, const void* w, const float* bias, void* out,
                      const void* mask, int B, int H, int W, int cin, int cout, int relu, int out_f32, hipStream_t s) {
  ConvArgs a{static_cast<const bf16*>(in), static_cast<const bf16*>(w), bias, out, B, H, W, cin, cout, relu, out_f32,
             static_cast<const bf16*>(mask), static_cast<const bf16*>(in2), c0, nullptr, nullptr, nullptr, 0};
  const long long M = (long long)B * H * W;
  if (cin % 8 != 0) return hipErrorInvalidValue;
  // the halo kernel stores (and reads the mask) 16 bytes at a time, the others
  // element by element
  if (halo_conv(cin, cout) && aligned16(out, mask)) return launch_halo(a, s);
  if (cout % 128 == 0) {
    conv3x3_lds_kernel<128, 128, 2, 2><<<dim3(blocks_for(M, 128), cout / 128), 256, 0, s>>>(a);
  } else if (cout % 64 == 0) {
    conv3x3_lds_kernel<128, 64, 2, 2><<<dim3(blocks_for(M, 128), cout / 64), 256, 0, s>>>(a);
  } else if (cout % 32 == 0) {
    conv3x3_lds_kernel<256, 32, 4, 1><<<dim3(blocks_for(M, 256), cout / 32), 256, 0, s>>>(a);
  } else {
    conv3x3_kernel<4, 1><<<dim3(blocks_for(M, 128), (cout + 31) / 32), 256, 0, s>>>(a);
  }
  return hipGetLastError();
}

long long nn_wgrad_splits(long long M) {
  // about 8192 pixels per block, at least one block
  long long n = (M + 8191) / 8192;
  return n < 1 ? 1 : n;
}

static hipError_t reduce_partials(const float* partial, float* out, long long n, const float* partial2, float* out2,
                                  int n2, long long rows, hipStream_t s) {
  const long long nb = (n + 63) / 64 + (n2 + 63) / 64;
  reduce_partials_kernel<<<(unsigned)nb, 256, 0, s>>>(partial, out, n, partial2, out2, n2, (int)rows);
  return hipGetLastError();
}

// wgrad_halo_kernel's shapes and its tile: input channels per chunk (0: none),
// output channels per block.  16-channel tiles serve what 32 does not divide.
static int halo_wgrad_cc(int cin, int cout) {
  if (cout % 16 != 0) return 0;
  return cin == 8 ? 8 : cin % 32 == 0 && cout % 32 == 0 ? 32 : cin % 16 == 0 ? 16 : 0;
}
static int halo_wgrad_co(int cc, int cout) { return cc == 32 && cout % 64 == 0 ? 64 : cout % 32 == 0 ? 32 : 16; }

// Pixel-range splits of wgrad_halo_kernel: as many as give the launch its two
// workgroups per CU at once, with at least 4 tiles each; and twice, three times
// as many, so that no FP32 accumulator holds more than kWgTiles tiles (8192
// pixels, as the gathered form's ranges) however large the batch is.
constexpr int kWgTiles = 8192 / (kWgTH * kWgTW);

static int halo_wgrad_splits(int B, int H, int W, int cin, int cout, int cc) {
  const long long ntile = (long long)B * ((W + kWgTW - 1) / kWgTW) * ((H + kWgTH - 1) / kWgTH);
  const long long blocks = (long long)(cout / halo_wgrad_co(cc, cout)) * (cin / cc);
  const long long once = 512 / blocks < 1 ? 1 : 512 / blocks;
  long long n = once;
  if (n > ntile / 4) n = ntile / 4 < 1 ? 1 : ntile / 4;
  if ((ntile + n - 1) / n > kWgTiles) n = ((ntile + kWgTiles - 1) / kWgTiles + once - 1) / once * once;
  return (int)n;
}

// Rows of partial sums a weight gradient may need: each holds cout * (9 cin +
// 1) floats, the weight partials of all rows first, then the bias partials.
long long nn_wgrad_parts(int B, int H, int W, int cin, int cout) {
  const long long n = nn_wgrad_splits((long long)B * H * W);
  const int cc = halo_wgrad_cc(cin, cout);
  if (cc == 0) return n;
  const long long h = halo_wgrad_splits(B, H, W, cin, cout, cc);
  return h > n ? h : n;
}

template <int CO_T, int CC>
static void run_wgrad_halo(const WgradArgs& a, dim3 grid, int tiles_per_split, hipStream_t s) {
  if (a.W % kWgTW || a.H % kWgTH) wgrad_halo_kernel<CO_T, CC, true><<<grid, 256, 0, s>>>(a, tiles_per_split);
  else wgrad_halo_kernel<CO_T, CC, false><<<grid, 256, 0, s>>>(a, tiles_per_split);
}

hipError_t nn_wgrad(const void* x, const void* x2, int c0, const void* dy, float* dw, float* db, float* partial, int B,
                    int H, int W, int cin, int cout, hipStream_t s) {
  const long long M = (long long)B * H * W;
  const int K = 9 * cin;
  const int cc = halo_wgrad_cc(cin, cout);
  const bool halo = cc != 0 && (!x2 || c0 % cc == 0) &&
                    (long long)B * ((W + kWgTW - 1) / kWgTW) * ((H + kWgTH - 1) / kWgTH) < (1LL << 30);
  long long parts = nn_wgrad_splits(M);
  const long long per = ((M + parts - 1) / parts + 63) / 64 * 64;
  WgradArgs a{static_cast<const bf16*>(x), static_cast<const bf16*>(dy), partial, B, H, W, cin, cout, per,
              static_cast<const bf16*>(x2), c0, nullptr};
  if (halo) {
    const int ns = halo_wgrad_splits(B, H, W, cin, cout, cc), co = halo_wgrad_co(cc, cout);
    const dim3 grid(cout / co, cin / cc, ns);
    const int ntile = B * ((W + kWgTW - 1) / kWgTW) * ((H + kWgTH - 1) / kWgTH), tps = (ntile + ns - 1) / ns;
    parts = ns;
    a.bias_partial = db ? partial + parts * cout * K : nullptr;
    if (cc == 32 && co == 64) run_wgrad_halo<64, 32>(a, grid, tps, s);
    else if (cc == 32) run_wgrad_halo<32, 32>(a, grid, tps, s);
    else if (cc == 16 && co == 32) run_wgrad_halo<32, 16>(a, grid, tps, s);
    else if (cc == 16) run_wgrad_halo<16, 16>(a, grid, tps, s);
    else if (co == 32) run_wgrad_halo<32, 8>(a, grid, tps, s);
    else run_wgrad_halo<16, 8>(a, grid, tps, s);
  } else {
    a.bias_partial = db ? partial + parts * cout * K : nullptr;
    if (cout <= 32) wgrad_kernel<32><<<dim3(1, (K + 127) / 128, (unsigned)parts), 256, 0, s>>>(a);
    else wgrad_kernel<64><<<dim3((cout + 63) / 64, (K + 63) / 64, (unsigned)parts), 256, 0, s>>>(a);
  }
  return reduce_partials(partial, dw, (long long)cout * K, a.bias_partial, db, db ? cout : 0, parts, s);
}

hipError_t nn_colsum_bf16(const void* a, float* out, float* partial, long long M, int C, hipStream_t s) {
  const long long ns = (M + 4095) / 4096;
  colsum_kernel<bf16><<<(unsigned)ns, 256, 0, s>>>(static_cast<const bf16*>(a), partial, M, C, 4096);
  return reduce_partials(partial, out, C, nullptr, nullptr, 0, ns, s);
}

hipError_t nn_pad_input(const float* x, void* out8, long long n, hipStream_t s) {
  pad_input_kernel<<<blocks_for(n), 256, 0, s>>>(x, static_cast<bf16*>(out8), n);
  return hipGetLastError();
}

// The vector kernels take 8 channels as aligned vectors, index one image in 32
// bits and the image by grid.y.
static bool vec8(long long per_image, int B, int C) { return C % 8 == 0 && per_image < (1LL << 31) && B < 65536; }

hipError_t nn_pool2(const void* src, void* dst, int B, int H, int W, int C, hipStream_t s) {
  if (vec8((long long)H * W * C, B, C) && aligned16(src, dst)) {
    const dim3 grid(blocks_for((long long)H * W * (C / 8)), (unsigned)B);
    pool2_vec_kernel<<<grid, 256, 0, s>>>(static_cast<const bf16*>(src), static_cast<bf16*>(dst), H, W, C / 8);
    return hipGetLastError();
  }
  pool2_kernel<<<blocks_for((long long)B * H * W * C), 256, 0, s>>>(static_cast<const bf16*>(src),
                                                                   static_cast<bf16*>(dst), B, H, W, C);
  return hipGetLastError();
}

hipError_t nn_pool2_back(const float* dv, float* gsrc, void* out, const void* mask, int B, int H, int W, int C,
                         hipStream_t s) {
  if (out && vec8(4LL * H * W * C, B, C) && aligned16(dv, gsrc, out, mask)) {
    const dim3 grid(blocks_for(4LL * H * W * (C / 8)), (unsigned)B);
    pool2_back_vec_kernel<<<grid, 256, 0, s>>>(dv, gsrc, static_cast<bf16*>(out), static_cast<const bf16*>(mask), H, W,
                                               C / 8);
    return hipGetLastError();
  }
  pool2_back_kernel<<<blocks_for((long long)B * 4 * H * W * C), 256, 0, s>>>(
      dv, gsrc, static_cast<bf16*>(out), static_cast<const bf16*>(mask), B, H, W, C);
  return hipGetLastError();
}

hipError_t nn_upcat(const void* low, const void* skip, void* dst, int B, int H, int W, int C0, int C1,
                    hipStream_t s) {
  upcat_kernel<<<blocks_for((long long)B * H * W * (C0 + C1)), 256, 0, s>>>(
      static_cast<const bf16*>(low), static_cast<const bf16*>(skip), static_cast<bf16*>(dst), B, H, W, C0, C1);
  return hipGetLastError();
}

hipError_t nn_upcat_back(const float* dv, float* glow, void* glow_out, const void* glow_mask, float* gskip,
                         int skip_accumulate, int B, int H, int W, int C0, int C1, hipStream_t s) {
  upcat_back_low_kernel<<<blocks_for((long long)B * (H / 2) * (W / 2) * C0), 256, 0, s>>>(
      dv, glow, static_cast<bf16*>(glow_out), static_cast<const bf16*>(glow_mask), B, H, W, C0, C1);
  upcat_back_skip_kernel<<<blocks_for((long long)B * H * W * C1), 256, 0, s>>>(dv, gskip, B, H, W, C0, C1,
                                                                               skip_accumulate);
  return hipGetLastError();
}

hipError_t nn_head(const void* d0, const float* w, const float* b, const float* x, float* y, long long M, int C,
                   hipStream_t s) {
  head_kernel<<<blocks_for(M), 256, 0, s>>>(static_cast<const bf16*>(d0), w, b, x, y, M, C);
  return hipGetLastError();
}

hipError_t nn_head_back(const float* y, const float* target, const float* w, const void* d0, float* dy, float* gd0,
                        void* gd0_out, const void* mask, float* gw, float* partial, long long M, int C,
                        hipStream_t s) {
  const int c8 = C / 8;
  if (gd0_out && C % 8 == 0 && c8 <= 16 && (c8 & (c8 - 1)) == 0 && aligned16(d0, gd0_out, mask)) {
    const long long nb = (M + 4095) / 4096;
    head_back_vec_kernel<<<(unsigned)nb, 256, 0, s>>>(y, target, w, static_cast<const bf16*>(d0), dy,
                                                      static_cast<bf16*>(gd0_out), static_cast<const bf16*>(mask),
                                                      partial, M, c8, 2.0f / (float)M);
    return reduce_partials(partial, gw, C + 1, nullptr, nullptr, 0, nb, s);
  }
  head_back_kernel<<<blocks_for(M * C), 256, 0, s>>>(y, target, w, dy, gd0, static_cast<bf16*>(gd0_out),
                                                 static_cast<const bf16*>(mask), M, C, 2.0f / (float)M);
  const long long ns = (M + 4095) / 4096;
  head_wgrad_kernel<<<(unsigned)ns, 256, 0, s>>>(dy, static_cast<const bf16*>(d0), partial, M, C, 4096);
  return reduce_partials(partial, gw, C + 1, nullptr, nullptr, 0, ns, s);
}

hipError_t nn_relu_mask(const float* g, const void* act, void* out, long long n, hipStream_t s) {
  relu_mask_kernel<<<blocks_for(n), 256, 0, s>>>(g, static_cast<const bf16*>(act), static_cast<bf16*>(out), n);
  return hipGetLastError();
}

hipError_t nn_flip_weights(const void* w, void* wt, int cin, int cout, hipStream_t s) {
  flip_weights_kernel<<<blocks_for((long long)cin * 9 * cout), 256, 0, s>>>(static_cast<const bf16*>(w),
                                                                           static_cast<bf16*>(wt), cin, cout);
  return hipGetLastError();
}

hipError_t nn_adam(float* w32, void* w16, const float* g, float* m, float* v, long long n, float lr, float b1,
                   float b2, float eps, int step, hipStream_t s) {
  const float c1 = 1.0f / (1.0f - powf(b1, (float)step)), c2 = 1.0f / (1.0f - powf(b2, (float)step));
  adam_kernel<<<blocks_for(n), 256, 0, s>>>(w32, static_cast<bf16*>(w16), g, m, v, n, lr, b1, b2, eps, c1, c2);
  return hipGetLastError();
}

hipError_t nn_fill(float* p, long long n, float value, hipStream_t s) {
  fill_kernel<<<blocks_for(n), 256, 0, s>>>(p, n, value);
  return hipGetLastError();
}

hipError_t nn_to_bf16(const float* src, void* dst, long long n, hipStream_t s) {
  to_bf16_kernel<<<blocks_for(n), 256, 0, s>>>(src, static_cast<bf16*>(dst), n);
  return hipGetLastError();
}

}  // namespace sgdct
