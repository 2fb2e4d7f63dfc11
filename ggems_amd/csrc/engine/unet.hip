// 3x3 convolutions of the scatter surrogate's U-Net on the matrix cores:
// BF16 operands, FP32 accumulation (v_mfma_f32_16x16x32_bf16).
//
// Layouts: activations NHWC (channels fastest), weights [Cout][9][Cin]
// (tap = 3 * (dy + 1) + (dx + 1)), so that the GEMM's reduction index
// k = tap * Cin + ci runs over contiguous memory in both operands.  Cin and
// Cout are multiples of 8 and 16 (the first layer pads its two input
// channels); W is a multiple of 16 and N H W of 32.
//
// Every kernel reads 8 channels of a tensor, or 8 weights, in one 16-byte load.
// Two sets of kernels.  The channel counts of the U-Net take the tile kernels
// (conv_tile_kernel, conv_wgrad_tile_kernel): an input tile with its halo goes
// to LDS once and serves all nine taps.  Other counts, and in the forward pass
// and the data gradient an output that is not 8-byte aligned (the tile kernel
// stores four channels at a time), take the general ones, whose order of
// additions the tile kernels keep there:
//
// Forward (implicit GEMM, M = pixels, N = Cout, K = 9 Cin): a wave owns
// 32 consecutive pixels (two runs of 16 within image rows) and up to 64 output
// channels, i.e. 2 x 4 accumulator tiles of 16 x 16; each K step of 32 loads
// one 16-byte A fragment per pixel tile from memory and one B fragment per
// channel tile from the block's LDS copy of the weights, and issues 8 MFMAs.
// Bias and ReLU are applied in the epilogue.  The data gradient
// is the same kernel on the flipped, transposed weights.
//
// Weight gradient (M = Cout, N = 9 Cin, K = pixels): both operands have
// pixels as their strided index.  A block stages 32 pixels of dY and of the
// shifted input in LDS as they lie in memory (channels contiguous, 16-byte
// stores) and the waves read MFMA fragments with gfx950's transposing LDS
// read; blocks split the pixels and add their partial sums atomically in
// FP32 (the tile kernel in a work space, summed in order).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <string>

#include "../../../include/ggems_engine.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

thread_local std::string g_unet_error;

int ufail(int code, const std::string& msg) {
  g_unet_error = msg;
  return code;
}

constexpr int kWaves = 4;
constexpr int kFwdPix = 32;  // pixels per wave
constexpr int kFwdCh = 64;   // output channels per wave

__device__ inline bf16x8 zero8() {
  bf16x8 z;
  for (int i = 0; i < 8; ++i) z[i] = (__bf16)0.0f;
  return z;
}

// A fragment: 8 consecutive k of pixel (y, x) for reduction index k0
// (k0 multiple of 8; all 8 lie in one tap because Cin is a multiple of 8)
__device__ inline bf16x8 load_a(const __bf16* x, int img, int y, int xx, int k0, int K, int Cin, int H, int W) {
  if (k0 >= K) return zero8();
  const int tap = k0 / Cin, ci = k0 - tap * Cin;
  const int yy = y + tap / 3 - 1, xs = xx + tap % 3 - 1;
  if (yy < 0 || yy >= H || xs < 0 || xs >= W) return zero8();
  return *reinterpret_cast<const bf16x8*>(x + (((size_t)img * H + yy) * W + xs) * Cin + ci);
}

// The blocks go to the eight XCDs in turn (block b to XCD b % 8), and each
// XCD has its own L2.  xcd_tile() numbers the tiles so that each XCD takes a
// contiguous run of them: neighbouring pixel tiles, which read the same
// image rows through the 3x3 stencil, then share one L2.  Blocks past the
// last tile return at once.
constexpr int kXcds = 8;

__device__ inline int xcd_tile(int n_tiles) {
  const int per = (int)((gridDim.x + kXcds - 1) / kXcds);
  return (int)(blockIdx.x % kXcds) * per + (int)(blockIdx.x / kXcds);
}

// The block's four waves share one tile of 16 NT output channels and take
// four consecutive 32-pixel tiles; each K step's weight chunk (16 NT
// channels x 32 k) is staged once per block in LDS, double-buffered, instead
// of being fetched from L2 by every wave.  NT is 4 for 64 or more output
// channels and 1 or 2 for the narrow layers, which would otherwise multiply
// zero weights.
constexpr int kBRow = 32 + 8;  // bf16 per staged weight row (padded against bank conflicts)

template <int NT>
__global__ __launch_bounds__(64 * kWaves) void conv_fwd_kernel(const __bf16* __restrict__ x,
                                                               const __bf16* __restrict__ w,
                                                               const float* __restrict__ bias,
                                                               __bf16* __restrict__ y, int N, int H, int W, int Cin,
                                                               int Cout, int relu) {
  constexpr int kCh = 16 * NT;
  __shared__ __bf16 sB[2][kCh * kBRow];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int pix_tiles = (N * H * W) / kFwdPix;
  const int ch_tiles = (Cout + kCh - 1) / kCh;
  const int block_tiles = ((pix_tiles + kWaves - 1) / kWaves) * ch_tiles;
  const int bt = xcd_tile(block_tiles);
  if (bt >= block_tiles) return;  // the whole block: no barrier is skipped
  const int ct = bt % ch_tiles;
  const int pt = (bt / ch_tiles) * kWaves + wave;
  const bool active = pt < pix_tiles;  // every wave stages and synchronises; only active ones compute
  const int p0 = (active ? pt : 0) * kFwdPix;
  // each run of 16 pixels lies in one image row (W is a multiple of 16)
  int img[2], yrow[2], x0[2];
  for (int i = 0; i < 2; ++i) {
    const int q = p0 + 16 * i, rem = q % (H * W);
    img[i] = q / (H * W);
    yrow[i] = rem / W;
    x0[i] = rem - yrow[i] * W;
  }
  const int c0 = ct * kCh;
  const int K = 9 * Cin;
  const int r = lane & 15, g = lane >> 4;  // fragment row / k group
  // staging: thread t < 4 kCh copies 8 k of channel c0 + t / 4
  const int s_co = threadIdx.x >> 2, s_kq = (threadIdx.x & 3) * 8;
  const bool stager = s_co < kCh;
  auto stage = [&](int buf, int k0) {
    if (!stager) return;
    const int co = c0 + s_co, k = k0 + s_kq;
    bf16x8 v = (co < Cout && k < K) ? *reinterpret_cast<const bf16x8*>(w + (size_t)co * K + k) : zero8();
    *reinterpret_cast<bf16x8*>(&sB[buf][s_co * kBRow + s_kq]) = v;
  };
  f32x4 acc[2][NT];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  stage(0, 0);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += 32) {
    if (k0 + 32 < K) stage(buf ^ 1, k0 + 32);  // the next chunk, while this one is used
    const int kk = k0 + 8 * g;
    bf16x8 a[2], b[NT];
    for (int i = 0; i < 2; ++i) a[i] = load_a(x, img[i], yrow[i], x0[i] + r, kk, K, Cin, H, W);
    for (int j = 0; j < NT; ++j) b[j] = *reinterpret_cast<const bf16x8*>(&sB[buf][(16 * j + r) * kBRow + 8 * g]);
    for (int i = 0; i < 2; ++i)
      for (int j = 0; j < NT; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    __syncthreads();
    buf ^= 1;
  }
  if (!active) return;
  // C fragment: column r (output channel), rows 4 g .. 4 g + 3 (pixels)
  for (int j = 0; j < NT; ++j) {
    const int co = c0 + 16 * j + r;
    if (co >= Cout) continue;
    const float bv = bias ? bias[co] : 0.0f;
    for (int i = 0; i < 2; ++i)
      for (int e = 0; e < 4; ++e) {
        float v = acc[i][j][e] + bv;
        if (relu) v = v > 0.0f ? v : 0.0f;
        const int px = p0 + 16 * i + 4 * g + e;
        y[(size_t)px * Cout + co] = (__bf16)v;
      }
  }
}

// Split-K variant for deep layers (K = 9 Cin of many 32-steps): the block's
// four waves share one 32-pixel x 64-channel output tile and take every
// fourth K chunk; a group of four chunks is staged in LDS at a time and the
// four partial tiles are summed through LDS at the end.  A layer with few
// pixel tiles gets four times the waves this way.
__global__ __launch_bounds__(64 * kWaves) void conv_fwd_splitk_kernel(const __bf16* __restrict__ x,
                                                                      const __bf16* __restrict__ w,
                                                                      const float* __restrict__ bias,
                                                                      __bf16* __restrict__ y, int N, int H, int W,
                                                                      int Cin, int Cout, int relu) {
  __shared__ __bf16 sB[kWaves][kFwdCh * kBRow];
  __shared__ float sP[kWaves][32][64 + 1];  // partial tiles: [wave][element][lane]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ch_tiles = (Cout + kFwdCh - 1) / kFwdCh;
  const int n_tiles = ((N * H * W) / kFwdPix) * ch_tiles;
  const int bt = xcd_tile(n_tiles);
  if (bt >= n_tiles) return;  // the whole block: no barrier is skipped
  const int ct = bt % ch_tiles, pt = bt / ch_tiles;
  const int p0 = pt * kFwdPix;
  int img[2], yrow[2], x0[2];
  for (int i = 0; i < 2; ++i) {
    const int q = p0 + 16 * i, rem = q % (H * W);
    img[i] = q / (H * W);
    yrow[i] = rem / W;
    x0[i] = rem - yrow[i] * W;
  }
  const int c0 = ct * kFwdCh;
  const int K = 9 * Cin;
  const int r = lane & 15, g = lane >> 4;
  const int s_co = threadIdx.x >> 2, s_kq = (threadIdx.x & 3) * 8;
  f32x4 acc[2][4];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int kg = 0; kg < K; kg += 32 * kWaves) {
    // stage the group's four chunks: thread t copies 8 k of channel c0 + t / 4 of each
    for (int c = 0; c < kWaves; ++c) {
      const int co = c0 + s_co, k = kg + 32 * c + s_kq;
      bf16x8 v = (co < Cout && k < K) ? *reinterpret_cast<const bf16x8*>(w + (size_t)co * K + k) : zero8();
      *reinterpret_cast<bf16x8*>(&sB[c][s_co * kBRow + s_kq]) = v;
    }
    __syncthreads();
    const int k0 = kg + 32 * wave;
    if (k0 < K) {
      const int kk = k0 + 8 * g;
      bf16x8 a[2], b[4];
      for (int i = 0; i < 2; ++i) a[i] = load_a(x, img[i], yrow[i], x0[i] + r, kk, K, Cin, H, W);
      for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const bf16x8*>(&sB[wave][(16 * j + r) * kBRow + 8 * g]);
      for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 4; ++j)
      for (int e = 0; e < 4; ++e) sP[wave][(i * 4 + j) * 4 + e][lane] = acc[i][j][e];
  __syncthreads();
  // wave w sums and stores elements 8 w .. 8 w + 7 of every lane's tile
  for (int q = 0; q < 8; ++q) {
    const int idx = 8 * wave + q, i = idx >> 4, j = (idx >> 2) & 3, e = idx & 3;
    const float sum = sP[0][idx][lane] + sP[1][idx][lane] + sP[2][idx][lane] + sP[3][idx][lane];
    const int co = c0 + 16 * j + r;
    if (co >= Cout) continue;
    float v = sum + (bias ? bias[co] : 0.0f);
    if (relu) v = v > 0.0f ? v : 0.0f;
    const int px = p0 + 16 * i + 4 * g + e;
    y[(size_t)px * Cout + co] = (__bf16)v;
  }
}

// The forward convolution of the U-Net's channel counts.  A block takes a tile
// of 8 x 16 pixels: its input with the halo (10 x 18 pixels, every channel)
// is loaded into LDS once and serves all nine taps, and each wave multiplies
// two rows of 16 pixels by 16 NT output channels.  The kernel above fetched
// every tap's fragment from the caches and divided to find it, which cost
// about 70 operations for every two fragments.  Here a fragment is one
// 16-byte LDS read at a constant from the tap; a pixel's channels are padded
// by 16 bytes, so that eight pixels in a row start in different banks.  The
// weights pass through LDS in slices of three K steps, double-buffered (one
// slice where Cin is no multiple of 32 and K is short).  The products of a
// K step and their order are those of the other kernels, so their outputs are
// equal bit for bit; with kSplit, the sums are the four of the split-K kernel.
// The weights multiply from the left, so that a lane ends with four
// neighbouring channels of one pixel: an 8-byte store.
// Bound by LDS reads for 16 and 32 output channels and by MFMA issue and the
// tile's load for the others.  16 x 256 x 256, 16 -> 16 channels: 43 us before,
// 21 us; 16 x 64 x 64, 192 -> 64: 84 us before, 43 us (333 TFLOP/s).
constexpr int kTileH = 8, kTileW = 16, kHaloW = kTileW + 2, kHaloPix = (kTileH + 2) * kHaloW;

template <int CIN, bool kSplit>
struct ConvTile {
  static constexpr int kPixBytes = 2 * CIN + 16;
  static constexpr int kK = 9 * CIN, kChunks = (kK + 31) / 32;
  static constexpr int kSlice = CIN % 32 != 0 ? kChunks : (kSplit ? 4 : 3);  // K steps
  static constexpr int kSlices = (kChunks + kSlice - 1) / kSlice;
  static constexpr int kRow = kSlice * 32 + 8;                               // bf16 per staged weight row
  static constexpr int kXBytes = kHaloPix * kPixBytes + 16;                  // the tile, then 16 zero bytes
  static constexpr int lds(int nt) { return kXBytes + (kSlices > 1 ? 2 : 1) * 16 * nt * kRow * 2; }
};

// 8 weights of one row from memory, BF16 or rounded from the FP32 masters
template <bool kF32>
__device__ inline bf16x8 load_w8(const void* w, size_t at) {
  if (!kF32) return *reinterpret_cast<const bf16x8*>(static_cast<const __bf16*>(w) + at);
  const float4* f = reinterpret_cast<const float4*>(static_cast<const float*>(w) + at);
  const float4 a = f[0], b = f[1];
  bf16x8 v;
  v[0] = (__bf16)a.x; v[1] = (__bf16)a.y; v[2] = (__bf16)a.z; v[3] = (__bf16)a.w;
  v[4] = (__bf16)b.x; v[5] = (__bf16)b.y; v[6] = (__bf16)b.z; v[7] = (__bf16)b.w;
  return v;
}

// 8 channels of a gradient behind a ReLU: zero where the layer's output y is not positive
__device__ inline bf16x8 masked8(bf16x8 v, bf16x8 y) {
  for (int e = 0; e < 8; ++e) v[e] = (float)y[e] > 0.0f ? v[e] : (__bf16)0.0f;
  return v;
}

// kMask: the input is a gradient, masked by the output `mask` of its layer's ReLU as it is loaded
template <int CIN, int NT, bool kSplit, bool kF32, bool kMask>
__global__ __launch_bounds__(64 * kWaves) void conv_tile_kernel(const __bf16* __restrict__ x,
                                                                const void* __restrict__ w,
                                                                const float* __restrict__ bias,
                                                                __bf16* __restrict__ y, int N, int H, int W, int Cout,
                                                                int relu, const __bf16* __restrict__ mask) {
  using T = ConvTile<CIN, kSplit>;
  constexpr int kCh = 16 * NT, kSums = kSplit ? 4 : 1;
  extern __shared__ __attribute__((aligned(16))) char s_mem[];
  __bf16* s_b = reinterpret_cast<__bf16*>(s_mem + T::kXBytes);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles_x = W / kTileW, tiles_y = (H + kTileH - 1) / kTileH;
  const int n_tiles = N * tiles_x * tiles_y;
  const int bt = xcd_tile(n_tiles);
  if (bt >= n_tiles) return;  // the whole block: no barrier is skipped
  const int img = bt / (tiles_x * tiles_y), rest = bt % (tiles_x * tiles_y);
  const int y0 = rest / tiles_x * kTileH, x0 = rest % tiles_x * kTileW;
  const int ch_tiles = (Cout + kCh - 1) / kCh;
  const int r = lane & 15, g = lane >> 4;  // fragment row / k group

  // weights: slice `s` of channel tile `ct`, through registers
  constexpr int kPieces = kCh * T::kSlice * 4, kPerThread = (kPieces + 64 * kWaves - 1) / (64 * kWaves);
  bf16x8 next[kPerThread];
  auto fetch = [&](int ct, int s) {
#pragma unroll
    for (int q = 0; q < kPerThread; ++q) {
      const int t = threadIdx.x + q * 64 * kWaves;
      const int row = t / (T::kSlice * 4), k = s * T::kSlice * 32 + t % (T::kSlice * 4) * 8;
      const int co = ct * kCh + row;
      next[q] = zero8();
      if (t < kPieces && co < Cout && k < T::kK) next[q] = load_w8<kF32>(w, (size_t)co * T::kK + k);
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int q = 0; q < kPerThread; ++q) {
      const int t = threadIdx.x + q * 64 * kWaves;
      if (t < kPieces)
        *reinterpret_cast<bf16x8*>(s_b + (size_t)buf * kCh * T::kRow + t / (T::kSlice * 4) * T::kRow +
                                   t % (T::kSlice * 4) * 8) = next[q];
    }
  };
  fetch(blockIdx.y, 0);
  // the input tile
  constexpr int kXPieces = kHaloPix * (CIN / 8);
#pragma unroll 6
  for (int t = threadIdx.x; t < kXPieces; t += 64 * kWaves) {
    const int p = t / (CIN / 8), c8 = t % (CIN / 8) * 8;
    const int yy = y0 - 1 + p / kHaloW, xx = x0 - 1 + p % kHaloW;
    bf16x8 v = zero8();
    if (yy >= 0 && yy < H && xx >= 0 && xx < W) {
      const size_t at = (((size_t)img * H + yy) * W + xx) * CIN + c8;
      v = *reinterpret_cast<const bf16x8*>(x + at);
      if (kMask) v = masked8(v, *reinterpret_cast<const bf16x8*>(mask + at));
    }
    *reinterpret_cast<bf16x8*>(s_mem + p * T::kPixBytes + c8 * 2) = v;
  }
  if (threadIdx.x == 0) *reinterpret_cast<bf16x8*>(s_mem + T::kXBytes - 16) = zero8();
  stage(0);
  __syncthreads();

  const int base = (2 * wave * kHaloW + r) * T::kPixBytes + (CIN % 32 == 0 ? 16 * g : 0);
  const int row_y = y0 + 2 * wave;
  int buf = 0;
  for (int ct = blockIdx.y; ct < ch_tiles; ct += gridDim.y) {
    f32x4 acc[kSums][2][NT];
    for (int m = 0; m < kSums; ++m)
      for (int i = 0; i < 2; ++i)
        for (int j = 0; j < NT; ++j) acc[m][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < T::kSlices; ++s) {
      const bool last = s + 1 == T::kSlices;
      const bool more = !last || ct + (int)gridDim.y < ch_tiles;
      if (more && T::kSlices > 1) fetch(last ? ct + gridDim.y : ct, last ? 0 : s + 1);
#pragma unroll
      for (int q = 0; q < T::kSlice; ++q) {
        const int c = s * T::kSlice + q;
        if (T::kChunks % T::kSlice != 0 && c >= T::kChunks) break;
        int at;
        bool tail = false;
        if (CIN % 32 == 0) {
          const int tap = 32 * c / CIN;
          at = base + (tap / 3 * kHaloW + tap % 3) * T::kPixBytes + (32 * c - tap * CIN) * 2;
        } else {
          const int k = 32 * c + 8 * g, tap = k / CIN;
          tail = k >= T::kK;  // K ends inside the step: zeros
          at = base + (tap / 3 * kHaloW + tap % 3) * T::kPixBytes + (k - tap * CIN) * 2;
        }
        bf16x8 a[2], b[NT];
        for (int i = 0; i < 2; ++i)
          a[i] = *reinterpret_cast<const bf16x8*>(
              s_mem + (tail ? T::kXBytes - 16 : at + i * kHaloW * T::kPixBytes));
        for (int j = 0; j < NT; ++j)
          b[j] = *reinterpret_cast<const bf16x8*>(s_b + (size_t)buf * kCh * T::kRow + (16 * j + r) * T::kRow + 32 * q +
                                                  8 * g);
        for (int i = 0; i < 2; ++i)
          for (int j = 0; j < NT; ++j)
            acc[q % kSums][i][j] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[q % kSums][i][j], 0, 0, 0);
      }
      if (T::kSlices > 1) {
        if (more) stage(buf ^ 1);  // nobody reads it during this slice
        __syncthreads();
        buf ^= 1;
      } else if (more) {  // one slice: the next channel tile's weights replace it
        fetch(ct + gridDim.y, 0);
        __syncthreads();
        stage(0);
        __syncthreads();
      }
    }
    // C fragment: column r (pixel), rows 4 g .. 4 g + 3 (output channels)
    for (int j = 0; j < NT; ++j) {
      const int co = ct * kCh + 16 * j + 4 * g;
      if (co >= Cout) continue;
      float bb[4];
      for (int e = 0; e < 4; ++e) bb[e] = bias ? bias[co + e] : 0.0f;
      for (int i = 0; i < 2; ++i) {
        if (row_y + i >= H) continue;
        bf16x4 o;
        for (int e = 0; e < 4; ++e) {
          float v = acc[0][i][j][e];
          for (int m = 1; m < kSums; ++m) v += acc[m][i][j][e];
          v += bb[e];
          if (relu) v = v > 0.0f ? v : 0.0f;
          o[e] = (__bf16)v;
        }
        *reinterpret_cast<bf16x4*>(y + (((size_t)img * H + row_y + i) * W + x0 + r) * Cout + co) = o;
      }
    }
  }
}

struct ConvArgs {
  const __bf16* x;
  const void* w;
  const float* bias;
  __bf16* y;
  int n, h, wd, cin, cout, relu;
  const __bf16* mask;
  hipStream_t st;
};

template <int CIN, int NT, bool kSplit, bool kF32, bool kMask>
void launch_tile_nt(const ConvArgs& A) {
  const unsigned tiles = (unsigned)(A.n * (A.wd / kTileW) * ((A.h + kTileH - 1) / kTileH));
  const unsigned ch_tiles = (unsigned)((A.cout + 16 * NT - 1) / (16 * NT));
  // channel tiles in one block keep its input tile; a small image spreads them
  // over blocks.  128 x 128 images, 32 -> 96 channels at 256, 768, 1,024 and 4,096
  // tiles: 10.0, 14.3, 16.4 and 55.4 us in one block, 7.7, 15.3, 18.1 and 61.8
  // spread; 64 -> 128: 15.8, 24.3, 34.2 and 107, spread 12.1, 24.8, 33.6 and 116;
  // 128 -> 128: 22.8, 49.4, 56.2 and 204, spread 17.3, 49.0, 65.3 and 237.
  const unsigned gy = tiles >= 1024 ? 1 : ch_tiles;
  hipLaunchKernelGGL((conv_tile_kernel<CIN, NT, kSplit, kF32, kMask>), dim3((tiles + kXcds - 1) / kXcds * kXcds, gy),
                     dim3(64 * kWaves), (ConvTile<CIN, kSplit>::lds(NT)), A.st, A.x, A.w, A.bias, A.y, A.n, A.h, A.wd,
                     A.cout, A.relu, A.mask);
}

template <int CIN, bool kSplit, bool kF32, bool kMask>
void launch_tile_ch(const ConvArgs& A) {
  const long long tiles = (long long)A.n * (A.wd / kTileW) * ((A.h + kTileH - 1) / kTileH);
  int nt = A.cout % 64 == 0 ? 4 : (A.cout % 48 == 0 ? 3 : (A.cout % 32 == 0 ? 2 : 1));
  // fewer blocks than compute units: fewer channels a block (two suffice for the split sums' registers)
  while (nt % 2 == 0 && nt > 1 && (tiles * (A.cout / (16 * nt)) < 256 || (kSplit && nt > 2))) nt /= 2;
  if (nt == 4) launch_tile_nt<CIN, kSplit ? 2 : 4, kSplit, kF32, kMask>(A);
  else if (nt == 3) launch_tile_nt<CIN, 3, kSplit, kF32, kMask>(A);
  else if (nt == 2) launch_tile_nt<CIN, 2, kSplit, kF32, kMask>(A);
  else launch_tile_nt<CIN, 1, kSplit, kF32, kMask>(A);
}

// deep layers with few output tiles take four sums over the K steps
bool split_sums(const ConvArgs& A) {
  const int pix_tiles = A.n * A.h * A.wd / kFwdPix, ch_tiles = (A.cout + kFwdCh - 1) / kFwdCh;
  return 9 * A.cin >= 8 * 32 * kWaves && pix_tiles * ch_tiles < 1024;
}

// launches the tile kernel where there is one for the channel count (a
// gradient has the count of a layer's output); false: the general kernels
template <bool kF32, bool kMask>
bool launch_tile(const ConvArgs& A) {
  if (reinterpret_cast<uintptr_t>(A.y) % 8) return false;  // it stores 8 bytes at a time
  const bool split = split_sums(A);
  switch (A.cin) {
    case 16: launch_tile_ch<16, false, kF32, kMask>(A); return true;
    case 32: launch_tile_ch<32, false, kF32, kMask>(A); return true;
    case 64: launch_tile_ch<64, false, kF32, kMask>(A); return true;
    case 128:
      if (split) launch_tile_ch<128, true, kF32, kMask>(A);
      else launch_tile_ch<128, false, kF32, kMask>(A);
      return true;
    default: break;
  }
  if constexpr (!kMask) {
    switch (A.cin) {
      case 8: launch_tile_ch<8, false, kF32, false>(A); return true;
      case 48: launch_tile_ch<48, false, kF32, false>(A); return true;
      case 96: launch_tile_ch<96, false, kF32, false>(A); return true;
      case 192:
        if (split) launch_tile_ch<192, true, kF32, false>(A);
        else launch_tile_ch<192, false, kF32, false>(A);
        return true;
      default: break;
    }
  }
  return false;
}

constexpr int kWgPix = 32;   // pixels per K step
constexpr int kWgN = 64;     // (tap, ci) columns per block
constexpr int kWgMaxM = 128; // output channels per block (all of them)
// staged rows: [pixel][channel], padded by 32 bytes so that the 16 rows one
// transposing read touches per half-wave start 8 banks apart
constexpr int kWgDyRow = kWgMaxM + 16;
constexpr int kWgXRow = kWgN + 16;

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// ds_read_b64_tr_b16 (gfx950): within each group of 16 lanes, element e of
// lane i's result is 16-bit element i % 4 of the 8 bytes that lane
// 4 e + i / 4 of the group addressed (checked on the hardware).  Lane (g, j)
// of an MFMA fragment (j = lane % 16, g = lane / 16) therefore addresses
// row 4 g + j / 4 (+ 16 for the second half), column col0 + 4 (j % 4), and
// receives column col0 + j of rows 4 g .. 4 g + 3 and 16 + 4 g .. 16 + 4 g
// + 3: the fragment's k = 8 g + t is staged pixel 16 (t / 4) + 4 g + t % 4.
// Both operands use this order, so the sum over pixels is unchanged.
__device__ inline bf16x8 frag_tr(const __bf16* tile, int row_len, int col0, int g, int j) {
  const __bf16* p0 = tile + (4 * g + (j >> 2)) * row_len + col0 + 4 * (j & 3);
  const __bf16* p1 = p0 + 16 * row_len;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p0);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p1);
  const s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8, v);
}

__global__ __launch_bounds__(64 * kWaves) void conv_wgrad_kernel(const __bf16* __restrict__ x,
                                                                 const __bf16* __restrict__ dy,
                                                                 float* __restrict__ dw, int N, int H, int W,
                                                                 int Cin, int Cout, int pix_per_split) {
  // double-buffered: step k + 1's global loads are in flight while step k's
  // MFMAs run, and land in the other buffer
  __shared__ __attribute__((aligned(16))) __bf16 s_dy[2][kWgPix * kWgDyRow];  // [buf][pixel][co]
  __shared__ __attribute__((aligned(16))) __bf16 s_x[2][kWgPix * kWgXRow];    // [buf][pixel][n]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int K9 = 9 * Cin;
  const int n0 = blockIdx.x * kWgN;
  const int P = N * H * W;
  const int pbeg = blockIdx.y * pix_per_split;
  const int pend = min(P, pbeg + pix_per_split);
  const int r = lane & 15, g = lane >> 4;
  const int m_tiles = Cout / 16;
  // per thread: up to two 8-channel pieces of dY (Cout <= 128: 32 x 16 pieces)
  // and one 8-column piece of the shifted input (32 x 8 pieces)
  constexpr int kDyPieces = kWgPix * (kWgMaxM / 8) / (64 * kWaves);
  const int n_dy = kWgPix * (Cout / 8);
  bf16x8 vdy[kDyPieces], vx;
  auto load = [&](int pc) {
    for (int q = 0; q < kDyPieces; ++q) {
      const int t = threadIdx.x + q * 64 * kWaves;
      vdy[q] = zero8();
      if (t < n_dy) {
        const int p = t / (Cout / 8), c8 = (t - p * (Cout / 8)) * 8;
        const int px = pc + p;
        if (px < pend) vdy[q] = *reinterpret_cast<const bf16x8*>(dy + (size_t)px * Cout + c8);
      }
    }
    {
      const int t = threadIdx.x;  // kWgPix * kWgN / 8 == 64 * kWaves pieces
      const int p = t / (kWgN / 8), n8 = (t - p * (kWgN / 8)) * 8;
      const int n = n0 + n8, px = pc + p;
      vx = zero8();
      if (px < pend && n < K9) {
        const int tap = n / Cin, ci = n - tap * Cin;
        const int img = px / (H * W), rem = px - img * H * W, yy = rem / W + tap / 3 - 1, xs = rem % W + tap % 3 - 1;
        if (yy >= 0 && yy < H && xs >= 0 && xs < W)
          vx = *reinterpret_cast<const bf16x8*>(x + (((size_t)img * H + yy) * W + xs) * Cin + ci);
      }
    }
  };
  auto store = [&](int buf) {  // as loaded: channels contiguous, one 16-byte store per piece
    for (int q = 0; q < kDyPieces; ++q) {
      const int t = threadIdx.x + q * 64 * kWaves;
      if (t < n_dy) {
        const int p = t / (Cout / 8), c8 = (t - p * (Cout / 8)) * 8;
        *reinterpret_cast<bf16x8*>(&s_dy[buf][p * kWgDyRow + c8]) = vdy[q];
      }
    }
    const int t = threadIdx.x;
    const int p = t / (kWgN / 8), n8 = (t - p * (kWgN / 8)) * 8;
    *reinterpret_cast<bf16x8*>(&s_x[buf][p * kWgXRow + n8]) = vx;
  };
  // wave w owns column tile w (16 of the block's 64 columns) and every row tile
  f32x4 acc[kWgMaxM / 16];
  for (int i = 0; i < kWgMaxM / 16; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  int buf = 0;
  if (pbeg < pend) {
    load(pbeg);
    store(0);
  }
  __syncthreads();
  for (int pc = pbeg; pc < pend; pc += kWgPix) {
    const bool more = pc + kWgPix < pend;
    if (more) load(pc + kWgPix);
    const bf16x8 b = frag_tr(s_x[buf], kWgXRow, 16 * wave, g, r);
#pragma unroll
    for (int i = 0; i < kWgMaxM / 16; ++i) {
      if (i >= m_tiles) break;
      const bf16x8 a = frag_tr(s_dy[buf], kWgDyRow, 16 * i, g, r);
      acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[i], 0, 0, 0);
    }
    if (more) store(buf ^ 1);  // the other buffer: nobody reads it during this step
    __syncthreads();
    buf ^= 1;
  }
  // C fragment: column n = n0 + 16 wave + r, rows co = 16 i + 4 g + e
  const int n = n0 + 16 * wave + r;
  if (n >= K9) return;
#pragma unroll
  for (int i = 0; i < kWgMaxM / 16; ++i) {
    if (i >= m_tiles) break;
    for (int e = 0; e < 4; ++e) {
      const int co = 16 * i + 4 * g + e;
      unsafeAtomicAdd(&dw[(size_t)co * K9 + n], acc[i][e]);
    }
  }
}

// The weight gradient from tiles.  The kernel above gives each 64 columns
// (tap, ci) a block of their own, which loads its pixels' dY and one shifted
// input per tap: dY crosses LDS once per 64 columns and the input nine times.
// Here a block loads dY of 8 x 16 pixels and the input with its halo once for
// all nine taps (a tap is an offset of the transposing read), for 16 MT output
// and 16 CIT input channels; a wave takes two image rows, i.e. one K step of
// 32 pixels, and keeps all MT x CIT x 9 <= 36 sums in registers over the
// tiles its block walks.  The waves' sums meet in LDS, and a block adds each
// weight to memory once.  Staged rows are an odd multiple of 32 bytes, so the
// four rows that 16 lanes read lie in different banks.  Bound by LDS reads
// for few output channels (one fragment feeds MT products) and by the tiles'
// load from L2 otherwise, with the additions to memory on top.  16 x 256 x 256,
// 48 -> 16 channels: 217 us before, 46 us; 16 x 64 x 64, 192 -> 64: 127 us
// before, 44 us.
template <int MT, int CIT, bool kC8>
struct WgTile {
  static constexpr int kDyRow = MT == 1 ? 16 : 16 * MT + 16;            // bf16 per staged pixel
  static constexpr int kXRow = kC8 ? 8 : (CIT % 2 ? 16 * CIT : 16 * CIT + 16);
  static constexpr int kCols = kC8 ? 5 : 9 * CIT;                        // column tiles of 16
  static constexpr int kDyBytes = kTileH * kTileW * kDyRow * 2, kXBytes = kHaloPix * kXRow * 2;
  static constexpr int kSumBytes = MT * kCols * 64 * 16;
  static constexpr int kPart = MT * kCols * 256 + 16 * MT;  // floats of a block's sums: weights, then bias
  // the weight that float k of the sums belongs to, -1 for none: C fragments
  // of (row tile, column tile), lane, then row 4 (lane / 16) + e, column lane % 16
  static __host__ __device__ int weight(int k, int cin, int co0, int ci0) {
    const int e = k & 3, l = k >> 2 & 63, i = k / 256 / kCols, c = k / 256 % kCols, col = l & 15;
    const int tap = kC8 ? 2 * c + (col >> 3) : c / CIT, ch = kC8 ? col & 7 : 16 * (c % CIT) + col;
    return tap < 9 ? ((co0 + 16 * i + 4 * (l >> 4) + e) * 9 + tap) * cin + ci0 + ch : -1;
  }
  static constexpr int lds() {
    return kDyBytes + kXBytes > kSumBytes ? kDyBytes + kXBytes : kSumBytes;
  }
};

template <int MT, int CIT, bool kC8, bool kMask>
__global__ __launch_bounds__(64 * kWaves, 2) void conv_wgrad_tile_kernel(const __bf16* __restrict__ x,
                                                                         const __bf16* __restrict__ dy,
                                                                         float* __restrict__ dw, int N, int H, int W,
                                                                         int Cin, int Cout,
                                                                         const __bf16* __restrict__ mask,
                                                                         float* __restrict__ part) {
  using T = WgTile<MT, CIT, kC8>;
  constexpr int kCi = kC8 ? 8 : 16 * CIT, kCo = 16 * MT;
  extern __shared__ __attribute__((aligned(16))) char s_mem[];
  __bf16* s_dy = reinterpret_cast<__bf16*>(s_mem);
  __bf16* s_x = reinterpret_cast<__bf16*>(s_mem + T::kDyBytes);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = lane & 15, g = lane >> 4;
  const int co_groups = Cout / kCo;
  const int co0 = (int)(blockIdx.y % co_groups) * kCo, ci0 = (int)(blockIdx.y / co_groups) * kCi;
  const int tiles_x = W / kTileW, tiles_y = (H + kTileH - 1) / kTileH;
  const int n_tiles = N * tiles_x * tiles_y;

  constexpr int kDyPieces = kTileH * kTileW * kCo / 8, kXPieces = kHaloPix * kCi / 8;
  constexpr int kDyPer = (kDyPieces + 64 * kWaves - 1) / (64 * kWaves);
  constexpr int kXPer = (kXPieces + 64 * kWaves - 1) / (64 * kWaves);
  bf16x8 vdy[kDyPer], vmask[kMask ? kDyPer : 1], vx[kXPer];
  // the bias gradient: a thread's pieces of dY are the same 8 channels every time
  static_assert(64 * kWaves % (kCo / 8) == 0, "a thread keeps its 8 channels");
  float bias_sum[8];
  for (int e = 0; e < 8; ++e) bias_sum[e] = 0.0f;
  auto fetch = [&](int tile) {
    const int img = tile / (tiles_x * tiles_y), rest = tile % (tiles_x * tiles_y);
    const int y0 = rest / tiles_x * kTileH, x0 = rest % tiles_x * kTileW;
#pragma unroll
    for (int q = 0; q < kDyPer; ++q) {
      const int t = threadIdx.x + q * 64 * kWaves;
      const int p = t / (kCo / 8), c8 = t % (kCo / 8) * 8;
      const int yy = y0 + p / kTileW, xx = x0 + p % kTileW;
      vdy[q] = zero8();
      if (t < kDyPieces && yy < H) {
        const size_t at = (((size_t)img * H + yy) * W + xx) * Cout + co0 + c8;
        vdy[q] = *reinterpret_cast<const bf16x8*>(dy + at);
        if (kMask) vmask[q] = *reinterpret_cast<const bf16x8*>(mask + at);
      }
    }
#pragma unroll
    for (int q = 0; q < kXPer; ++q) {
      const int t = threadIdx.x + q * 64 * kWaves;
      const int p = t / (kCi / 8), c8 = t % (kCi / 8) * 8;
      const int yy = y0 - 1 + p / kHaloW, xx = x0 - 1 + p % kHaloW;
      vx[q] = zero8();
      if (t < kXPieces && yy >= 0 && yy < H && xx >= 0 && xx < W)
        vx[q] = *reinterpret_cast<const bf16x8*>(x + (((size_t)img * H + yy) * W + xx) * Cin + ci0 + c8);
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int q = 0; q < kDyPer; ++q) {
      const int t = threadIdx.x + q * 64 * kWaves;
      if (t < kDyPieces) {
        if (kMask) vdy[q] = masked8(vdy[q], vmask[q]);
        *reinterpret_cast<bf16x8*>(s_dy + t / (kCo / 8) * T::kDyRow + t % (kCo / 8) * 8) = vdy[q];
        if (part)
          for (int e = 0; e < 8; ++e) bias_sum[e] += (float)vdy[q][e];
      }
    }
#pragma unroll
    for (int q = 0; q < kXPer; ++q) {
      const int t = threadIdx.x + q * 64 * kWaves;
      if (t < kXPieces) *reinterpret_cast<bf16x8*>(s_x + t / (kCi / 8) * T::kXRow + t % (kCi / 8) * 8) = vx[q];
    }
  };
  // column tile c of 16 columns: tap and first channel; with 8 channels a
  // tile holds two taps, whose columns the lanes' addresses tell apart
  auto x_at = [&](int c) {
    const int q = j & 3;
    const int tap = kC8 ? (2 * c + (q >> 1) < 9 ? 2 * c + (q >> 1) : 8) : c / CIT;
    const int ch = kC8 ? 4 * (q & 1) : 16 * (c % CIT) + 4 * q;
    return s_x + ((2 * wave + tap / 3) * kHaloW + tap % 3 + 4 * g + (j >> 2)) * T::kXRow + ch;
  };
  auto frag = [](const __bf16* p0, const __bf16* p1) {
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p0);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p1);
    return __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  f32x4 acc[MT][T::kCols];
  for (int i = 0; i < MT; ++i)
    for (int c = 0; c < T::kCols; ++c) acc[i][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  int tile = blockIdx.x;
  if (tile < n_tiles) fetch(tile);
  for (; tile < n_tiles; tile += gridDim.x) {
    store();
    __syncthreads();
    if (tile + (int)gridDim.x < n_tiles) fetch(tile + gridDim.x);  // in flight during this tile's products
    const int y0 = tile % (tiles_x * tiles_y) / tiles_x * kTileH;
    if (y0 + 2 * wave < H) {  // H is even: both of the wave's rows or none
      bf16x8 a[MT];
      for (int i = 0; i < MT; ++i) {
        const __bf16* p0 = s_dy + (32 * wave + 4 * g + (j >> 2)) * T::kDyRow + 16 * i + 4 * (j & 3);
        a[i] = frag(p0, p0 + 16 * T::kDyRow);
      }
#pragma unroll
      for (int c = 0; c < T::kCols; ++c) {
        const __bf16* p0 = x_at(c);
        const bf16x8 b = frag(p0, p0 + kHaloW * T::kXRow);
#pragma unroll
        for (int i = 0; i < MT; ++i)
          acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b, acc[i][c], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // the waves' sums, one wave after the other, then one addition per weight
  f32x4* s_sum = reinterpret_cast<f32x4*>(s_mem);
  for (int w = 0; w < kWaves; ++w) {
    if (wave == w) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int c = 0; c < T::kCols; ++c) {
          f32x4* at = s_sum + (i * T::kCols + c) * 64 + lane;
          *at = w == 0 ? acc[i][c] : *at + acc[i][c];
        }
    }
    __syncthreads();
  }
  if (part) {
    // this block's sums, for wgrad_sum_kernel
    float* mine = part + ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * T::kPart;
    for (int t = threadIdx.x; t < MT * T::kCols * 64; t += 64 * kWaves) reinterpret_cast<f32x4*>(mine)[t] = s_sum[t];
    for (int off = 32; off >= kCo / 8; off >>= 1)
      for (int e = 0; e < 8; ++e) bias_sum[e] += __shfl_xor(bias_sum[e], off, 64);
    __syncthreads();
    float* s_bias = reinterpret_cast<float*>(s_mem);
    if (lane < kCo / 8)
      for (int e = 0; e < 8; ++e) s_bias[wave * kCo + lane * 8 + e] = bias_sum[e];
    __syncthreads();
    if (threadIdx.x < kCo)
      mine[MT * T::kCols * 256 + threadIdx.x] = (s_bias[threadIdx.x] + s_bias[kCo + threadIdx.x]) +
                                                (s_bias[2 * kCo + threadIdx.x] + s_bias[3 * kCo + threadIdx.x]);
    return;
  }
  for (int t = threadIdx.x; t < MT * T::kCols * 64; t += 64 * kWaves) {
    const f32x4 v = s_sum[t];
    for (int e = 0; e < 4; ++e) {
      const int at = T::weight(4 * t + e, Cin, co0, ci0);
      if (at >= 0) unsafeAtomicAdd(&dw[at], v[e]);
    }
  }
}

// The blocks' sums into dw and db: thread k of a group's sums adds kSumRun
// blocks in order, and one addition to memory takes the place of kSumRun.
// (Added by the blocks themselves, the weights of a layer met up to 512 times
// at the same addresses, and that took longer than the products.)
constexpr int kSumBlock = 256, kSumRun = 32;
template <int MT, int CIT, bool kC8>
__global__ __launch_bounds__(kSumBlock) void wgrad_sum_kernel(const float* __restrict__ part, int splits,
                                                              float* __restrict__ dw, float* __restrict__ db, int Cin,
                                                              int Cout) {
  using T = WgTile<MT, CIT, kC8>;
  const int k = blockIdx.x * kSumBlock + threadIdx.x;
  if (k >= T::kPart) return;
  const int co_groups = Cout / (16 * MT), group = blockIdx.z;
  const int co0 = group % co_groups * 16 * MT, ci0 = group / co_groups * (kC8 ? 8 : 16 * CIT);
  const int first = blockIdx.y * kSumRun, last = min(splits, first + kSumRun);
  const float* at = part + ((size_t)group * splits + first) * T::kPart + k;
  float sum = 0.0f;
#pragma unroll 8
  for (int s = first; s < last; ++s, at += T::kPart) sum += *at;
  constexpr int kWeights = MT * T::kCols * 256;
  if (k >= kWeights) {
    if (ci0 == 0) unsafeAtomicAdd(&db[co0 + k - kWeights], sum);
  } else {
    const int w = T::weight(k, Cin, co0, ci0);
    if (w >= 0) unsafeAtomicAdd(&dw[w], sum);
  }
}

struct WgradArgs {
  const __bf16 *x, *dy;
  float* dw;
  int n, h, wd, cin, cout;
  const __bf16* mask;  // the layer's output behind its ReLU, or null
  float *db, *part;    // the bias gradient and the blocks' sums, or null: blocks add to dw
  hipStream_t st;
};

int wgrad_tiles(const WgradArgs& A) { return A.n * (A.wd / kTileW) * ((A.h + kTileH - 1) / kTileH); }

// work: the blocks' sums go to a work space
template <int MT, int CIT, bool kC8>
int wgrad_splits(const WgradArgs& A, bool work, int* groups) {
  const int tiles = wgrad_tiles(A);
  *groups = (A.cout / (16 * MT)) * (kC8 ? 1 : A.cin / (16 * CIT));
  // each block walks its share of the tiles.  Two blocks of the large variants
  // fit a compute unit; one with 9 sums or fewer leaves room for four (512 and
  // 1,024 blocks: 25.2 and 22.9 us at 16 x 256 x 256, 16 -> 16, but 20 and 30 us
  // at 128 x 128, 32 -> 32)
  int blocks = MT * WgTile<MT, CIT, kC8>::kCols <= 9 ? 1024 : 512;
  // Blocks that add to dw themselves: each adds its group's weights once, at the
  // addresses of every other block of the group, so their number weighs against
  // the tiles a block walks.  The best of 32 to 1,024 blocks over 19 layer shapes
  // at batch 1, 4 and 16 grows with the root of the tiles, and less than the
  // groups do (128 x 128, 32 -> 32 channels, batch 4: 18.6 us, 37 with 512 blocks;
  // 64 x 64, 64 -> 16, batch 16: 21 and 44; 256 x 256, 16 -> 16, batch 16: 29 and
  // 42 with 1,024).
  if (!work) blocks = std::min(blocks, (int)(4.5f * std::sqrt((float)tiles) * std::pow((float)*groups, 2.0f / 3.0f)));
  return std::max(1, std::min(tiles, blocks / *groups));
}

// launches the kernels; with `floats`, only says how much `part` must hold
template <int MT, int CIT, bool kC8>
void launch_wgrad_tile(const WgradArgs& A, size_t* floats) {
  int groups;
  const int splits = wgrad_splits<MT, CIT, kC8>(A, A.part || floats, &groups);
  using T = WgTile<MT, CIT, kC8>;
  if (floats) {
    *floats = (size_t)groups * splits * T::kPart;
    return;
  }
  const dim3 grid(splits, groups), block(64 * kWaves);
  if (A.mask)
    hipLaunchKernelGGL((conv_wgrad_tile_kernel<MT, CIT, kC8, true>), grid, block, T::lds(), A.st, A.x, A.dy, A.dw, A.n,
                       A.h, A.wd, A.cin, A.cout, A.mask, A.part);
  else
    hipLaunchKernelGGL((conv_wgrad_tile_kernel<MT, CIT, kC8, false>), grid, block, T::lds(), A.st, A.x, A.dy, A.dw,
                       A.n, A.h, A.wd, A.cin, A.cout, A.mask, A.part);
  if (A.part)
    hipLaunchKernelGGL((wgrad_sum_kernel<MT, CIT, kC8>),
                       dim3((T::kPart + kSumBlock - 1) / kSumBlock, (splits + kSumRun - 1) / kSumRun, groups),
                       dim3(kSumBlock), 0, A.st, A.part, splits, A.dw, A.db, A.cin, A.cout);
}

// false: the general kernel (a height that leaves a wave one row, channels that do not fill a tile)
bool wgrad_tile(const WgradArgs& A, size_t* floats = nullptr) {
  const int cin = A.cin, cout = A.cout;
  if (A.h % 2 || (cin != 8 && cin % 16)) return false;
  if (cout % 64 == 0) {
    if (cin == 8) launch_wgrad_tile<4, 1, true>(A, floats);
    else launch_wgrad_tile<4, 1, false>(A, floats);
  } else if (cout % 32 == 0) {
    if (cin == 8) launch_wgrad_tile<2, 1, true>(A, floats);
    else if (cin % 32 == 0) launch_wgrad_tile<2, 2, false>(A, floats);
    else launch_wgrad_tile<2, 1, false>(A, floats);
  } else {
    if (cin == 8) launch_wgrad_tile<1, 1, true>(A, floats);
    else if (cin % 64 == 0) launch_wgrad_tile<1, 4, false>(A, floats);
    else if (cin % 48 == 0) launch_wgrad_tile<1, 3, false>(A, floats);
    else if (cin % 32 == 0) launch_wgrad_tile<1, 2, false>(A, floats);
    else launch_wgrad_tile<1, 1, false>(A, floats);
  }
  return true;
}

// The backward of a layer's ReLU and bias in one pass: dy_out = dy where
// the layer's output y > 0 (everywhere without ReLU), as BF16, and
// db[c] += sum over pixels of dy_out[., c] in FP32.  A thread takes 8
// channels of a pixel; the grid's thread count is a multiple of C / 8, so a
// thread keeps the same 8 channels over its whole grid-stride loop and sums
// them in registers; the wave folds those sums onto its first C / 8 lanes,
// which add them into the block's LDS sums, and one global atomic per
// channel and block finishes.
constexpr int kMaskBlock = 256;

template <bool kF32>
__global__ __launch_bounds__(kMaskBlock) void relu_bias_backward_kernel(const void* __restrict__ dy_in,
                                                                        const __bf16* __restrict__ y, int relu,
                                                                        __bf16* __restrict__ dy_out,
                                                                        float* __restrict__ db, long long pieces,
                                                                        int C) {
  __shared__ float s_db[kWgMaxM];
  for (int i = threadIdx.x; i < C; i += kMaskBlock) s_db[i] = 0.0f;
  __syncthreads();
  const int groups = C / 8;
  const long long stride = (long long)gridDim.x * kMaskBlock;
  long long q = (long long)blockIdx.x * kMaskBlock + threadIdx.x;
  const int c8 = (int)(q % groups) * 8;  // the same for every q of this thread: stride % groups == 0
  float acc[8];
  for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
  for (; q < pieces; q += stride) {
    float v[8];
    if (kF32) {
      const float4* src = reinterpret_cast<const float4*>(static_cast<const float*>(dy_in) + q * 8);
      const float4 a = src[0], b = src[1];
      v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
      const bf16x8 d = reinterpret_cast<const bf16x8*>(dy_in)[q];
      for (int e = 0; e < 8; ++e) v[e] = (float)d[e];
    }
    bf16x8 o;
    if (relu) {
      const bf16x8 yy = reinterpret_cast<const bf16x8*>(y)[q];
      for (int e = 0; e < 8; ++e) o[e] = (float)yy[e] > 0.0f ? (__bf16)v[e] : (__bf16)0.0f;
    } else {
      for (int e = 0; e < 8; ++e) o[e] = (__bf16)v[e];
    }
    reinterpret_cast<bf16x8*>(dy_out)[q] = o;
    for (int e = 0; e < 8; ++e) acc[e] += (float)o[e];
  }
  // lanes l and l xor off (off a multiple of C / 8, a power of two) hold the
  // same channels: fold the wave onto its first C / 8 lanes, which then add
  // into the block's sums
  for (int off = 32; off >= groups; off >>= 1)
    for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], off, 64);
  if ((int)(threadIdx.x & 63) < groups)
    for (int e = 0; e < 8; ++e) atomicAdd(&s_db[c8 + e], acc[e]);
  __syncthreads();
  for (int i = threadIdx.x; i < C; i += kMaskBlock) unsafeAtomicAdd(&db[i], s_db[i]);
}

// The U-Net's 2 x 2 max pooling and its nearest-neighbour upsampling with
// the skip concatenation, NHWC BF16, one thread per 8 channels of a pixel:
// bandwidth kernels in place of the strided copies, reductions and masks
// that the same steps take as tensor operations.  The pooling keeps, per
// channel, which input of the window (row-major: 0 top left .. 3 bottom
// right) held the first maximum, and its backward routes the gradient
// there, as max_pool2d does.
constexpr int kGlueBlock = 256;

unsigned glue_grid(long long pieces) {
  const long long b = (pieces + kGlueBlock - 1) / kGlueBlock;
  return (unsigned)(b < 4096 ? (b > 0 ? b : 1) : 4096);
}

__global__ __launch_bounds__(kGlueBlock) void pool2x2_kernel(const __bf16* __restrict__ x, __bf16* __restrict__ y,
                                                             uint8_t* __restrict__ arg, int n, int h, int w, int c) {
  const int ho = h / 2, wo = w / 2, g = c / 8;
  const long long total = (long long)n * ho * wo * g;
  for (long long q = blockIdx.x * (long long)kGlueBlock + threadIdx.x; q < total;
       q += (long long)gridDim.x * kGlueBlock) {
    const int c8 = (int)(q % g) * 8;
    long long p = q / g;  // output pixel
    const int xo = (int)(p % wo);
    p /= wo;
    const int yo = (int)(p % ho);
    const long long img = p / ho;
    const __bf16* base = x + ((img * h + 2 * yo) * (long long)w + 2 * xo) * c + c8;
    bf16x8 v[4];
    v[0] = *reinterpret_cast<const bf16x8*>(base);
    v[1] = *reinterpret_cast<const bf16x8*>(base + c);
    v[2] = *reinterpret_cast<const bf16x8*>(base + (long long)w * c);
    v[3] = *reinterpret_cast<const bf16x8*>(base + (long long)w * c + c);
    bf16x8 m;
    uint64_t a = 0;
    for (int e = 0; e < 8; ++e) {
      float best = (float)v[0][e];
      int bi = 0;
      for (int k = 1; k < 4; ++k) {
        const float t = (float)v[k][e];
        if (t > best) {
          best = t;
          bi = k;
        }
      }
      m[e] = v[bi][e];
      a |= (uint64_t)bi << (8 * e);
    }
    *reinterpret_cast<bf16x8*>(y + q * 8) = m;  // output pixel p, channels c8.. : element p c + c8 = 8 q
    *reinterpret_cast<uint64_t*>(arg + q * 8) = a;
  }
}

__global__ __launch_bounds__(kGlueBlock) void pool2x2_backward_kernel(const __bf16* __restrict__ dy,
                                                                      const uint8_t* __restrict__ arg,
                                                                      __bf16* __restrict__ dx, int n, int h, int w,
                                                                      int c) {
  const int ho = h / 2, wo = w / 2, g = c / 8;
  const long long total = (long long)n * ho * wo * g;
  for (long long q = blockIdx.x * (long long)kGlueBlock + threadIdx.x; q < total;
       q += (long long)gridDim.x * kGlueBlock) {
    const int c8 = (int)(q % g) * 8;
    long long p = q / g;
    const int xo = (int)(p % wo);
    p /= wo;
    const int yo = (int)(p % ho);
    const long long img = p / ho;
    const bf16x8 d = *reinterpret_cast<const bf16x8*>(dy + q * 8);
    const uint64_t a = *reinterpret_cast<const uint64_t*>(arg + q * 8);
    __bf16* base = dx + ((img * h + 2 * yo) * (long long)w + 2 * xo) * c + c8;
    __bf16* out[4] = {base, base + c, base + (long long)w * c, base + (long long)w * c + c};
    for (int k = 0; k < 4; ++k) {
      bf16x8 v;
      for (int e = 0; e < 8; ++e) v[e] = ((a >> (8 * e)) & 0xffu) == (uint64_t)k ? d[e] : (__bf16)0.0f;
      *reinterpret_cast<bf16x8*>(out[k]) = v;
    }
  }
}

// out [n][h][w][cz + cs] = (z upsampled 2x by repetition, s): the decoder's
// input, channels of z first
__global__ __launch_bounds__(kGlueBlock) void upcat_kernel(const __bf16* __restrict__ z, const __bf16* __restrict__ s,
                                                           __bf16* __restrict__ out, int n, int h, int w, int cz,
                                                           int cs) {
  const int g = (cz + cs) / 8;
  const long long total = (long long)n * h * w * g;
  for (long long q = blockIdx.x * (long long)kGlueBlock + threadIdx.x; q < total;
       q += (long long)gridDim.x * kGlueBlock) {
    const int c8 = (int)(q % g) * 8;
    long long p = q / g;
    const int xx = (int)(p % w);
    p /= w;
    const int yy = (int)(p % h);
    const long long img = p / h;
    const bf16x8 v = c8 < cz
        ? *reinterpret_cast<const bf16x8*>(z + ((img * (h / 2) + yy / 2) * (long long)(w / 2) + xx / 2) * cz + c8)
        : *reinterpret_cast<const bf16x8*>(s + ((img * h + yy) * (long long)w + xx) * cs + (c8 - cz));
    *reinterpret_cast<bf16x8*>(out + q * 8) = v;
  }
}

// backward of upcat: dz = the sum of dout's z channels over each 2 x 2 block
// (FP32, one rounding), ds = dout's s channels
__global__ __launch_bounds__(kGlueBlock) void upcat_backward_kernel(const __bf16* __restrict__ dout,
                                                                    __bf16* __restrict__ dz, __bf16* __restrict__ ds,
                                                                    int n, int h, int w, int cz, int cs) {
  const int ct = cz + cs, gz = cz / 8, gs = cs / 8;
  const long long nz = (long long)n * (h / 2) * (w / 2) * gz, ns = (long long)n * h * w * gs;
  for (long long q = blockIdx.x * (long long)kGlueBlock + threadIdx.x; q < nz + ns;
       q += (long long)gridDim.x * kGlueBlock) {
    if (q < nz) {
      const int c8 = (int)(q % gz) * 8;
      long long p = q / gz;
      const int xo = (int)(p % (w / 2));
      p /= (w / 2);
      const int yo = (int)(p % (h / 2));
      const long long img = p / (h / 2);
      const __bf16* base = dout + ((img * h + 2 * yo) * (long long)w + 2 * xo) * ct + c8;
      const bf16x8 v0 = *reinterpret_cast<const bf16x8*>(base);
      const bf16x8 v1 = *reinterpret_cast<const bf16x8*>(base + ct);
      const bf16x8 v2 = *reinterpret_cast<const bf16x8*>(base + (long long)w * ct);
      const bf16x8 v3 = *reinterpret_cast<const bf16x8*>(base + (long long)w * ct + ct);
      bf16x8 o;
      for (int e = 0; e < 8; ++e) o[e] = (__bf16)((((float)v0[e] + (float)v1[e]) + (float)v2[e]) + (float)v3[e]);
      *reinterpret_cast<bf16x8*>(dz + q * 8) = o;
    } else {
      const long long r = q - nz;
      const int c8 = (int)(r % gs) * 8;
      const long long p = r / gs;
      *reinterpret_cast<bf16x8*>(ds + r * 8) = *reinterpret_cast<const bf16x8*>(dout + p * ct + cz + c8);
    }
  }
}

// The BF16 operands of a layer's forward and data-gradient convolutions from
// its FP32 master weights, in one pass: w [cout][9][cin] rounded to nearest
// even, and the data gradient's weights [cin][9][cout] with the taps
// reversed (tap 8 - t), in place of a cast, a flip and a transposing copy.
constexpr int kPrepBlock = 256;
__global__ __launch_bounds__(kPrepBlock) void weights_bf16_kernel(const float* __restrict__ w, __bf16* __restrict__ wb,
                                                                   __bf16* __restrict__ wt, float* __restrict__ dw,
                                                                   float* __restrict__ db, int cout, int cin) {
  const int n = cout * 9 * cin;
  for (int i = blockIdx.x * kPrepBlock + threadIdx.x; i < n; i += gridDim.x * kPrepBlock) {
    const int ci = i % cin, t = (i / cin) % 9, co = i / (9 * cin);
    const __bf16 v = (__bf16)w[i];
    wb[i] = v;
    wt[((size_t)ci * 9 + (8 - t)) * cout + co] = v;
    // the layer's gradient accumulators, zeroed here instead of by fills of their own
    if (dw) dw[i] = 0.0f;
    if (db && i < cout) db[i] = 0.0f;
  }
}

// The network's input: k <= 8 FP32 channels as BF16, zero-padded to 8.
__global__ __launch_bounds__(kGlueBlock) void pad8_kernel(const float* __restrict__ x, __bf16* __restrict__ z,
                                                          long long pixels, int k) {
  for (long long p = blockIdx.x * (long long)kGlueBlock + threadIdx.x; p < pixels;
       p += (long long)gridDim.x * kGlueBlock) {
    bf16x8 v = zero8();
    for (int c = 0; c < 8; ++c)
      if (c < k) v[c] = (__bf16)x[p * k + c];
    *reinterpret_cast<bf16x8*>(z + 8 * p) = v;
  }
}

// The 16 -> 1 head in one pass: out = sum_c z_c head_c + bias in FP32, one
// thread a pixel.  The sixteen products are added in the order the tensor
// reduction was seen to take (neighbours, then neighbouring pairs), which a
// test holds bit for bit.  As tensor operations the head wrote and read an FP32 copy of
// its input twice: 62 us at 16 x 256 x 256, 7.5 us here.
constexpr int kHeadCh = 16;
__global__ __launch_bounds__(kGlueBlock) void head_kernel(const __bf16* __restrict__ z, const float* __restrict__ head,
                                                          const float* __restrict__ bias, float* __restrict__ out,
                                                          long long pixels) {
  for (long long p = blockIdx.x * (long long)kGlueBlock + threadIdx.x; p < pixels;
       p += (long long)gridDim.x * kGlueBlock) {
    const bf16x8 a = *reinterpret_cast<const bf16x8*>(z + kHeadCh * p);
    const bf16x8 b = *reinterpret_cast<const bf16x8*>(z + kHeadCh * p + 8);
    float m[kHeadCh];
    for (int c = 0; c < 8; ++c) {
      m[c] = (float)a[c] * head[c];
      m[8 + c] = (float)b[c] * head[8 + c];
    }
#pragma unroll
    for (int left = kHeadCh / 2; left > 0; left /= 2)
      for (int c = 0; c < left; ++c) m[c] = m[2 * c] + m[2 * c + 1];
    out[p] = m[0] + bias[0];
  }
}

// Its backward: dz_c = dout head_c rounded to BF16, dhead_c += sum over pixels
// of dout z_c, dbias += sum of dout.  Four tensor kernels and a reduction
// before, 125 us at 16 x 256 x 256; 19 us.
__global__ __launch_bounds__(kGlueBlock) void head_backward_kernel(const float* __restrict__ dout,
                                                                   const __bf16* __restrict__ z,
                                                                   const float* __restrict__ head,
                                                                   __bf16* __restrict__ dz, float* __restrict__ dhead,
                                                                   float* __restrict__ dbias, long long pixels) {
  __shared__ float s_sum[kHeadCh + 1][kGlueBlock / 64];
  float acc[kHeadCh + 1];
  for (int c = 0; c <= kHeadCh; ++c) acc[c] = 0.0f;
  for (long long p = blockIdx.x * (long long)kGlueBlock + threadIdx.x; p < pixels;
       p += (long long)gridDim.x * kGlueBlock) {
    const float d = dout[p];
    acc[kHeadCh] += d;
    for (int h = 0; h < 2; ++h) {
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(z + kHeadCh * p + 8 * h);
      bf16x8 o;
      for (int c = 0; c < 8; ++c) {
        acc[8 * h + c] += d * (float)v[c];
        o[c] = (__bf16)(d * head[8 * h + c]);
      }
      *reinterpret_cast<bf16x8*>(dz + kHeadCh * p + 8 * h) = o;
    }
  }
  for (int c = 0; c <= kHeadCh; ++c) {
    for (int off = 32; off > 0; off >>= 1) acc[c] += __shfl_xor(acc[c], off, 64);
    if ((threadIdx.x & 63) == 0) s_sum[c][threadIdx.x >> 6] = acc[c];
  }
  __syncthreads();
  if (threadIdx.x <= kHeadCh) {
    float t = 0.0f;
    for (int w = 0; w < kGlueBlock / 64; ++w) t += s_sum[threadIdx.x][w];
    unsafeAtomicAdd(threadIdx.x < kHeadCh ? &dhead[threadIdx.x] : dbias, t);
  }
}

bool shapes_ok(int N, int H, int W, int Cin, int Cout) {
  return N > 0 && H > 0 && W > 0 && W % 16 == 0 && ((long long)N * H * W) % kFwdPix == 0 && Cin > 0 &&
         Cin % 8 == 0 && Cout > 0 && Cout % 16 == 0 && (long long)N * H * W * (Cin > Cout ? Cin : Cout) < (1ll << 31);
}

}  // namespace

extern "C" {

const char* ggh_unet_last_error(void) { return g_unet_error.c_str(); }

int ggh_conv3x3_forward(const void* x, const void* w, const float* bias, void* y, int32_t n, int32_t h, int32_t wd,
                        int32_t cin, int32_t cout, int32_t relu, void* stream) {
  if (!x || !w || !y) return ufail(-1, "null pointer");
  if (!shapes_ok(n, h, wd, cin, cout)) return ufail(-2, "unsupported shape (W % 16, N H W % 32, Cin % 8, Cout % 16)");
  const int pix_tiles = n * h * wd / kFwdPix, ch_tiles = (cout + kFwdCh - 1) / kFwdCh;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  const __bf16 *xb = static_cast<const __bf16*>(x), *wb = static_cast<const __bf16*>(w);
  __bf16* yb = static_cast<__bf16*>(y);
  const ConvArgs args = {xb, w, bias, yb, n, h, wd, cin, cout, relu, nullptr, st};
  if (launch_tile<false, false>(args)) {
    // the U-Net's channel counts
  } else if (split_sums(args)) {
    const dim3 grid((unsigned)((pix_tiles * ch_tiles + kXcds - 1) / kXcds * kXcds));
    hipLaunchKernelGGL(conv_fwd_splitk_kernel, grid, dim3(64 * kWaves), 0, st, xb, wb, bias, yb, n, h, wd, cin, cout,
                       relu);
  } else {
    // output channels per wave: 64, or 16 / 32 for the narrow layers
    const int nt = cout >= 64 ? 4 : (cout >= 32 ? 2 : 1);
    const int block_tiles = ((pix_tiles + kWaves - 1) / kWaves) * ((cout + 16 * nt - 1) / (16 * nt));
    const dim3 grid((unsigned)((block_tiles + kXcds - 1) / kXcds * kXcds));
    if (nt == 4)
      hipLaunchKernelGGL(conv_fwd_kernel<4>, grid, dim3(64 * kWaves), 0, st, xb, wb, bias, yb, n, h, wd, cin, cout, relu);
    else if (nt == 2)
      hipLaunchKernelGGL(conv_fwd_kernel<2>, grid, dim3(64 * kWaves), 0, st, xb, wb, bias, yb, n, h, wd, cin, cout, relu);
    else
      hipLaunchKernelGGL(conv_fwd_kernel<1>, grid, dim3(64 * kWaves), 0, st, xb, wb, bias, yb, n, h, wd, cin, cout, relu);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ufail(-100 - (int)e, std::string("conv forward: ") + hipGetErrorString(e));
  return 0;
}

int ggh_relu_bias_backward(const void* dy, int32_t dy_is_f32, const void* y, int32_t relu, void* dy_out, float* db,
                           int64_t n_pixels, int32_t c, void* stream) {
  if (!dy || !dy_out || !db || (relu && !y)) return ufail(-1, "null pointer");
  // C / 8 must divide the block size (a thread keeps its 8 channels)
  if (n_pixels <= 0 || (c != 8 && c != 16 && c != 32 && c != 64 && c != 128))
    return ufail(-2, "unsupported shape (C one of 8, 16, 32, 64, 128)");
  const long long pieces = (long long)n_pixels * (c / 8);
  const long long want = (pieces + kMaskBlock - 1) / kMaskBlock;
  // one block per compute unit: every block ends with one global atomic per
  // channel onto the same C addresses, and more blocks queue up there
  // (measured over a training run: 92.7 ms at 256 blocks, 100 at 512, 143 at
  // 1,024, 294 at 4,096, 125 at 128)
  const unsigned blocks = (unsigned)(want < 256 ? want : 256);
  const hipStream_t st = static_cast<hipStream_t>(stream);
  if (dy_is_f32)
    hipLaunchKernelGGL(relu_bias_backward_kernel<true>, dim3(blocks), dim3(kMaskBlock), 0, st, dy,
                       static_cast<const __bf16*>(y), relu, static_cast<__bf16*>(dy_out), db, pieces, c);
  else
    hipLaunchKernelGGL(relu_bias_backward_kernel<false>, dim3(blocks), dim3(kMaskBlock), 0, st, dy,
                       static_cast<const __bf16*>(y), relu, static_cast<__bf16*>(dy_out), db, pieces, c);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ufail(-100 - (int)e, std::string("ReLU / bias backward: ") + hipGetErrorString(e));
  return 0;
}

int ggh_conv3x3_weights_bf16(const float* w, void* w_bf16, void* wt_bf16, float* dw_zero, float* db_zero,
                             int32_t cout, int32_t cin, void* stream) {
  if (!w || !w_bf16 || !wt_bf16) return ufail(-1, "null pointer");
  if (cout < 1 || cin < 1 || (long long)cout * 9 * cin >= (1ll << 31)) return ufail(-2, "unsupported shape");
  const long long n = (long long)cout * 9 * cin;
  const unsigned blocks = (unsigned)((n + kPrepBlock - 1) / kPrepBlock < 4096 ? (n + kPrepBlock - 1) / kPrepBlock : 4096);
  hipLaunchKernelGGL(weights_bf16_kernel, dim3(blocks), dim3(kPrepBlock), 0, static_cast<hipStream_t>(stream), w,
                     static_cast<__bf16*>(w_bf16), static_cast<__bf16*>(wt_bf16), dw_zero, db_zero, cout, cin);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ufail(-100 - (int)e, std::string("BF16 weights: ") + hipGetErrorString(e));
  return 0;
}

int ggh_conv3x3_weight_grad(const void* x, const void* dy, float* dw, int32_t n, int32_t h, int32_t wd, int32_t cin,
                            int32_t cout, int32_t splits, void* stream) {
  if (!x || !dy || !dw) return ufail(-1, "null pointer");
  if (!shapes_ok(n, h, wd, cin, cout) || cout > kWgMaxM) return ufail(-2, "unsupported shape (Cout <= 128)");
  const __bf16 *xb = static_cast<const __bf16*>(x), *db = static_cast<const __bf16*>(dy);
  const WgradArgs args = {xb, db, dw, n, h, wd, cin, cout, nullptr, nullptr, nullptr, static_cast<hipStream_t>(stream)};
  // few tiles and few output channels: the tile kernel's additions to dw take
  // longer than the general kernel's repeated loads (64 x 64, 64 -> 16, batch 1
  // and 4: 10.8 and 14.5 us against 6.5 and 10.3; 128 x 128, 96 -> 32: 15.5 against
  // 13.9; from 64 channels on the tile kernel is the faster one at any size)
  const bool few = cout < 64 && wgrad_tiles(args) <= 128;
  if (!few && wgrad_tile(args)) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return ufail(-100 - (int)e, std::string("conv weight gradient: ") + hipGetErrorString(e));
    return 0;
  }
  const int P = n * h * wd;
  if (splits < 1) splits = 1;
  int per = (P + splits - 1) / splits;
  per = (per + kWgPix - 1) / kWgPix * kWgPix;
  splits = (P + per - 1) / per;
  const int cols = (9 * cin + kWgN - 1) / kWgN;
  hipLaunchKernelGGL(conv_wgrad_kernel, dim3(cols, splits), dim3(64 * kWaves), 0, static_cast<hipStream_t>(stream),
                     xb, db, dw, n, h, wd, cin, cout, per);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ufail(-100 - (int)e, std::string("conv weight gradient: ") + hipGetErrorString(e));
  return 0;
}

int ggh_conv3x3_forward_f32w(const void* x, const float* w, const float* bias, void* y, int32_t n, int32_t h,
                             int32_t wd, int32_t cin, int32_t cout, int32_t relu, void* stream) {
  if (!x || !w || !y) return ufail(-1, "null pointer");
  if (!shapes_ok(n, h, wd, cin, cout)) return ufail(-2, "unsupported shape (W % 16, N H W % 32, Cin % 8, Cout % 16)");
  if (reinterpret_cast<uintptr_t>(w) % 16) return ufail(-2, "weights not 16-byte aligned");
  const ConvArgs args = {static_cast<const __bf16*>(x), w, bias, static_cast<__bf16*>(y), n, h, wd, cin, cout, relu,
                         nullptr, static_cast<hipStream_t>(stream)};
  if (!launch_tile<true, false>(args)) return ufail(-2, "unsupported channel count or output alignment");
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ufail(-100 - (int)e, std::string("conv forward: ") + hipGetErrorString(e));
  return 0;
}

int ggh_unet_pad(const float* x, void* z, int64_t pixels, int32_t k, void* stream) {
  if (!x || !z) return ufail(-1, "null pointer");
  if (pixels <= 0 || k < 1 || k > 8) return ufail(-2, "unsupported shape");
  hipLaunchKernelGGL(pad8_kernel, dim3(glue_grid(pixels)), dim3(kGlueBlock), 0, static_cast<hipStream_t>(stream), x,
                     static_cast<__bf16*>(z), (long long)pixels, k);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ufail(-100 - (int)e, std::string("input padding: ") + hipGetErrorString(e));
  return 0;
}

int ggh_unet_head(const void* z, const float* head, const float* bias, float* out, int64_t pixels, void* stream) {
  if (!z || !head || !bias || !out) return ufail(-1, "null pointer");
  if (pixels <= 0) return ufail(-2, "unsupported shape");
  hipLaunchKernelGGL(head_kernel, dim3(glue_grid(pixels)), dim3(kGlueBlock), 0, static_cast<hipStream_t>(stream),
                     static_cast<const __bf16*>(z), head, bias, out, (long long)pixels);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ufail(-100 - (int)e, std::string("head: ") + hipGetErrorString(e));
  return 0;
}

int ggh_unet_head_backward(const float* dout, const void* z, const float* head, void* dz, float* dhead, float* dbias,
                           int64_t pixels, void* stream) {
  if (!dout || !z || !head || !dz || !dhead || !dbias) return ufail(-1, "null pointer");
  if (pixels <= 0) return ufail(-2, "unsupported shape");
  // two blocks a compute unit: every block ends with an addition per channel to the same addresses
  const unsigned grid = std::min(glue_grid(pixels), 512u);
  hipLaunchKernelGGL(head_backward_kernel, dim3(grid), dim3(kGlueBlock), 0, static_cast<hipStream_t>(stream), dout,
                     static_cast<const __bf16*>(z), head, static_cast<__bf16*>(dz), dhead, dbias, (long long)pixels);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ufail(-100 - (int)e, std::string("head backward: ") + hipGetErrorString(e));
  return 0;
}

size_t ggh_conv3x3_backward_work(int32_t n, int32_t h, int32_t wd, int32_t cin, int32_t cout) {
  size_t floats = 0;
  const bool bias = cout == 16 || cout == 32 || cout == 64 || cout == 128;  // as ggh_relu_bias_backward, here from 16
  if (!bias || !shapes_ok(n, h, wd, cin, cout)) return 0;
  return wgrad_tile({nullptr, nullptr, nullptr, n, h, wd, cin, cout, nullptr, nullptr, nullptr, nullptr}, &floats)
             ? floats * sizeof(float)
             : 0;
}

int ggh_conv3x3_backward(const void* x, const void* y, const void* dy, const void* wt, void* dx, float* dw, float* db,
                         float* work, size_t work_bytes, int32_t n, int32_t h, int32_t wd, int32_t cin, int32_t cout,
                         void* stream) {
  if (!x || !dy || !dw || !db || !work || (dx && !wt)) return ufail(-1, "null pointer");
  const size_t need = ggh_conv3x3_backward_work(n, h, wd, cin, cout);
  if (need == 0 || (dx && cin % 16)) return ufail(-2, "unsupported shape: the layer's gradients one by one");
  if (work_bytes < need || reinterpret_cast<uintptr_t>(work) % 16 || reinterpret_cast<uintptr_t>(dx) % 8)
    return ufail(-2, "work space too small or a pointer not aligned");
  const hipStream_t st = static_cast<hipStream_t>(stream);
  const __bf16 *dyb = static_cast<const __bf16*>(dy), *yb = static_cast<const __bf16*>(y);
  if (dx) {
    // the data gradient: the convolution of the masked gradient with the flipped weights
    const ConvArgs args = {dyb, wt, nullptr, static_cast<__bf16*>(dx), n, h, wd, cout, cin, 0, yb, st};
    if (yb) launch_tile<false, true>(args);
    else launch_tile<false, false>(args);
  }
  wgrad_tile({static_cast<const __bf16*>(x), dyb, dw, n, h, wd, cin, cout, yb, db, work, st});
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ufail(-100 - (int)e, std::string("conv backward: ") + hipGetErrorString(e));
  return 0;
}

int ggh_pool2x2_forward(const void* x, void* y, uint8_t* arg, int32_t n, int32_t h, int32_t wd, int32_t c,
                        void* stream) {
  if (!x || !y || !arg) return ufail(-1, "null pointer");
  if (n <= 0 || h <= 0 || wd <= 0 || h % 2 || wd % 2 || c <= 0 || c % 8) return ufail(-2, "unsupported shape");
  const long long pieces = (long long)n * (h / 2) * (wd / 2) * (c / 8);
  hipLaunchKernelGGL(pool2x2_kernel, dim3(glue_grid(pieces)), dim3(kGlueBlock), 0, static_cast<hipStream_t>(stream),
                     static_cast<const __bf16*>(x), static_cast<__bf16*>(y), arg, n, h, wd, c);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ufail(-100 - (int)e, std::string("pooling: ") + hipGetErrorString(e));
  return 0;
}

int ggh_pool2x2_backward(const void* dy, const uint8_t* arg, void* dx, int32_t n, int32_t h, int32_t wd, int32_t c,
                         void* stream) {
  if (!dy || !arg || !dx) return ufail(-1, "null pointer");
  if (n <= 0 || h <= 0 || wd <= 0 || h % 2 || wd % 2 || c <= 0 || c % 8) return ufail(-2, "unsupported shape");
  const long long pieces = (long long)n * (h / 2) * (wd / 2) * (c / 8);
  hipLaunchKernelGGL(pool2x2_backward_kernel, dim3(glue_grid(pieces)), dim3(kGlueBlock), 0,
                     static_cast<hipStream_t>(stream), static_cast<const __bf16*>(dy), arg, static_cast<__bf16*>(dx), n,
                     h, wd, c);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ufail(-100 - (int)e, std::string("pooling backward: ") + hipGetErrorString(e));
  return 0;
}

int ggh_upcat_forward(const void* z, const void* s, void* out, int32_t n, int32_t h, int32_t wd, int32_t cz,
                      int32_t cs, void* stream) {
  if (!z || !s || !out) return ufail(-1, "null pointer");
  if (n <= 0 || h <= 0 || wd <= 0 || h % 2 || wd % 2 || cz <= 0 || cz % 8 || cs <= 0 || cs % 8)
    return ufail(-2, "unsupported shape");
  const long long pieces = (long long)n * h * wd * ((cz + cs) / 8);
  hipLaunchKernelGGL(upcat_kernel, dim3(glue_grid(pieces)), dim3(kGlueBlock), 0, static_cast<hipStream_t>(stream),
                     static_cast<const __bf16*>(z), static_cast<const __bf16*>(s), static_cast<__bf16*>(out), n, h, wd,
                     cz, cs);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ufail(-100 - (int)e, std::string("upsampling: ") + hipGetErrorString(e));
  return 0;
}

int ggh_upcat_backward(const void* dout, void* dz, void* ds, int32_t n, int32_t h, int32_t wd, int32_t cz, int32_t cs,
                       void* stream) {
  if (!dout || !dz || !ds) return ufail(-1, "null pointer");
  if (n <= 0 || h <= 0 || wd <= 0 || h % 2 || wd % 2 || cz <= 0 || cz % 8 || cs <= 0 || cs % 8)
    return ufail(-2, "unsupported shape");
  const long long pieces = (long long)n * (h / 2) * (wd / 2) * (cz / 8) + (long long)n * h * wd * (cs / 8);
  hipLaunchKernelGGL(upcat_backward_kernel, dim3(glue_grid(pieces)), dim3(kGlueBlock), 0,
                     static_cast<hipStream_t>(stream), static_cast<const __bf16*>(dout), static_cast<__bf16*>(dz),
                     static_cast<__bf16*>(ds), n, h, wd, cz, cs);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ufail(-100 - (int)e, std::string("upsampling backward: ") + hipGetErrorString(e));
  return 0;
}

}  // extern "C"
