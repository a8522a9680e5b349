// pm_net.hip -- gfx950 kernels of the plane-proposal network: a 3x3
// convolution on bf16 NHWC activations as an implicit GEMM on the matrix
// cores (v_mfma_f32_16x16x32_bf16, fp32 accumulation), its weight gradient
// (v_mfma_f32_16x16x4_f32), and the pooling, gradient routing, loss, Adam and
// input packing kernels of a U-Net training step.
#include <algorithm>
#include <cstdint>

#include "pm_net_kernels.h"

namespace pm {
namespace net {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef __attribute__((__vector_size__(16))) uint32_t u32x4;

#define NET_LAUNCH(kernel, grid, block, lds, st, ...)               \
  do {                                                              \
    (void)hipGetLastError();                                        \
    hipLaunchKernelGGL(kernel, grid, block, lds, st, __VA_ARGS__);  \
    return hipGetLastError();                                       \
  } while (0)

__device__ __forceinline__ bf16x8 load8(const bf16* p) {
  return *reinterpret_cast<const bf16x8*>(p);
}

__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = (bf16)0.0f;
  return z;
}

// Every convolution multiplies weights (rows: output channels) by pixels
// (columns): lane l ends with channels 4 (l / 16) .. + 3 of pixel l % 16, so
// it writes 8 bytes (16 in fp32) where the other order writes 2.  vec: the
// output rows are aligned for that (an output given by a caller may not be).
__device__ __forceinline__ f32x4 conv_bias4(const ConvArgs& a, int co) {
  f32x4 b = {0.f, 0.f, 0.f, 0.f};
  if (a.bias) {
#pragma unroll
    for (int j = 0; j < 4; ++j) b[j] = a.bias[std::min(co + j, a.cout - 1)];
  }
  return b;
}

__device__ __forceinline__ void conv_store4(const ConvArgs& a, size_t p,
                                            int co, const f32x4& acc,
                                            const f32x4& bias, bool vec) {
  if (co >= a.cout) return;
  float v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v[j] = acc[j] + bias[j];
    if (a.relu) v[j] = fmaxf(v[j], 0.0f);
  }
  float* yf = a.yf + p * a.ys + co;
  if (a.yf2 && co >= a.split)
    yf = a.yf2 + p * (a.cout - a.split) + (co - a.split);
  if (vec) {
    if (a.mask) {
      const bf16x4 m =
          *reinterpret_cast<const bf16x4*>(a.mask + p * a.ys + co);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = (float)m[j] > 0.0f ? v[j] : 0.0f;
    }
    if (a.yf) {
      *reinterpret_cast<float4*>(yf) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
      bf16x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = (bf16)v[j];
      *reinterpret_cast<bf16x4*>(a.y + p * a.ys + co) = o;
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (co + j >= a.cout) continue;
    if (a.mask && !((float)a.mask[p * a.ys + co + j] > 0.0f)) v[j] = 0.0f;
    if (a.yf)
      yf[j] = v[j];
    else
      a.y[p * a.ys + co + j] = (bf16)v[j];
  }
}

static bool conv_vec_store(const ConvArgs& a) {
  const uintptr_t ptr = a.yf ? reinterpret_cast<uintptr_t>(a.yf) |
                                   reinterpret_cast<uintptr_t>(a.yf2)
                             : 2 * (reinterpret_cast<uintptr_t>(a.y) |
                                    reinterpret_cast<uintptr_t>(a.mask));
  return a.ys % 4 == 0 && a.cout % 4 == 0 && ptr % 16 == 0;
}

// ---------------------------------------------------------------------
// lattice convolution: any dilation, any channels.  The pixels a dilated
// kernel couples are a lattice (every dil-th column and row), so a
// work-group takes a tile of 16 x kMT lattice pixels with its one-pixel rim,
// stages all their input channels in LDS once and shares them among its
// wavefronts, each of 16 kNT output channels.  Per K step of 32 a lane reads
// its pixel's 8 consecutive k (one tap, 8 channels) from there and its
// weight row's from memory (L2), kDepth steps ahead: with one step at a
// time the layers here are a chain of trips to L2.  An LDS pixel takes an
// odd number of 16-byte pieces, so 16 neighbours hit distinct banks.
// K is summed tap by tap, channels within a tap.
// Against a gather of every operand from memory, one wavefront with 64
// pixels x 64 channels: 128 -> 128 channels at 160 x 90, dilation 2 / 4 / 8,
// 54 / 53 / 52 -> 18 / 18 / 20 us, at 40 x 30 50 -> 11; 112 -> 96 at 320 x 180
// 61 -> 28; 8 -> 32 at 1280 x 720, whose bound is the 59 MB it writes, 46 -> 24.
// The dilated layers at 160 x 90 are 960 wavefronts, fewer than the SIMDs.
// ---------------------------------------------------------------------
constexpr int kLatX = 16;

static int lattice_pieces(int cin) { return cin / 8 | 1; }

template <int kMT>
static size_t lattice_lds(int cin) {
  return ((kLatX + 2) * (kMT + 2) * lattice_pieces(cin) + 1) * sizeof(uint4);
}

template <int kMT, int kNT, int kDepth>
__global__ void __launch_bounds__(512)
k_conv_lattice(ConvArgs a, int tiles_x, int tiles_y, bool vec) {
  constexpr int kRimX = kLatX + 2, kRimY = kMT + 2;
  extern __shared__ uint4 smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = lane & 15, grp = lane >> 4;
  const int cin = a.c1 + a.c2, P = cin / 8, stride = P | 1;
  const int kpad = conv_kpad(cin), steps = kpad / 32;
  const int H2 = a.up2 ? (a.H + 1) >> 1 : a.H;
  const int W2 = a.up2 ? (a.W + 1) >> 1 : a.W;
  // tile, then the lattice's offset, then the image
  int t = blockIdx.x;
  const int lx0 = t % tiles_x * kLatX;
  t /= tiles_x;
  const int ly0 = t % tiles_y * kMT;
  t /= tiles_y;
  const int ox = t % a.dil;
  t /= a.dil;
  const int oy = t % a.dil, n = t / a.dil;
  const int co0 = (blockIdx.y * (blockDim.x >> 6) + wave) * (16 * kNT);
  const bool busy = co0 < conv_cpad(a.cout);

  // this lane's weights, kDepth steps ahead
  const bf16* wrow = a.w + (size_t)(busy ? co0 + row : 0) * kpad + 8 * grp;
  u32x4 bw[kDepth][kNT];
  int next = 0;
  auto load = [&](u32x4 (&v)[kNT]) {
    const int k = 32 * std::min(next, steps - 1);
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
      v[nt] = *reinterpret_cast<const u32x4*>(wrow + nt * 16 * kpad + k);
    ++next;
  };
#pragma unroll
  for (int d = 0; d < kDepth; ++d) load(bw[d]);

  for (int q = tid; q < kRimX * kRimY * P; q += blockDim.x) {
    const int pix = q / P, g = q - pix * P;
    const int r = pix / kRimX, c = pix - r * kRimX;
    const int yy = (ly0 + r - 1) * a.dil + oy;
    const int xx = (lx0 + c - 1) * a.dil + ox;
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if (yy >= 0 && yy < a.H && xx >= 0 && xx < a.W) {
      if (8 * g < a.c1) {
        v = *reinterpret_cast<const uint4*>(
            a.x1 + (((size_t)n * a.H + yy) * a.W + xx) * a.c1 + 8 * g);
      } else {
        const int y2 = a.up2 ? yy >> 1 : yy, x2 = a.up2 ? xx >> 1 : xx;
        v = *reinterpret_cast<const uint4*>(
            a.x2 + (((size_t)n * H2 + y2) * W2 + x2) * a.c2 +
            (8 * g - a.c1));
      }
    }
    smem[pix * stride + g] = v;
  }
  constexpr int kRim = kRimX * kRimY;
  if (tid == 0) smem[kRim * stride] = make_uint4(0u, 0u, 0u, 0u);
  __syncthreads();
  if (!busy) return;

  f32x4 acc[kMT][kNT];
#pragma unroll
  for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // this lane's k as (tap, piece); from tap 9 on there are no real k, and
  // the piece of zeros behind the window is read
  int tap = grp / P, g = grp - tap * P;
  const int step_tap = 4 / P, step_g = 4 - step_tap * P;
  auto multiply = [&](const u32x4 (&w)[kNT]) {
    const int ty = (tap * 11) >> 5;  // tap / 3 for the taps there are
    const int at = (ty * kRimX + tap - 3 * ty + row) * stride + g;
    const bool real = tap < 9;
#pragma unroll
    for (int mt = 0; mt < kMT; ++mt) {
      const uint4 v =
          smem[real ? at + mt * kRimX * stride : kRim * stride];
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8, w[nt]), __builtin_bit_cast(bf16x8, v),
            acc[mt][nt], 0, 0, 0);
    }
    g += step_g;
    tap += step_tap + (g >= P ? 1 : 0);
    g -= g >= P ? P : 0;
  };
  int s = 0;
  for (; s + kDepth <= steps; s += kDepth) {
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
      multiply(bw[d]);
      load(bw[d]);
      __builtin_amdgcn_sched_barrier(0);  // or all loads come last
    }
  }
#pragma unroll
  for (int d = 0; d < kDepth - 1; ++d)
    if (s + d < steps) multiply(bw[d]);

  f32x4 bias[kNT];
#pragma unroll
  for (int nt = 0; nt < kNT; ++nt)
    bias[nt] = conv_bias4(a, co0 + nt * 16 + 4 * grp);
  const int x = (lx0 + row) * a.dil + ox;
  if (x >= a.W) return;
#pragma unroll
  for (int mt = 0; mt < kMT; ++mt) {
    const int y = (ly0 + mt) * a.dil + oy;
    if (y >= a.H) continue;
    const size_t p = ((size_t)n * a.H + y) * a.W + x;
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
      conv_store4(a, p, co0 + nt * 16 + 4 * grp, acc[mt][nt], bias[nt], vec);
  }
}

template <int kMT, int kNT, int kDepth, int kWaves>
static hipError_t launch_lattice(hipStream_t st, const ConvArgs& a,
                                 bool vec) {
  const int lw = (a.W + a.dil - 1) / a.dil, lh = (a.H + a.dil - 1) / a.dil;
  const int tiles_x = (lw + kLatX - 1) / kLatX, tiles_y = (lh + kMT - 1) / kMT;
  const int groups = conv_cpad(a.cout) / (16 * kNT);
  const int waves = std::min(groups, kWaves);
  const size_t lds = lattice_lds<kMT>(a.c1 + a.c2);
  if (lds > 65536) return hipErrorInvalidValue;
  NET_LAUNCH((k_conv_lattice<kMT, kNT, kDepth>),
             dim3((unsigned)((long)tiles_x * tiles_y * a.dil * a.dil * a.N),
                  (unsigned)((groups + waves - 1) / waves)),
             dim3(64 * waves), lds, st, a, tiles_x, tiles_y, vec);
}

// ---------------------------------------------------------------------
// LDS-tiled convolution (dilation 1, c1 and c2 multiples of 32): a
// work-group of four wavefronts computes a 64 x 4 pixel tile of one image
// (wavefront w: tile row w) x 16 kNT output channels.  The input channels
// are taken 32 at a time: the chunk's (4 + 2) x (64 + 2) pixel window and
// its weights for the 9 taps are staged in LDS, and every tap is one K
// step of 32 read from there, so each input pixel is fetched from memory
// 1.5 times per chunk instead of 9.  The next chunk's global loads are in
// flight during the current chunk's matrix-core work.  LDS rows of 64
// bytes (32 channels) are read 16 bytes per lane by 16 consecutive
// pixels; the 16-byte slot of channel group g of window column x is
// g ^ ((x >> 1) & 3), so any 8 consecutive columns hit distinct banks.
// K is summed chunk by chunk, tap by tap within a chunk.
// ---------------------------------------------------------------------
constexpr int kTileX = 64, kTileY = 4;
constexpr int kWinX = kTileX + 2, kWinY = kTileY + 2;
constexpr int kWinPieces = kWinY * kWinX * 4;   // 16-byte pieces

__device__ __forceinline__ int lds_slot(int g, int col) {
  return g ^ ((col >> 1) & 3);
}

// kWalk: one chunk (32 input channels), the full-resolution layers, which
// are bound by memory and latency: a work-group walks tiles (a run of them,
// top to bottom, so that the two shared rows are in its L2), stages its
// weights once and reads the next tile's window during this one's products.
// With one tile per work-group nothing overlapped its fetch: 32 -> 32
// channels at 1280 x 720 (59 MB in, 59 out) 62 -> 32 us, the head 46 -> 24.
// With more chunks the weights of all have to stay in LDS, and walking was
// the slower form (96 -> 32: 88 us without, 99 with).
template <int kNT, bool kWalk>
__device__ __forceinline__ void conv_lds_block(const ConvArgs& a, int tiles_x,
                                               int tiles_y, int tiles,
                                               bool vec) {
  constexpr int kCO = 16 * kNT;
  constexpr int kWPieces = 9 * kCO * 4;
  constexpr int kAIters = (kWinPieces + 255) / 256;
  constexpr int kBIters = (kWPieces + 255) / 256;
  __shared__ uint4 sA[kWinPieces];
  __shared__ uint4 sB[kWPieces];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = lane & 15, grp = lane >> 4;
  const int co0 = blockIdx.y * kCO;
  const int cin = a.c1 + a.c2;
  const int kpad = conv_kpad(cin);
  const int H2 = a.up2 ? (a.H + 1) >> 1 : a.H;
  const int W2 = a.up2 ? (a.W + 1) >> 1 : a.W;
  const int nchunks = kWalk ? 1 : cin / 32;
  int t = blockIdx.x, t_end = t + 1;
  if (kWalk) {
    t = (int)((long)blockIdx.x * tiles / gridDim.x);
    t_end = (int)((long)(blockIdx.x + 1) * tiles / gridDim.x);
  }
  int n, x0, y0;
  auto place = [&](int tile) {
    if (kWalk) {  // top to bottom first
      y0 = (tile % tiles_y) * kTileY;
      tile /= tiles_y;
      x0 = (tile % tiles_x) * kTileX;
      n = tile / tiles_x;
    } else {
      x0 = (tile % tiles_x) * kTileX;
      tile /= tiles_x;
      y0 = (tile % tiles_y) * kTileY;
      n = tile / tiles_y;
    }
  };

  uint4 ra[kAIters], rb[kBIters];
  // global loads of channels 32 c .. 32 c + 31 of the window and the weights
  auto fetch_a = [&](int c) {
    const int cc = 32 * c;
#pragma unroll
    for (int i = 0; i < kAIters; ++i) {
      const int q = tid + 256 * i;
      uint4 v = make_uint4(0u, 0u, 0u, 0u);
      if (q < kWinPieces) {
        const int r = q / (kWinX * 4), rem = q - r * (kWinX * 4);
        const int xt = rem >> 2, g = rem & 3;
        const int yy = y0 - 1 + r, xx = x0 - 1 + xt;
        if (yy >= 0 && yy < a.H && xx >= 0 && xx < a.W) {
          if (cc < a.c1) {
            v = *reinterpret_cast<const uint4*>(
                a.x1 + (((size_t)n * a.H + yy) * a.W + xx) * a.c1 + cc +
                8 * g);
          } else {
            const int y2 = a.up2 ? yy >> 1 : yy, x2 = a.up2 ? xx >> 1 : xx;
            v = *reinterpret_cast<const uint4*>(
                a.x2 + (((size_t)n * H2 + y2) * W2 + x2) * a.c2 +
                (cc - a.c1) + 8 * g);
          }
        }
      }
      ra[i] = v;
    }
  };
  auto fetch_b = [&](int c) {
#pragma unroll
    for (int i = 0; i < kBIters; ++i) {
      const int q = tid + 256 * i;
      uint4 v = make_uint4(0u, 0u, 0u, 0u);
      if (q < kWPieces) {
        const int tap = q / (kCO * 4), rem = q - tap * (kCO * 4);
        const int co = rem >> 2, g = rem & 3;
        v = *reinterpret_cast<const uint4*>(
            a.w + (size_t)(co0 + co) * kpad + tap * cin + 32 * c + 8 * g);
      }
      rb[i] = v;
    }
  };
  auto stage_a = [&]() {
#pragma unroll
    for (int i = 0; i < kAIters; ++i) {
      const int q = tid + 256 * i;
      if (q < kWinPieces) {
        const int r = q / (kWinX * 4), rem = q - r * (kWinX * 4);
        const int xt = rem >> 2, g = rem & 3;
        sA[(r * kWinX + xt) * 4 + lds_slot(g, xt)] = ra[i];
      }
    }
  };
  auto stage_b = [&]() {
#pragma unroll
    for (int i = 0; i < kBIters; ++i) {
      const int q = tid + 256 * i;
      if (q < kWPieces) {
        const int tap = q / (kCO * 4), rem = q - tap * (kCO * 4);
        const int co = rem >> 2, g = rem & 3;
        sB[(tap * kCO + co) * 4 + lds_slot(g, co)] = rb[i];
      }
    }
  };

  f32x4 acc[4][kNT];
  auto clear = [&]() {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt)
        acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto multiply = [&]() {
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
      const int dy = tap / 3, dx = tap % 3;  // window offsets 0..2
      bf16x8 A[4], B[kNT];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        const int xt = mt * 16 + row + dx;
        A[mt] = __builtin_bit_cast(
            bf16x8, sA[((wave + dy) * kWinX + xt) * 4 + lds_slot(grp, xt)]);
      }
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt) {
        const int co = nt * 16 + row;
        B[nt] = __builtin_bit_cast(
            bf16x8, sB[(tap * kCO + co) * 4 + lds_slot(grp, co)]);
      }
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              B[nt], A[mt], acc[mt][nt], 0, 0, 0);
    }
  };
  f32x4 bias[kNT];
  auto load_bias = [&]() {
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
      bias[nt] = conv_bias4(a, co0 + nt * 16 + 4 * grp);
  };
  auto store = [&](int sn, int sx, int sy) {
    const int y = sy + wave;
    if (y >= a.H) return;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int x = sx + mt * 16 + row;
      if (x >= a.W) continue;
      const size_t p = ((size_t)sn * a.H + y) * a.W + x;
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt)
        conv_store4(a, p, co0 + nt * 16 + 4 * grp, acc[mt][nt], bias[nt],
                    vec);
    }
  };

  place(t);
  fetch_a(0);
  fetch_b(0);
  if (kWalk) {
    load_bias();
    stage_b();
    for (; t < t_end; ++t) {
      __syncthreads();  // every wavefront is done reading the last window
      stage_a();
      __syncthreads();
      const int sn = n, sx = x0, sy = y0;
      if (t + 1 < t_end) {
        place(t + 1);
        fetch_a(0);
      }
      clear();
      multiply();
      store(sn, sx, sy);
    }
  } else {
    clear();
    for (int c = 0; c < nchunks; ++c) {
      __syncthreads();  // every wavefront is done reading the previous chunk
      stage_a();
      stage_b();
      __syncthreads();
      if (c + 1 < nchunks) {
        fetch_a(c + 1);
        fetch_b(c + 1);
      }
      multiply();
    }
    load_bias();
    store(n, x0, y0);
  }
}

// three wavefronts per SIMD
template <int kNT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
k_conv_lds_walk(ConvArgs a, int tiles_x, int tiles_y, int tiles, bool vec) {
  conv_lds_block<kNT, true>(a, tiles_x, tiles_y, tiles, vec);
}

// Two work-groups per CU, which the 64-channel form needs said: at 264
// registers it ran one (64 -> 64 at 640 x 360: 49 us, 37 at 250 registers).
template <int kNT>
__global__ void __launch_bounds__(256, 2)
k_conv_lds(ConvArgs a, int tiles_x, int tiles_y, int tiles, bool vec) {
  conv_lds_block<kNT, false>(a, tiles_x, tiles_y, tiles, vec);
}

template <int kNT>
static hipError_t launch_lds(hipStream_t st, const ConvArgs& a, bool vec) {
  const int tiles_x = (a.W + kTileX - 1) / kTileX;
  const int tiles_y = (a.H + kTileY - 1) / kTileY;
  const int tiles = (int)((long)tiles_x * tiles_y * a.N);
  NET_LAUNCH(k_conv_lds<kNT>,
             dim3((unsigned)tiles, (unsigned)(conv_cpad(a.cout) / (16 * kNT))),
             dim3(256), 0, st, a, tiles_x, tiles_y, tiles, vec);
}

template <int kNT>
static hipError_t launch_walk(hipStream_t st, const ConvArgs& a, bool vec) {
  const int tiles_x = (a.W + kTileX - 1) / kTileX;
  const int tiles_y = (a.H + kTileY - 1) / kTileY;
  const int tiles = (int)((long)tiles_x * tiles_y * a.N);
  // work-groups that run at once (3 per CU), each a run of tiles
  NET_LAUNCH(k_conv_lds_walk<kNT>,
             dim3((unsigned)std::min(tiles, 768),
                  (unsigned)((a.cout + 16 * kNT - 1) / (16 * kNT))),
             dim3(256), 0, st, a, tiles_x, tiles_y, tiles, vec);
}

// All forms sum K in the order that their layers always had, so a layer
// gives the same bits whichever runs.
hipError_t launch_conv(hipStream_t st, const ConvArgs& a) {
  const int cpad = conv_cpad(a.cout), cin = a.c1 + a.c2;
  const bool vec = conv_vec_store(a);
  if (a.dil == 1 && a.c1 % 32 == 0 && a.c2 % 32 == 0 && cin > 0) {
    if (cin == 32)
      return a.cout <= 16 ? launch_walk<1>(st, a, vec)
                          : launch_walk<2>(st, a, vec);
    return cpad % 64 == 0 ? launch_lds<4>(st, a, vec)
                          : launch_lds<2>(st, a, vec);
  }
  // Tiles of 16 x 8 share the weights' loads among twice the pixels, but need
  // enough wavefronts to hide them: 128 -> 128, dilation 2, at 160 x 90 (960
  // wavefronts) takes 18 us with 16 x 8 and 17 with 16 x 4, dilation 4 and 8 18
  // and 20 against 21; at 40 x 30 (128 wavefronts) 14-16 against 11.
  const long waves = (long)((a.W + kLatX * a.dil - 1) / (kLatX * a.dil)) *
                     ((a.H + 8 * a.dil - 1) / (8 * a.dil)) * a.dil * a.dil *
                     a.N * (cpad / 16);
  return waves >= 512 ? launch_lattice<8, 1, 4, 8>(st, a, vec)
                      : launch_lattice<4, 1, 8, 4>(st, a, vec);
}

// ---------------------------------------------------------------------
// weight gradient on the matrix cores: dw[co][tap, ci] = sum over pixels p
// of g[p][co] x[p + tap][ci], a GEMM whose contraction runs over the
// pixels.
//
// The order of the sum is part of the kernel.  Adam's first steps take the
// sign of a gradient, so where one is about zero another rounding of it
// moves the weight the other way and the next step sees another network:
// with the bf16 instruction, which adds up 32 products at a time, and
// gradients as near to 64-bit sums as before (3.4e-7 to 6.1e-7), the second
// step's were 2e-4 away from those of the kernel before it.  So a sum is
// what it was with one fmaf per pixel: kWgChunk pixels in order, in fp32.
// v_mfma_f32_16x16x4_f32 gives exactly that chain (checked on the card:
// no element of 64 products differs, denormals included), a product of two
// bf16 is exact, and a pixel beyond the image or the chunk adds a zero.
// The chunks' sums are added up in their order, in fp32, which also makes a
// step repeatable bit for bit.  That kernel added them up with atomics as
// they came, nearly in order: over 40 seeds its second and third step's
// gradients differ from themselves by a median of 2.0e-7 and by more than
// 2e-5 for 2 and 5 seeds (a weight went the other way), and from these by
// 2.0e-7 and for 2 and 5.  Added up in 64 bits they differ by 7.1e-7, and for
// 3 and 10 seeds.
//
// Layout.  A wavefront owns one chunk, 32 output channels (16 for the
// head) and kTiles tiles of 32 k = (tap, ci).  The activations are NHWC:
// lane 16 kk + i reads the bf16 pair of channels 2 i, 2 i + 1 of the step's
// pixel kk, which as two fp32 are its operands of two matrix tiles, the
// even and the odd channels.  So a step of 4 pixels is kTiles + 1 loads of
// 4 bytes a lane, kWgAhead steps in flight, for 4 kTiles instructions of
// 32 cycles: no LDS, no barrier.  Where the inputs' channels are multiples
// of 32, a tile is one tap of one input and its address is scalar work; a
// step with a tap outside the image selects each lane's address.
// Bound: the SIMDs' fp32 units, which this instruction shares with vector
// instructions (matrix pipe 67 % busy, vector issue 24 %; 157 TFLOP/s
// nominal, 76-97 reached from 96 channels on).  A training step on 8 pairs of
// 512 x 384 (449 GFLOP here): 29.0 ms with one fmaf at a time, 8.6 with this;
// 3.9 with the bf16 instruction.
// ---------------------------------------------------------------------
constexpr int kWgChunk = 1024;
constexpr int kWgAhead = 4;

// what a lane reads for a pixel outside the image
__device__ const uint32_t g_zero_pair = 0u;

// a pair of channels, the memory's address space in the type: a read from
// one of two pointers stays a global one
typedef const __attribute__((address_space(1))) uint32_t* PairPtr;
__device__ __forceinline__ PairPtr pair_at(const void* p) {
  return (PairPtr)(p);
}

__device__ __forceinline__ float bf16_lo(uint32_t v) {
  return __uint_as_float(v << 16);
}
__device__ __forceinline__ float bf16_hi(uint32_t v) {
  return __uint_as_float(v & 0xffff0000u);
}

// The 4 pixels of a step: the first one's index, column, row in the batch
// and row in the image (uniform).
struct WgStep {
  int p, x, yrow, y;
  __device__ __forceinline__ void next(const ConvArgs& a) {
    p += 4;
    x += 4;
    while (x >= a.W) {
      x -= a.W;
      ++yrow;
      if (++y == a.H) y = 0;
    }
  }
  // pixel kk's column, row in the batch and in the image
  __device__ __forceinline__ void lane(const ConvArgs& a, int kk, int* xl,
                                       int* rl, int* yl) const {
    *xl = x + kk;
    *rl = yrow;
    *yl = y;
    while (*xl >= a.W) {
      *xl -= a.W;
      ++*rl;
      if (++*yl == a.H) *yl = 0;
    }
  }
};

// the loads of a tile's steps; k0: the tile's first k
// any channels (even), neither input upsampled
struct WgTileAny {
  const bf16* xp;
  int dy, dx, c;
  bool real;
  __device__ __forceinline__ void init(const ConvArgs& a, int k0, int kk,
                                       int i, int pb) {
    const int cin = a.c1 + a.c2, k = k0 + 2 * i;
    const int tap = k / cin, ci = k - tap * cin;
    const bool second = ci >= a.c1;
    c = second ? a.c2 : a.c1;
    // k beyond the real ones: sums that nothing reads, of the pixel itself
    real = tap < 9;
    dy = real ? (tap / 3 - 1) * a.dil : 0;
    dx = real ? (tap % 3 - 1) * a.dil : 0;
    xp = second ? a.x2 + (ci - a.c1) : a.x1 + ci;
    xp += ((ptrdiff_t)(pb + kk) + (ptrdiff_t)dy * a.W + dx) * c;
  }
  __device__ __forceinline__ PairPtr inner(const ConvArgs&, const WgStep&, int,
                                           int) const {
    return pair_at(xp);
  }
  __device__ __forceinline__ PairPtr outer(const ConvArgs&, int, int, int,
                                           int) const {
    return pair_at(xp);
  }
  __device__ __forceinline__ void next() { xp += 4 * c; }
};

// c1 and c2 multiples of 32: all but the lane's channel pair is uniform
struct WgTile32 {
  const bf16* xp;  // channel 0 of the tile at the step's first pixel's tap,
                   // or, upsampled, at the input's first pixel
  int dy, dx, c;
  bool up;
  static constexpr bool real = true;
  __device__ __forceinline__ void init(const ConvArgs& a, int k0, int, int,
                                       int pb) {
    const int cin = a.c1 + a.c2;
    const int tap = k0 / cin, ci = k0 - tap * cin;
    const bool second = ci >= a.c1;
    c = second ? a.c2 : a.c1;
    dy = (tap / 3 - 1) * a.dil;
    dx = (tap % 3 - 1) * a.dil;
    up = second && a.up2;
    xp = second ? a.x2 + (ci - a.c1) : a.x1 + ci;
    if (!up) xp += ((ptrdiff_t)pb + (ptrdiff_t)dy * a.W + dx) * c;
  }
  // H and W are even where x2 is upsampled, so the batch's rows halve as
  // the image's do
  __device__ __forceinline__ PairPtr inner(const ConvArgs& a, const WgStep& s,
                                           int kk, int i) const {
    if (!up) return pair_at(xp + (unsigned)(kk * c + 2 * i));
    const int col = s.x + dx;
    const bf16* q =
        xp + ((size_t)((s.yrow + dy) >> 1) * (a.W >> 1) + (col >> 1)) * c;
    return pair_at(q + (unsigned)(((kk + (col & 1)) >> 1) * c + 2 * i));
  }
  __device__ __forceinline__ PairPtr outer(const ConvArgs& a, int xl, int rl,
                                           int kk, int i) const {
    if (!up) return pair_at(xp + (unsigned)(kk * c + 2 * i));
    return pair_at(xp +
                   ((ptrdiff_t)((rl + dy) >> 1) * (a.W >> 1) +
                    ((xl + dx) >> 1)) * c + 2 * i);
  }
  __device__ __forceinline__ void next() { xp += up ? 0 : 4 * c; }
};

// part: per chunk its sums, [cpad][kpad], and after those of all chunks
// their bias sums, [cpad] per chunk.  kCT: matrix tiles of output channels.
template <int kCT, int kTiles, typename Tile>
__global__ void __launch_bounds__(256)
k_conv_wgrad(ConvArgs a, const bf16* __restrict__ g, float* __restrict__ part,
             bool with_bias, int groups, int cts, int chunks) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int i = lane & 15, kk = lane >> 4;
  // each XCD takes a run of units, which share their pixels in its L2
  const unsigned per = gridDim.x / 8;
  const unsigned unit =
      (blockIdx.x % 8 * per + blockIdx.x / 8) * 4 + (unsigned)wave;
  if (unit >= (unsigned)groups * cts * chunks) return;
  const int kg = (int)(unit % groups), ct = (int)(unit / groups % cts);
  const int chunk = (int)(unit / groups / cts);
  const int cin = a.c1 + a.c2, kpad = conv_kpad(cin), cpad = conv_cpad(a.cout);
  const int npix = a.N * a.H * a.W;
  const int pb = chunk * kWgChunk;
  const int pe = std::min(npix - pb, kWgChunk) + pb;
  const PairPtr zero = pair_at(&g_zero_pair);

  WgStep s;
  s.p = pb;
  s.yrow = pb / a.W;
  s.x = pb - s.yrow * a.W;
  s.y = s.yrow % a.H;
  // this lane's channels of g; rows beyond cout are sums that nothing reads
  const int co = 32 * ct + (kCT == 2 ? 2 * i : i & ~1);
  const unsigned gl = (unsigned)(kk * a.cout + std::min(co, a.cout - 2));
  const bf16* gp = g + (size_t)pb * a.cout;
  Tile tile[kTiles];
#pragma unroll
  for (int t = 0; t < kTiles; ++t)
    tile[t].init(a, 32 * (kTiles * kg + t), kk, i, pb);

  typedef uint32_t Pairs[kTiles + 1];
  auto issue = [&](Pairs& r) {
    // addresses on both sides of the branch, the loads after it: so each
    // wait counts the loads issued since
    PairPtr q[kTiles + 1];
    if (s.p + 4 <= pe && s.x >= a.dil && s.x + 4 + a.dil <= a.W &&
        s.y >= a.dil && s.y + a.dil < a.H) {
      q[0] = pair_at(gp + gl);
#pragma unroll
      for (int t = 0; t < kTiles; ++t) q[t + 1] = tile[t].inner(a, s, kk, i);
    } else {
      int xl, rl, yl;
      s.lane(a, kk, &xl, &rl, &yl);
      const bool there = s.p + kk < pe;
      q[0] = there ? pair_at(gp + gl) : zero;
#pragma unroll
      for (int t = 0; t < kTiles; ++t) {
        const bool ok = there && tile[t].real &&
                        (unsigned)(yl + tile[t].dy) < (unsigned)a.H &&
                        (unsigned)(xl + tile[t].dx) < (unsigned)a.W;
        q[t + 1] = tile[t].outer(a, xl, rl, kk, i);
        q[t + 1] = ok ? q[t + 1] : zero;
      }
    }
#pragma unroll
    for (int t = 0; t <= kTiles; ++t) r[t] = *q[t];
    gp += 4 * a.cout;
#pragma unroll
    for (int t = 0; t < kTiles; ++t) tile[t].next();
    s.next(a);
  };

  f32x4 acc[kTiles][kCT][2], accb[kCT];
#pragma unroll
  for (int c = 0; c < kCT; ++c) {
    accb[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
      acc[t][c][0] = acc[t][c][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const bool bias = with_bias && kg == 0;
  auto consume = [&](const Pairs& r) {
    float A[kCT];
    if (kCT == 2) {
      A[0] = bf16_lo(r[0]);
      A[kCT - 1] = bf16_hi(r[0]);
    } else {
      A[0] = i & 1 ? bf16_hi(r[0]) : bf16_lo(r[0]);
    }
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      const float B[2] = {bf16_lo(r[t + 1]), bf16_hi(r[t + 1])};
#pragma unroll
      for (int c = 0; c < kCT; ++c)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          acc[t][c][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(
              A[c], B[e], acc[t][c][e], 0, 0, 0);
    }
    if (bias) {
#pragma unroll
      for (int c = 0; c < kCT; ++c)
        accb[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[c], 1.0f, accb[c], 0,
                                                       0, 0);
    }
  };

  Pairs raw[kWgAhead];
#pragma unroll
  for (int d = 0; d < kWgAhead; ++d) issue(raw[d]);
  for (int q = pb; q < pe; q += 4 * kWgAhead) {
#pragma unroll
    for (int d = 0; d < kWgAhead; ++d) {
      consume(raw[d]);
      issue(raw[d]);  // of pixels beyond the chunk: zeros
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // a lane holds rows 4 kk .. 4 kk + 3 of column i of every tile
  float* const out = part + (size_t)chunk * cpad * kpad;
  float* const outb =
      part + (size_t)chunks * cpad * kpad + (size_t)chunk * cpad;
#pragma unroll
  for (int c = 0; c < kCT; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = 32 * ct + (kCT == 2 ? 2 * (4 * kk + j) + c : 4 * kk + j);
#pragma unroll
      for (int t = 0; t < kTiles; ++t) {
        const int k = 32 * (kTiles * kg + t) + 2 * i;
        if (k < kpad)
          *reinterpret_cast<float2*>(out + (size_t)row * kpad + k) =
              make_float2(acc[t][c][0][j], acc[t][c][1][j]);
      }
      if (bias && i == 0) outb[row] = accb[c][j];
    }
}

// The chunks' sums added up in order, 64 elements per work-group: 16
// wavefronts fetch kWgFetch chunks each ahead, the first adds.
constexpr int kWgSums = 16, kWgFetch = 8;

__global__ void __launch_bounds__(64 * kWgSums)
k_wgrad_sum(const float* __restrict__ part, int chunks, int cout, int cpad,
            int kpad, int kreal, int wblocks, float* __restrict__ dw,
            float* __restrict__ db) {
  constexpr int kBatch = kWgSums * kWgFetch;
  __shared__ float sums[kBatch][64];
  const int tx = threadIdx.x, ty = threadIdx.y;
  const bool bias = (int)blockIdx.x >= wblocks;
  const int e = ((int)blockIdx.x - (bias ? wblocks : 0)) * 64 + tx;
  const size_t stride = bias ? (size_t)cpad : (size_t)cpad * kpad;
  const float* src =
      part + (bias ? (size_t)chunks * cpad * kpad : (size_t)0) + e;
  const bool real = bias ? e < cout : e < cout * kpad && e % kpad < kreal;
  float s = 0.0f;
  for (int c0 = 0; c0 < chunks; c0 += kBatch) {
    float v[kWgFetch];
#pragma unroll
    for (int u = 0; u < kWgFetch; ++u) {
      const int c = c0 + ty + kWgSums * u;
      v[u] = real && c < chunks ? src[c * stride] : 0.0f;
    }
    __syncthreads();  // the batch before is added up
#pragma unroll
    for (int u = 0; u < kWgFetch; ++u) sums[ty + kWgSums * u][tx] = v[u];
    __syncthreads();
    if (ty == 0) {
      const int n = std::min(chunks - c0, kBatch);
#pragma unroll 8
      for (int c = 0; c < n; ++c) s += sums[c][tx];
    }
  }
  if (ty == 0 && real) (bias ? db : dw)[e] = s;
}

static int wgrad_chunks(int N, int H, int W) {
  return (int)(((long)N * H * W + kWgChunk - 1) / kWgChunk);
}

size_t wgrad_part_floats(int N, int H, int W, int cin, int cout) {
  return (size_t)wgrad_chunks(N, H, W) * conv_cpad(cout) *
         (conv_kpad(cin) + 1);
}

template <int kCT, int kTiles, typename Tile>
static hipError_t launch_wgrad_chains(hipStream_t st, const ConvArgs& a,
                                      const bf16* g, float* part,
                                      bool with_bias) {
  const int chunks = wgrad_chunks(a.N, a.H, a.W);
  const int tiles = conv_kpad(a.c1 + a.c2) / 32;
  const int groups = (tiles + kTiles - 1) / kTiles;
  const int cts = conv_cpad(a.cout) / 32;
  const long units = (long)groups * cts * chunks;
  NET_LAUNCH((k_conv_wgrad<kCT, kTiles, Tile>),
             dim3((unsigned)((units + 31) / 32 * 8)), dim3(256), 0, st, a, g,
             part, with_bias, groups, cts, chunks);
}

template <int kCT>
static hipError_t launch_wgrad_tiles(hipStream_t st, const ConvArgs& a,
                                     const bf16* g, float* part,
                                     bool with_bias) {
  if (a.c1 % 32 || a.c2 % 32)
    return launch_wgrad_chains<kCT, 3, WgTileAny>(st, a, g, part, with_bias);
  // Three tiles share a step's gradients.  Below 1.5 wavefronts per SIMD that
  // way (the 8 x 48 x 64 layers of a training batch: 864 and 1152), one tile
  // each leaves fewer of them with a second round: dilation 2, 4, 8 161 / 166
  // / 178 -> 120 / 122 / 129 us.  At 2592 it is even (214), at 4608 slower
  // (341 -> 373).
  const long units = (long)wgrad_chunks(a.N, a.H, a.W) *
                     (conv_cpad(a.cout) / 32) *
                     (conv_kpad(a.c1 + a.c2) / 96);
  if (units < 1536)
    return launch_wgrad_chains<kCT, 1, WgTile32>(st, a, g, part, with_bias);
  return launch_wgrad_chains<kCT, 3, WgTile32>(st, a, g, part, with_bias);
}

hipError_t launch_conv_wgrad(hipStream_t st, const ConvArgs& a, const bf16* g,
                             float* part, float* dw, float* db) {
  if (a.c1 % 2 || a.c2 % 2 || a.cout % 2 ||
      (a.up2 && (a.H % 2 || a.W % 2 || a.c1 % 32 || a.c2 % 32)))
    return hipErrorInvalidValue;
  const hipError_t e =
      a.cout <= 16 ? launch_wgrad_tiles<1>(st, a, g, part, db != nullptr)
                   : launch_wgrad_tiles<2>(st, a, g, part, db != nullptr);
  if (e != hipSuccess) return e;
  const int cpad = conv_cpad(a.cout), kpad = conv_kpad(a.c1 + a.c2);
  const int wblocks = (a.cout * kpad + 63) / 64;
  const int bblocks = db ? (a.cout + 63) / 64 : 0;
  NET_LAUNCH(k_wgrad_sum, dim3((unsigned)(wblocks + bblocks)),
             dim3(64, kWgSums), 0, st, part, wgrad_chunks(a.N, a.H, a.W),
             a.cout, cpad, kpad, 9 * (a.c1 + a.c2), wblocks, dw, db);
}

// ---------------------------------------------------------------------
// small kernels
// ---------------------------------------------------------------------
struct FlipTable {
  FlipLayer l[kMaxFlips];
};

// a row of work-groups per layer: 16 launches of 4 us each were 0.1 ms of a
// training step
__global__ void __launch_bounds__(256) k_flip_weights(FlipTable t) {
  const FlipLayer& f = t.l[blockIdx.y];
  const int kpt = conv_kpad(f.cout), rows = conv_cpad(f.cin);
  const int i = (int)blockIdx.x * 256 + (int)threadIdx.x;
  if (i >= rows * kpt) return;
  const int ci = i / kpt, kk = i - ci * kpt;
  bf16 v = (bf16)0.0f;
  if (ci < f.cin && kk < 9 * f.cout) {
    const int tap = kk / f.cout, co = kk - tap * f.cout;
    v = f.w[(size_t)co * conv_kpad(f.cin) + (size_t)(8 - tap) * f.cin + ci];
  }
  f.wt[i] = v;
}

hipError_t launch_flip_weights(hipStream_t st, const FlipLayer* layers,
                               int n) {
  if (n < 1 || n > kMaxFlips) return hipErrorInvalidValue;
  FlipTable t;
  int most = 0;
  for (int l = 0; l < n; ++l) {
    t.l[l] = layers[l];
    most = std::max(most, conv_cpad(layers[l].cin) *
                              conv_kpad(layers[l].cout));
  }
  NET_LAUNCH(k_flip_weights, dim3((unsigned)((most + 255) / 256), (unsigned)n),
             dim3(256), 0, st, t);
}

__device__ __forceinline__ void store_masked4(const float (&v)[4],
                                              const bf16* y, bf16* out) {
  const bf16x4 m = *reinterpret_cast<const bf16x4*>(y);
  bf16x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    o[j] = (bf16)((float)m[j] > 0.0f ? v[j] : 0.0f);
  *reinterpret_cast<bf16x4*>(out) = o;
}

// a thread: 4 consecutive channels of a pixel
__global__ void __launch_bounds__(256)
k_mask_pool(int N, int H, int W, int C, const float* __restrict__ g,
            const float* __restrict__ gp, const bf16* __restrict__ y,
            bf16* __restrict__ out) {
  const unsigned C4 = C / 4;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)N * H * W * C4) return;
  const unsigned c = (unsigned)(i % C4) * 4;
  const size_t q = i / C4;
  const unsigned x = (unsigned)(q % W);
  const size_t r = q / W;
  const unsigned yy = (unsigned)(r % H), n = (unsigned)(r / H);
  const float4 a = *reinterpret_cast<const float4*>(g + q * C + c);
  const float4 b = *reinterpret_cast<const float4*>(
      gp + (((size_t)n * (H / 2) + (yy >> 1)) * (W / 2) + (x >> 1)) * C + c);
  const float v[4] = {a.x + 0.25f * b.x, a.y + 0.25f * b.y,
                      a.z + 0.25f * b.z, a.w + 0.25f * b.w};
  store_masked4(v, y + q * C + c, out + q * C + c);
}

hipError_t launch_mask_pool(hipStream_t st, int N, int H, int W, int C,
                            const float* g, const float* gp, const bf16* y,
                            bf16* out) {
  if (C % 4) return hipErrorInvalidValue;
  const size_t n = (size_t)N * H * W * (C / 4);
  NET_LAUNCH(k_mask_pool, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
             N, H, W, C, g, gp, y, out);
}

__global__ void __launch_bounds__(256)
k_mask_up(int N, int H, int W, int C, const float* __restrict__ g,
          const bf16* __restrict__ y, bf16* __restrict__ out) {
  const unsigned C4 = C / 4;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)N * H * W * C4) return;
  const unsigned c = (unsigned)(i % C4) * 4;
  const size_t q = i / C4;
  const unsigned x = (unsigned)(q % W);
  const size_t r = q / W;  // image * H + row
  const float* p = g + (2 * r * 2 * W + 2 * x) * C + c;
  float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float4 t = *reinterpret_cast<const float4*>(
        p + ((size_t)(k >> 1) * 2 * W + (k & 1)) * C);
    v[0] += t.x;
    v[1] += t.y;
    v[2] += t.z;
    v[3] += t.w;
  }
  store_masked4(v, y + q * C + c, out + q * C + c);
}

hipError_t launch_mask_up(hipStream_t st, int N, int H, int W, int C,
                          const float* g, const bf16* y, bf16* out) {
  if (C % 4) return hipErrorInvalidValue;
  const size_t n = (size_t)N * H * W * (C / 4);
  NET_LAUNCH(k_mask_up, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
             N, H, W, C, g, y, out);
}

__global__ void __launch_bounds__(256)
k_avgpool(int N, int H, int W, int C, const bf16* __restrict__ x,
          bf16* __restrict__ y) {
  // a thread: 8 consecutive channels of one output pixel (C % 8 == 0)
  const int Ho = H / 2, Wo = W / 2, C8 = C / 8;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)N * Ho * Wo * C8) return;
  const int c = (int)(i % C8) * 8;
  const size_t q = i / C8;
  const int xo = (int)(q % Wo);
  const size_t r = q / Wo;
  const int yo = (int)(r % Ho), n = (int)(r / Ho);
  const size_t b = (((size_t)n * H + 2 * yo) * W + 2 * xo) * C + c;
  const bf16x8 v00 = load8(x + b), v01 = load8(x + b + C);
  const bf16x8 v10 = load8(x + b + (size_t)W * C);
  const bf16x8 v11 = load8(x + b + (size_t)W * C + C);
  bf16x8 o;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float s = ((float)v00[k] + (float)v01[k]) +
                    ((float)v10[k] + (float)v11[k]);
    o[k] = (bf16)(0.25f * s);
  }
  *reinterpret_cast<bf16x8*>(y + q * C + c) = o;
}

hipError_t launch_avgpool(hipStream_t st, int N, int H, int W, int C,
                          const bf16* x, bf16* y) {
  if (C % 8) return hipErrorInvalidValue;
  const size_t n = (size_t)N * (H / 2) * (W / 2) * (C / 8);
  NET_LAUNCH(k_avgpool, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
             N, H, W, C, x, y);
}

__global__ void __launch_bounds__(256)
k_l1_loss(size_t npix, const float* __restrict__ o, int os,
          const float4* __restrict__ t, float wd, float wn, float inv_count,
          bf16* __restrict__ g, float* __restrict__ loss) {
  __shared__ float part[256];
  float l = 0.0f;
  for (size_t p = (size_t)blockIdx.x * 256 + threadIdx.x; p < npix;
       p += (size_t)gridDim.x * 256) {
    const float4 tv = t[p];
    const float* op = o + p * os;
    bf16x8 gp = zero8();
    if (tv.x >= 0.0f) {
      const float d[4] = {op[0] - tv.x, op[1] - tv.y, op[2] - tv.z,
                          op[3] - tv.w};
      const float w[4] = {wd, wn, wn, wn};
      for (int c = 0; c < 4; ++c) {
        l += w[c] * fabsf(d[c]);
        gp[c] = (bf16)(d[c] > 0.0f ? w[c] * inv_count
                                   : (d[c] < 0.0f ? -w[c] * inv_count : 0.0f));
      }
    }
    for (int c = 8; c < os; c += 8)
      *reinterpret_cast<bf16x8*>(g + p * os + c) = zero8();
    *reinterpret_cast<bf16x8*>(g + p * os) = gp;
  }
  part[threadIdx.x] = l;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, part[0] * inv_count);
}

hipError_t launch_l1_loss(hipStream_t st, size_t npix, const float* o, int os,
                          const float* t, float wd, float wn, float inv_count,
                          bf16* g, float* loss) {
  if (os % 8) return hipErrorInvalidValue;
  // few work-groups, since each ends with an atomic add to the one sum
  // (1.6 million pixels in 6144: 84 us)
  NET_LAUNCH(k_l1_loss,
             dim3((unsigned)std::min<size_t>((npix + 255) / 256, 1024)),
             dim3(256), 0,
             st, npix, o, os, reinterpret_cast<const float4*>(t), wd, wn,
             inv_count, g, loss);
}

__global__ void __launch_bounds__(256)
k_adam(size_t n, float* __restrict__ w, const float* __restrict__ g,
       float* __restrict__ m, float* __restrict__ v, float lr, float b1,
       float b2, float eps, float c1, float c2, bf16* __restrict__ wb) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  wb[i] = (bf16)wi;
}

hipError_t launch_adam(hipStream_t st, size_t n, float* w, const float* g,
                       float* m, float* v, float lr, float b1, float b2,
                       float eps, float c1, float c2, bf16* wb) {
  NET_LAUNCH(k_adam, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n,
             w, g, m, v, lr, b1, b2, eps, c1, c2, wb);
}

__global__ void __launch_bounds__(256)
k_to_bf16(size_t n, const float* __restrict__ x, bf16* __restrict__ y) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) y[i] = (bf16)x[i];
}

hipError_t launch_to_bf16(hipStream_t st, size_t n, const float* x, bf16* y) {
  NET_LAUNCH(k_to_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
             n, x, y);
}

// ---------------------------------------------------------------------
// matching cost volumes: the network's explicit stereo evidence.  The
// packed pair is box-averaged (4 x 4 for the coarse volume, 2 x 2 for the
// fine one), and at every pixel of that resolution channel d of the
// volume is the mean over the 3 x 3 window of the summed |r, g, b|
// differences between the first image at (x + i, y + j) and the second at
// (x + i - d, y + j), d = 0 .. levels - 1 (coarse: 48 quarter pixels,
// 0 .. 188 px at full resolution; fine: 64 half pixels, 0 .. 126 px);
// coordinates are clamped to the image.  No parameters: the network
// learns what follows it.
// ---------------------------------------------------------------------
__global__ void __launch_bounds__(256)
k_down4(int N, int H, int W, const bf16* __restrict__ x,
        bf16* __restrict__ y) {
  const int Ho = H / 4, Wo = W / 4;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)N * Ho * Wo) return;
  const int xo = (int)(i % Wo);
  const size_t r = i / Wo;
  const int yo = (int)(r % Ho), n = (int)(r / Ho);
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int dy = 0; dy < 4; ++dy)
    for (int dx = 0; dx < 4; ++dx) {
      const bf16x8 v = load8(
          x + (((size_t)n * H + 4 * yo + dy) * W + 4 * xo + dx) * 8);
#pragma unroll
      for (int c = 0; c < 8; ++c) s[c] += (float)v[c];
    }
  bf16x8 o;
#pragma unroll
  for (int c = 0; c < 8; ++c) o[c] = (bf16)(s[c] * 0.0625f);
  *reinterpret_cast<bf16x8*>(y + i * 8) = o;
}

hipError_t launch_down4(hipStream_t st, int N, int H, int W, const bf16* x,
                        bf16* y) {
  const size_t n = (size_t)N * (H / 4) * (W / 4);
  NET_LAUNCH(k_down4, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, N,
             H, W, x, y);
}

// A work-group computes every level of 64 consecutive pixels of one row.
// It first stages, as float4 (r, g, b, 0) with clamped coordinates, the
// three window rows of the first image over columns x0 - 1 .. x0 + 64 and
// of the second image over x0 - levels .. x0 + 64 (the columns any level
// of the segment reads); then an item is a (pixel, 8 consecutive levels):
// levels 8 g .. 8 g + 7 over the taps x - 1 .. x + 1 read the second image
// at x + 1 - 8 g - 9 .. x + 1 - 8 g, ten pixels per window row.  levels: a
// multiple of 8, at most kCvMaxLevels.
constexpr int kCvSeg = 64;
constexpr int kCvMaxLevels = 64;
constexpr int kCvAW = kCvSeg + 2;                  // first-image columns
constexpr int kCvBW = kCvSeg + 1 + kCvMaxLevels;   // second-image columns

__global__ void __launch_bounds__(256)
k_cost_volume(int N, int H4, int W4, int levels, int segs,
              const bf16* __restrict__ d4, bf16* __restrict__ cv) {
  __shared__ float4 sa[3][kCvAW];
  __shared__ float4 sb[3][kCvBW];
  int t = blockIdx.x;
  const int seg = t % segs;
  t /= segs;
  const int y = t % H4, n = t / H4;
  const int x0 = seg * kCvSeg;
  const int bw = kCvSeg + 1 + levels;  // second-image columns x0 - levels ..
  for (int i = threadIdx.x; i < 3 * (kCvAW + bw); i += 256) {
    const int j = i / (kCvAW + bw), c = i - j * (kCvAW + bw);
    const int yy = min(max(y + j - 1, 0), H4 - 1);
    const bf16* row = d4 + ((size_t)n * H4 + yy) * W4 * 8;
    if (c < kCvAW) {
      const bf16x8 v = load8(row + (size_t)min(max(x0 - 1 + c, 0), W4 - 1) * 8);
      sa[j][c] = make_float4((float)v[0], (float)v[1], (float)v[2], 0.0f);
    } else {
      const int cb = c - kCvAW;
      const bf16x8 v =
          load8(row + (size_t)min(max(x0 - levels + cb, 0), W4 - 1) * 8);
      sb[j][cb] = make_float4((float)v[4], (float)v[5], (float)v[6], 0.0f);
    }
  }
  __syncthreads();
  const int groups = levels / 8;
  for (int item = threadIdx.x; item < kCvSeg * groups; item += 256) {
    const int xl = item % kCvSeg, grp = item / kCvSeg;
    const int x = x0 + xl;
    if (x >= W4) continue;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // second-image column of t = 1, d = 8 g, as an index into sb
    const int b0 = xl + 1 - 8 * grp + levels;
    for (int j = 0; j < 3; ++j) {
      float4 ar[3], br[10];
#pragma unroll
      for (int tt = 0; tt < 3; ++tt) ar[tt] = sa[j][xl + tt];
      // br[m] = second image at column x + 1 - 8 g - m
#pragma unroll
      for (int m = 0; m < 10; ++m) br[m] = sb[j][b0 - m];
      // tap tt (x + tt - 1) at level 8 g + k reads br[2 - tt + k]
#pragma unroll
      for (int tt = 0; tt < 3; ++tt)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float4 bb = br[2 - tt + k];
          acc[k] += (fabsf(ar[tt].x - bb.x) + fabsf(ar[tt].y - bb.y)) +
                    fabsf(ar[tt].z - bb.z);
        }
    }
    bf16x8 o;
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = (bf16)(acc[k] * (1.0f / 9.0f));
    const size_t p = ((size_t)n * H4 + y) * W4 + x;
    *reinterpret_cast<bf16x8*>(cv + p * levels + grp * 8) = o;
  }
}

hipError_t launch_cost_volume(hipStream_t st, int N, int H4, int W4,
                              int levels, const bf16* d4, bf16* cv) {
  if (levels < 8 || levels % 8 || levels > kCvMaxLevels)
    return hipErrorInvalidValue;
  const int segs = (W4 + kCvSeg - 1) / kCvSeg;
  const size_t blocks = (size_t)N * H4 * segs;
  NET_LAUNCH(k_cost_volume, dim3((unsigned)blocks), dim3(256), 0, st, N, H4,
             W4, levels, segs, d4, cv);
}

__global__ void __launch_bounds__(256)
k_pack_pair(const float* __restrict__ left, const float* __restrict__ right,
            int W, int H, int C, int stride, int Hp, int Wp, int mirror,
            bf16* __restrict__ x) {
  const int xo = blockIdx.x * 64 + (threadIdx.x & 63);
  const int yo = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (xo >= Wp || yo >= Hp) return;
  const int ys = min(yo, H - 1);
  int xs = min(xo, W - 1);
  const float* a = left;
  const float* b = right;
  if (mirror) {
    xs = W - 1 - xs;
    a = right;
    b = left;
  }
  bf16x8 v;
  const float* pa = a + (size_t)ys * stride;
  const float* pb = b + (size_t)ys * stride;
  for (int c = 0; c < 4; ++c) {
    v[c] = (bf16)(C == 1 ? pa[xs] : pa[4 * (size_t)xs + c]);
    v[4 + c] = (bf16)(C == 1 ? pb[xs] : pb[4 * (size_t)xs + c]);
  }
  *reinterpret_cast<bf16x8*>(x + ((size_t)yo * Wp + xo) * 8) = v;
}

hipError_t launch_pack_pair(hipStream_t st, const float* left,
                            const float* right, int W, int H, int channels,
                            int stride, int Hp, int Wp, int mirror, bf16* x) {
  const dim3 grid((unsigned)((Wp + 63) / 64), (unsigned)((Hp + 3) / 4));
  NET_LAUNCH(k_pack_pair, grid, dim3(256), 0, st, left, right, W, H, channels,
             stride, Hp, Wp, mirror, x);
}

}  // namespace net
}  // namespace pm
