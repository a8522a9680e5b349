// pm_net_kernels.h -- internal interface of the plane-proposal network kernels
// (pm_net.hip): a 3x3 convolution on bf16 NHWC activations with fp32
// accumulation on the matrix cores, its weight gradient, and the small
// kernels a U-Net training step and a proposal need.  Internal to the
// library: the public boundary is include/pm_net.h.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "pm_engine.h"

namespace pm {
namespace net {

typedef __bf16 bf16;

// K of a 3x3 convolution over cin channels, padded to the MFMA's 32
__host__ __device__ inline int conv_kpad(int cin) {
  return (9 * cin + 31) / 32 * 32;
}
// output channels padded to the 32 of a work-group's tile
__host__ __device__ inline int conv_cpad(int cout) {
  return (cout + 31) / 32 * 32;
}

// One 3x3 convolution, stride 1, zero padding, dilation `dil`.  The input
// is the channel concatenation of x1 (c1 channels, N x H x W) and x2 (c2
// channels; N x H x W, or N x ceil(H/2) x ceil(W/2) read nearest-upsampled
// when up2 is set).  c1, c2 and cout are multiples of 8.  Weights
// w[co][k], co < conv_cpad(cout), k = tap * (c1 + c2) + ci < conv_kpad(c1 +
// c2), tap = 3 (dy + 1) + (dx + 1), bf16, zero beyond the real ones.
// Output (N x H x W, channel stride ys >= cout) with the bias (when not
// null) and an optional ReLU: bf16 into y, or fp32 into yf when set.  For
// the gradient of an input: mask (N x H x W, channel stride ys): the output
// is 0 where it is not above 0; yf2: output channels from split on go there,
// with channel stride cout - split.  split is a multiple of 4.
struct ConvArgs {
  const bf16* x1 = nullptr;
  const bf16* x2 = nullptr;
  int c1 = 0, c2 = 0, up2 = 0;
  const bf16* w = nullptr;
  const float* bias = nullptr;
  int N = 0, H = 0, W = 0;
  int cout = 0, dil = 1, relu = 0;
  bf16* y = nullptr;
  float* yf = nullptr;
  int ys = 0;
  const bf16* mask = nullptr;
  float* yf2 = nullptr;
  int split = 0;
};
hipError_t launch_conv(hipStream_t st, const ConvArgs& a);

// Weight gradient of the convolution above: dw[co][k] = sum over the
// N x H x W pixels of g[p][co] * x(p, k), g bf16 with cout channels, for the
// real co and k; and db[co] = sum of g[p][co] when db is not null.  The
// pixels (image, row, column) are summed 1024 at a time, in order, with one
// fp32 fmaf each; then those sums in order, in fp32.  c1, c2 and cout even; when up2, H
// and W even, c1 and c2 multiples of 32.  part: wgrad_part_floats floats to
// work in.
size_t wgrad_part_floats(int N, int H, int W, int cin, int cout);
hipError_t launch_conv_wgrad(hipStream_t st, const ConvArgs& a,
                             const bf16* g, float* part, float* dw,
                             float* db);

// w'[ci][k'] for the gradient of the input: the convolution of the output
// gradient (cout channels) with the flipped, transposed kernel, k' = (8 -
// tap) * cout + co; w' has conv_cpad(cin) rows of conv_kpad(cout)
// for up to kMaxFlips layers in one launch
struct FlipLayer {
  const bf16* w = nullptr;
  bf16* wt = nullptr;
  int cin = 0, cout = 0;
};
constexpr int kMaxFlips = 16;
hipError_t launch_flip_weights(hipStream_t st, const FlipLayer* layers,
                               int n);

// Masked gradients, bf16, C a multiple of 4.  k_mask_pool: of a tensor whose
// gradient is g (N x H x W x C, fp32) plus a quarter of that of its 2 x 2
// average, gp; k_mask_up: of a tensor (N x H x W x C) read nearest-upsampled,
// the sum of g (N x 2H x 2W x C) over 2 x 2 blocks.  0 where y is not above 0.
hipError_t launch_mask_pool(hipStream_t st, int N, int H, int W, int C,
                            const float* g, const float* gp, const bf16* y,
                            bf16* out);
hipError_t launch_mask_up(hipStream_t st, int N, int H, int W, int C,
                          const float* g, const bf16* y, bf16* out);

// 2 x 2 average pooling, bf16 (N x H x W x C -> N x H/2 x W/2 x C, H and
// W even, C a multiple of 8)
hipError_t launch_avgpool(hipStream_t st, int N, int H, int W, int C,
                          const bf16* x, bf16* y);

// Masked L1 loss of the head output o (N x H x W x os fp32, channels 0..3
// = disparity / kDispScale, nx, ny, nz) against t (N x H x W x 4; a
// disparity below 0 marks a pixel without a target): g = dloss / do
// (channels 0..3, 0 elsewhere; bf16, os a multiple of 8), loss += sum /
// count.  count: valid pixels.
hipError_t launch_l1_loss(hipStream_t st, size_t npix, const float* o,
                          int os, const float* t, float wd, float wn,
                          float inv_count, bf16* g, float* loss);

// Adam on n fp32 parameters; writes their bf16 copy
hipError_t launch_adam(hipStream_t st, size_t n, float* w, const float* g,
                       float* m, float* v, float lr, float b1, float b2,
                       float eps, float c1, float c2, bf16* wb);

// fp32 -> bf16, n elements
hipError_t launch_to_bf16(hipStream_t st, size_t n, const float* x, bf16* y);

// network input of a stereo pair: N = 1, Hp x Wp x 8 bf16 = (left rgba,
// right rgba) of the engine's images (channels 1 or 4, row stride in
// floats), edge-replicated beyond W x H; mirror: the pair seen as a left
// view by flipping both images horizontally and swapping them
hipError_t launch_pack_pair(hipStream_t st, const float* left,
                            const float* right, int W, int H, int channels,
                            int stride, int Hp, int Wp, int mirror, bf16* x);

// disparity levels of the matching cost volumes: the coarse one at
// quarter resolution (quarter pixels), the fine one at half resolution
constexpr int kCvLevels = 48;
constexpr int kCvFineLevels = 64;

// 4 x 4 box average of N x H x W x 8 bf16 (H, W multiples of 4)
hipError_t launch_down4(hipStream_t st, int N, int H, int W, const bf16* x,
                        bf16* y);

// N x H4 x W4 x levels bf16 matching costs of a downsampled pair
// (N x H4 x W4 x 8: first image rgba, second image rgba); levels a
// multiple of 8, at most 64
hipError_t launch_cost_volume(hipStream_t st, int N, int H4, int W4,
                              int levels, const bf16* d4, bf16* cv);

}  // namespace net

}  // namespace pm
