// pm_engine.hip -- gfx950 kernels of the PatchMatch stereo engine.
//
// Work decomposition (kernels that evaluate plane costs):
//  - a work-group is a block of pixels, each wavefront a run of one row: 64
//    x 4 pixels in general; for the propagate also 128 x 8 with a window of
//    the other view (the wide tile, images that fill the GPU with it), or
//    16 x 4 with four lanes per pixel (teams, images that do not fill it);
//  - blocks are renumbered so that each XCD walks one contiguous band of
//    the image (its L2 then holds the rows the band reads);
//  - the block stages its own-view tile (pixels plus an r halo: colour and
//    gradient sign bits) in LDS once; support weights are recomputed per
//    tap from that tile instead of being streamed from HBM;
//  - the other view is sampled from its colour and gradient planes (two
//    adjacent 16-byte records of each per linear sample), by the wide tile
//    from packed 12-byte colours and the window's gradients in LDS.
// The cost loops run wave-uniformly over patch rows (one image row per
// wavefront) and every lane stays resident (no early return): lanes are
// masked with flags, and kernels reach the block barrier with all threads.
//
// Per-pixel work follows cvt/cl/kernel/pmhstereo.cl (cited per kernel);
// the arithmetic contract is in pm_device.h.
#include <algorithm>
#include <climits>
#include <cmath>
#include <type_traits>

#include "pm_device.h"
#include "pm_engine.h"

namespace pm {

// ---------------------------------------------------------------------
// A^(2^i) mod M, folded at compile time
// ---------------------------------------------------------------------
struct ApowTable {
  uint64_t v[64];
};

constexpr uint64_t cx_mulmod(uint64_t a, uint64_t b) {
  unsigned __int128 p = (unsigned __int128)a * b;
  while ((p >> 64) != 0)
    p = (unsigned __int128)(uint64_t)(p >> 64) * kMwcR + (uint64_t)p;
  uint64_t r = (uint64_t)p;
  return r >= kMwcM ? r - kMwcM : r;
}

constexpr ApowTable make_apow() {
  ApowTable t{};
  uint64_t sq = kMwcA;
  for (int i = 0; i < 64; ++i) {
    t.v[i] = sq;
    sq = cx_mulmod(sq, sq);
  }
  return t;
}

__constant__ ApowTable c_apow_table = make_apow();

// state of draw k: decode(BASE * A^k mod M), x = v / A, c = v % A
__device__ __forceinline__ Mwc mwc_jump(uint64_t k) {
  uint64_t acc = 1;
  for (int i = 0; k != 0; ++i, k >>= 1)
    if (k & 1) acc = mulmod_m(acc, c_apow_table.v[i]);
  uint64_t v = mulmod_m(kMwcBase, acc);
  Mwc s;
  s.x = (uint32_t)(v / kMwcA);
  s.c = (uint32_t)(v % kMwcA);
  return s;
}

// ---------------------------------------------------------------------
// block geometry and LDS layout
// ---------------------------------------------------------------------
constexpr int kTX = kBlockCols;  // block width = one wavefront
constexpr int kTY = kBlockRows;  // wavefronts (rows) per block
constexpr int kXcds = 8;

// the blocks of a full-image launch: every block column and row
__host__ __forceinline__ dim3 grid_for(const Geometry& g) {
  return dim3((unsigned)((g.W + kTX - 1) / kTX),
              (unsigned)((g.H + kTY - 1) / kTY));
}

// records after a window row's columns (block_setup_at)
constexpr int kWinEdge = 8;

// LDS bytes of a tile block of cols x rows pixels: the own-view tile
// (colour and sign bits), followed for the colour+gradient cost by a tile
// of the own view's gradients, followed by the window of the other view's
// gradients (wcols columns, 0: none)
__host__ __device__ __forceinline__ size_t tile_lds_bytes(int R, int kind,
                                                          int cols, int rows,
                                                          int wcols) {
  const size_t tile = (size_t)(cols + 2 * R) * (rows + 2 * R);
  return ((kind == kCostColorGrad ? 2 * tile : tile) +
          (wcols ? (size_t)(wcols + kWinEdge) * (rows + 2 * R) : 0)) *
         sizeof(float4);
}

// The wide tile of the propagate: 128 x 8 pixels, 16 wavefronts, one to a
// CU, with the window of the other view's gradients in LDS.
constexpr int kWideCols = 128, kWideRows = 8;
constexpr size_t kLdsPerCu = 160 * 1024;
constexpr int kCus = 256;

// The window of a wide tile: x' = x - d (left view) or x + d (right), d in
// [0, dmax], and room on both sides for the patch, KLT's neighbours and
// the slope of steep planes.  A margin of 2 R + 8 was measured against R +
// 4 (1280 x 720, R = 4): 45.2 against 47.4 ms, for the texture reads of
// the lanes that leave the window.
__host__ __device__ __forceinline__ Window window_of(int R, float dmax,
                                                     int lr) {
  const int d = (int)ceilf(dmax), margin = 2 * R + 8;
  Window w;
  w.left = (lr ? d : 0) + margin;
  w.cols = kWideCols + d + 2 * margin;
  return w;
}

// sign bits of a gradient as one byte per component: byte k is 0xff when
// component k has its sign bit set (the tile's .w holds the own view's)
__device__ __forceinline__ uint32_t expand_signs(uint32_t m) {
  return ((m & 1u) ? 0x000000ffu : 0u) | ((m & 2u) ? 0x0000ff00u : 0u) |
         ((m & 4u) ? 0x00ff0000u : 0u) | ((m & 8u) ? 0xff000000u : 0u);
}

// Work-group (bx, by) of the image for the hardware work-group id.
// Consecutive work-groups are dispatched round-robin over the XCDs; this
// numbering gives XCD k the k-th contiguous eighth of the blocks.
__device__ __forceinline__ void xcd_block(int* bx, int* by) {
  const int nbx = (int)gridDim.x;
  const int n = nbx * (int)gridDim.y;
  const int hw = (int)blockIdx.y * nbx + (int)blockIdx.x;
  const int xcd = hw % kXcds, j = hw / kXcds;
  const int per = n / kXcds, rem = n % kXcds;
  const int logical = xcd * per + min(xcd, rem) + j;
  *bx = logical % nbx;
  *by = logical / nbx;
}

// LDS records with their address space in the type: a read of the window
// and the read of the texture row it may need instead stay two reads, never
// one generic read
typedef float v4f __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(3))) v4f* LdsRow;

__device__ __forceinline__ float4 lds_at(LdsRow p, int i) {
  const v4f v = p[i];
  return make_float4(v.x, v.y, v.z, v.w);
}

// Everything one lane needs to evaluate planes for its pixel.
struct Lane {
  int W, H, R;
  float Wf, cw;
  int x, y;      // y is the same for the whole wavefront
  bool valid;
  float xf, yf;
  size_t p;
  float4 tc;     // own pixel colour
  float bilw;    // sum of its support weights
  LdsRow trow0;         // LDS tile at this lane: tap (dx, dy) is
                        // trow0[(dy + R) * TW + dx + R]
  int TW;
  int GT;               // offset of the gradient tile (records), when
                        // staged: tap (dx, dy)'s gradient is at
                        // trow0[GT + (dy + R) * TW + dx + R]
  float kw;             // colour+gradient cost's support-weight factor
  int TS;               // texel row stride (records, with the edge pads)
  size_t GP;            // offset of the gradient plane (records)
  const float4* __restrict__ tex2;  // other view's colour record (0, 0)
  bool tame;            // both images are tame (see "Tame images")
  bool edge;            // a patch of this wavefront crosses the left or
                        // right border (or the columns next to it)
  LdsRow wrow0;         // window of the other view's gradients at this
                        // lane's first patch row: column c of row dy is
                        // wrow0[(dy + R) * wstride + c - wlo],
                        // and the records from wcols on are the row's
                        // right edge (4) and left edge (4), kEdge*
  int wlo, wcols, wstride;
  const float* __restrict__ col12;  // other view's packed colour (0, 0)
  float flo, fhi;       // x' in [flo, fhi] reads inside image and window
  float safe;           // a column that does: the block's first
  int sub;              // this lane's number in its pixel's team
};

// Block prologue shared by the cost-evaluating kernels, for the block
// (bx, by) of tile blocks of 64 kWX x kRows pixels: stages the own-view tile
// (r, g, b, gradient sign bits), for kGrad the tile of its gradients after
// it, for kWin the window of the other view's gradients after those, and
// returns the lane context.  For kRB (a red-black pass, g.color = 0 or 1)
// the block covers twice the columns and lane i takes column 2 i + ((y +
// color) & 1) of its row, the pixel of the pass's colour.  Must be reached
// by every thread of the block; the block is 64 kWX x kRows threads, and
// lanes of rows from row_end on are invalid.
// kTeam lanes share a pixel (see "Teams"), so the block covers kTeam times
// fewer columns.
template <bool kGrad, bool kRB, int kRows, int kWX = 1, bool kWin = false,
          int kTeam = 1>
__device__ Lane block_setup_at(const Geometry& g, const ViewBufs& self,
                               const ViewBufs& other, float4* smem, int x0,
                               int y0, int row_end, Window win = Window()) {
  const int R = g.R, W = g.W, H = g.H;
  constexpr int kThreads = kTX * kWX * kRows;
  const int cols = (kRB ? 2 : 1) * kTX * kWX / kTeam;
  const int TW = cols + 2 * R, TH = kRows + 2 * R;
  const int tid = threadIdx.y * (kTX * kWX) + threadIdx.x;
  const size_t gplane = (size_t)g.TS * H;
  for (int i = tid; i < TW * TH; i += kThreads) {
    const int gx = x0 - R + i % TW, gy = y0 - R + i / TW;
    float4 v = mk4(0.0f, 0.0f, 0.0f, 0.0f), gv = v;
    if (gx >= 0 && gx < W && gy >= 0 && gy < H) {
      const size_t rec = (size_t)gy * g.TS + kTexPadL + gx;
      const float4 a = self.tex[rec];
      v = mk4(a.x, a.y, a.z,
              __uint_as_float(expand_signs(self.sgn[(size_t)gy * W + gx])));
      if (kGrad) gv = self.tex[gplane + rec];
    }
    smem[i] = v;
    if (kGrad) smem[TW * TH + i] = gv;
  }
  float4* wtile = smem + (kGrad ? 2 : 1) * TW * TH;
  if (kWin) {
    // columns beyond the image replicate its edge texels, as the pads do;
    // after a row's columns the four texels that x' clamped to W reads (W -
    // 1 .. W + 2) and the four that x' clamped to -1 reads (-2 .. 1)
    const int stride = win.cols + kWinEdge;
    for (int i = tid; i < stride * TH; i += kThreads) {
      const int gy = y0 - R + i / stride, c = i % stride;
      int gx = x0 - win.left + c;
      if (c >= win.cols) gx = c < win.cols + 4 ? W - 1 : c - win.cols - 6;
      gx = clampi(gx, 0, W - 1);
      if (gy >= 0 && gy < H)
        wtile[i] = other.tex[gplane + (size_t)gy * g.TS + kTexPadL + gx];
    }
  }
  __syncthreads();
  // the row index is uniform per wavefront: keep it scalar
  const int ly = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
  // first column of this wavefront
  const int wx0 =
      x0 + __builtin_amdgcn_readfirstlane((int)threadIdx.x / kTX) *
               (kRB ? 2 * kTX : kTX);
  const int lx0 = (int)threadIdx.x / kTeam;
  const int lx = kRB ? 2 * lx0 + ((y0 + ly + g.color) & 1) : lx0;
  Lane L;
  L.W = W;
  L.H = H;
  L.R = R;
  L.Wf = (float)W;
  L.cw = g.color_weight;
  L.x = x0 + lx;
  L.y = y0 + ly;
  L.valid = L.x < W && L.y < row_end;
  L.xf = (float)L.x;
  L.yf = (float)L.y;
  L.p = L.valid ? (size_t)L.y * W + L.x : 0;
  L.TW = TW;
  L.GT = TW * TH;
  L.kw = g.cost_weight;
  L.TS = g.TS;
  L.GP = (size_t)g.TS * g.H;
  L.trow0 = (LdsRow)(smem + ly * TW + lx);
  L.tex2 = other.tex + kTexPadL;
  L.tame = false;
  L.edge = true;
  L.sub = (int)threadIdx.x % kTeam;
  if (kWin || kTeam > 1)
    L.tame = __builtin_amdgcn_readfirstlane(
                 (int)(*wild_word(self.tex, g.TS, H) |
                       *wild_word(other.tex, g.TS, H))) == 0;
  if (kWin) {
    L.edge = wx0 - R < 1 || wx0 + (kRB ? 2 * kTX : kTX) - 1 + R > W - 2;
    L.wcols = win.cols;
    L.wstride = win.cols + kWinEdge;
    L.wrow0 = (LdsRow)(wtile + ly * L.wstride);
    L.wlo = x0 - win.left;
    // KLT reads texels floor(x') - 1 .. floor(x') + 2
    L.flo = (float)max(L.wlo + 1, 0);
    L.fhi = (float)min(L.wlo + win.cols - 4, W - 1);
    L.safe = (float)x0;
    L.col12 = packed_colours(other.tex, g.TS, H) + 3 * kTexPadL;
  }
  L.tc = lds_at(L.trow0, R * TW + R);
  L.bilw = L.valid
               ? self.tex[(size_t)L.y * g.TS + kTexPadL + L.x].w
               : 1.0f;
  return L;
}

// The same for the full-image launches: 64 x kTY blocks, the block from
// the hardware work-group id in XCD order.
template <bool kGrad>
__device__ Lane block_setup(const Geometry& g, const ViewBufs& self,
                            const ViewBufs& other, float4* smem) {
  int bx, by;
  xcd_block(&bx, &by);
  return block_setup_at<kGrad, false, kTY>(g, self, other, smem, bx * kTX,
                                           by * kTY, g.H);
}

// Linear sample (CLK_FILTER_LINEAR, CLK_ADDRESS_CLAMP_TO_EDGE,
// pmhstereo.cl:71) of the other view at column u of a texel row:
// t0 + a*(t1 - t0), from adjacent records of the colour and the gradient
// plane.  The edge-padded rows stand in for the coordinate clamp: every
// column the kernels sample at lies in [-1, W], and the records it reads
// there are the image's or copies of its edge texels.
struct Sample {
  float r, g, b;
  float4 grad;
};

struct Texel {
  float4 A, G;  // (r, g, b, bilw), gradient
};

__device__ __forceinline__ Sample lerp_texels(const Texel& t0,
                                              const Texel& t1, float a) {
  Sample s;
  s.r = fmaf(a, t1.A.x - t0.A.x, t0.A.x);
  s.g = fmaf(a, t1.A.y - t0.A.y, t0.A.y);
  s.b = fmaf(a, t1.A.z - t0.A.z, t0.A.z);
  s.grad.x = fmaf(a, t1.G.x - t0.G.x, t0.G.x);
  s.grad.y = fmaf(a, t1.G.y - t0.G.y, t0.G.y);
  s.grad.z = fmaf(a, t1.G.z - t0.G.z, t0.G.z);
  s.grad.w = fmaf(a, t1.G.w - t0.G.w, t0.G.w);
  return s;
}

// texel at record p of the colour plane and p + gp of the gradient plane
__device__ __forceinline__ Texel texel_at(const float4* __restrict__ p,
                                          size_t gp) {
  Texel t;
  t.A = p[0];
  t.G = p[gp];
  return t;
}

// 8 x the gradient sign mismatches between expanded sign bytes m1x and
// the signs of g.  v_perm_b32 selectors 9 and 11 replicate the sign bit of
// the low and the high source operand into a whole byte, so the signs of
// g arrive in the layout of m1x; xor and count.
__device__ __forceinline__ int sign_mismatches8(uint32_t m1x, float4 g) {
  const uint32_t lo = __builtin_amdgcn_perm(__float_as_uint(g.y),
                                            __float_as_uint(g.x), 0x0c0c0b09u);
  const uint32_t hi = __builtin_amdgcn_perm(__float_as_uint(g.w),
                                            __float_as_uint(g.z), 0x0b090c0cu);
  return __popc((lo | hi) ^ m1x);
}

// ---------------------------------------------------------------------
// Tame images.  The loops below exist twice.  The general ones
// (cost_eval, cost_eval_cg, klt_pass) take any float an image can hold.
// The tame ones run when every colour value of both images is 0 or lies in
// [2^-60, lim] in magnitude and every alpha is finite, lim = 39 / max(colour
// weight, cost weight) (at most 1e4): ordinary images.  k_prepare decides
// it (wild_word).  There, and only there,
//  - no sample, difference or weight is NaN or infinite, no gradient is -0;
//  - the exponent of a support weight lies in [-80, 0], so the weight is a
//    normal number and 2^k is one integer addition to its exponent;
//  - min(|d|, 0.05) * 20 is min(20 |d|, 1) (rounding is monotone and 0.05 *
//    20 rounds to 1), one multiplication with the clamp modifier.
// Same operations, same order, same bits as the general loops.
//
// What they are shaped for, measured on gfx950 with four or more
// wavefronts per SIMD: f32 add, sub, mul, fma and mov with operands in
// vector registers, literals or inline constants issue in 2.3-2.5 cycles
// per wavefront; min, max, compares, cndmask, floor, conversions, perm,
// shifts, and every instruction that reads a scalar register, in 4.2-4.6.
// A gather of 16 bytes per lane holds a CU's texture path for 16 cycles
// however many lanes take part, so a load that one lane needs costs what a
// load of all lanes costs.  Hence constants in vector registers, the clamp
// modifier, rounding and 2^k by additions, and loads that all lanes issue
// together, early.
// ---------------------------------------------------------------------

typedef std::true_type Yes;
typedef std::false_type No;

// a constant the compiler keeps in a vector register
__device__ __forceinline__ float vconst(float v) {
  float r;
  asm("v_mov_b32 %0, %1" : "=v"(r) : "s"(v));
  return r;
}

// support_weight for tame images (cw negated): the same polynomial, with
// rint by the 1.5 * 2^23 addition (exact: |t| < 2^22) and 2^k by adding k
// to the exponent field
__device__ __forceinline__ float weight_tame(float dx, float dy, float dz,
                                             float negw) {
  const float x = fabsf(gray3(dx, dy, dz)) * negw;
  const float t = x * 0x1.715476p+0f;
  const float kf = t + 12582912.0f;
  const float k = kf - 12582912.0f;
  float r = fmaf(k, -0x1.62e400p-1f, x);
  r = fmaf(k, -0x1.7f7d1cp-20f, r);
  float p = 0x1.a01a02p-13f;
  p = fmaf(p, r, 0x1.6c16c2p-10f);
  p = fmaf(p, r, 0x1.111112p-7f);
  p = fmaf(p, r, 0x1.555556p-5f);
  p = fmaf(p, r, 0x1.555556p-3f);
  p = fmaf(p, r, 0.5f);
  p = fmaf(p, r, 1.0f);
  p = fmaf(p, r, 1.0f);
  return __uint_as_float(__float_as_uint(p) + (__float_as_uint(kf) << 23));
}

// min(|d|, 0.05) * 20 for finite d
__device__ __forceinline__ float clamp20(float d, float twenty) {
  return __builtin_amdgcn_fmed3f(fabsf(d) * twenty, 0.0f, 1.0f);
}

// sign_mismatches8 as a float: the count lands in the mantissa of 2^23
__device__ __forceinline__ float sign_mismatches8f(uint32_t m1x, float4 g) {
  const uint32_t lo = __builtin_amdgcn_perm(__float_as_uint(g.y),
                                            __float_as_uint(g.x), 0x0c0c0b09u);
  const uint32_t hi = __builtin_amdgcn_perm(__float_as_uint(g.w),
                                            __float_as_uint(g.z), 0x0b090c0cu);
  const uint32_t n = (uint32_t)__popc((lo | hi) ^ m1x) + 0x4b000000u;
  return __uint_as_float(n) - 8388608.0f;
}

// rows of the other view at image row qy: texel 0's packed colour and its
// gradient record (both uniform); texel t is 12 t and 16 t bytes on
__device__ __forceinline__ const char* colour_row(const Lane& L, int qy) {
  return reinterpret_cast<const char*>(L.col12 + (size_t)qy * L.TS * 3);
}
__device__ __forceinline__ const char* gradient_row(const Lane& L, int qy) {
  return reinterpret_cast<const char*>(L.tex2 + L.GP + (size_t)qy * L.TS);
}

struct Rgb {
  float r, g, b;
};

// 16 and 8 bytes at a 4-byte alignment
__device__ __forceinline__ float4 load16(const char* __restrict__ p) {
  float4 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}
__device__ __forceinline__ float2 load8b(const char* __restrict__ p) {
  float2 v;
  __builtin_memcpy(&v, p, 8);
  return v;
}

__device__ __forceinline__ float4 lerp4(float4 t0, float4 t1, float a) {
  return mk4(fmaf(a, t1.x - t0.x, t0.x), fmaf(a, t1.y - t0.y, t0.y),
             fmaf(a, t1.z - t0.z, t0.z), fmaf(a, t1.w - t0.w, t0.w));
}
__device__ __forceinline__ Rgb lerp_rgb(const Rgb& t0, const Rgb& t1,
                                        float a) {
  return Rgb{fmaf(a, t1.r - t0.r, t0.r), fmaf(a, t1.g - t0.g, t0.g),
             fmaf(a, t1.b - t0.b, t0.b)};
}

// The gradients of kN consecutive texels from texel t on, from the window
// row wrow.  For kInside every lane's lie inside the window.  Otherwise x'
// clamped to the image's ends (t = W - 1 or -2 for KLT's four) finds them
// after the row's columns, and lanes whose texels lie elsewhere outside the
// window read the texture row.
template <int kN, bool kInside>
__device__ __forceinline__ void window_gradients(
    const Lane& L, LdsRow wrow, const char* __restrict__ grow, int t,
    bool needed, float4 (&G)[kN]) {
  uint32_t c = (uint32_t)(t - L.wlo);
  const bool out = !kInside && c > (uint32_t)(L.wcols - kN);
  if (!kInside && __builtin_expect(__any(out), 0)) {
    asm volatile("");  // stays a scalar branch
    bool far = out && needed;
    if (out) {
      c = 0u;
      if (kN == 4 && t >= L.W - 1) c = (uint32_t)L.wcols;
      if (kN == 4 && t <= -2) c = (uint32_t)L.wcols + 4u;
      far = far && c == 0u;
    }
#pragma unroll
    for (int k = 0; k < kN; ++k) G[k] = lds_at(wrow, (int)c + k);
    if (far) {
      const char* g = grow + (ptrdiff_t)t * 16;
#pragma unroll
      for (int k = 0; k < kN; ++k)
        G[k] = *reinterpret_cast<const float4*>(g + 16 * k);
      // waited for here, not after the branches join: there the wait would
      // be for the look-ahead loads too
#pragma unroll
      for (int k = 0; k < kN; ++k)
        asm volatile("" : "+v"(G[k].x), "+v"(G[k].y), "+v"(G[k].z),
                     "+v"(G[k].w));
    }
  } else {
#pragma unroll
    for (int k = 0; k < kN; ++k) G[k] = lds_at(wrow, (int)c + k);
  }
}

// Whether every lane's x' lies in [flo, fhi] over the row: x' is monotone
// in the column (so is its rounding), so its ends decide; a NaN does not
// pass.
__device__ __forceinline__ bool row_inside(const Lane& L, float sx, float rowb,
                                           float sz, float px) {
  const float e0 = fmaf(sx, px, rowb) + sz;
  const float e1 = fmaf(sx, px + (float)(2 * L.R), rowb) + sz;
  const bool in = e0 >= L.flo && e0 <= L.fhi && e1 >= L.flo && e1 <= L.fhi;
  return __all(in);
}

// One cost tap's sample in flight: the colours of the two texels of x', the
// first one's index, x's fraction, and m, 1 when the tap counts (0 <= x' <
// W, own pixel inside the image), else 0.
struct CostTap {
  Rgb c0, c1;
  float a, m;
  int t;
};

// Issues the colour loads of the tap at column qx.  For kInside x' lies
// inside the image.  Otherwise x' outside [0, W), NaN included, is not the
// unsigned minimum of the bits (sz is never -0, so x' is not) and reads the
// last texel instead: every lane loads, none branches; m is 1 - 2^127 |x' -
// its minimum|, clamped to [0, 1]: 1 for a difference of 0, else 0 (the
// difference is then at least half a unit of x' near W; a NaN clamps to 0).
// The fence keeps the loads ahead of the work that follows in the source,
// kPlace keeps the compiler from merging the loads of two places into one.
template <int kPlace, bool kInside>
__device__ __forceinline__ void cost_fetch(const Lane& L, CostTap* t,
                                           const char* __restrict__ crow,
                                           float sx, float rowb, float sz,
                                           float qx, float big) {
  float xc = fmaf(sx, qx, rowb) + sz;
  t->m = 1.0f;
  if (!kInside) {
    const float xq = xc;
    xc = __uint_as_float(
        min(__float_as_uint(xq), __float_as_uint(L.Wf) - 1u));
    t->m =
        __builtin_amdgcn_fmed3f(fmaf(-fabsf(xq - xc), big, 1.0f), 0.0f, 1.0f);
  }
  if (L.edge) {
    asm volatile("");  // stays a scalar branch
    t->m = qx >= 0.0f && qx < L.Wf ? t->m : 0.0f;
  }
  t->a = __builtin_amdgcn_fractf(xc);
  t->t = (int)xc;
  const uint32_t off = __umul24((uint32_t)t->t, 12u);
  const float4 u = load16(crow + off);
  const float2 v = load8b(crow + off + 16u);
  t->c0 = Rgb{u.x, u.y, u.z};
  t->c1 = Rgb{u.w, v.x, v.y};
  asm volatile("; tap loads, place %0" : : "i"(kPlace) : "memory");
}

// The 2 R + 1 taps of one patch row for a cost: fetch(place, tap, column),
// use(tap, index), the loads of a tap issued while the one before is used.
// For rows that are not inside the taps follow each other.
template <bool kInside, typename Use>
__device__ __forceinline__ void cost_row(const Lane& L,
                                         const char* __restrict__ crow,
                                         float sx, float rowb, float sz,
                                         float big, Use use) {
  const int R = L.R;
  float qx = L.xf - (float)R;
  CostTap p;
  if (kInside) {
    CostTap q;
    cost_fetch<0, true>(L, &p, crow, sx, rowb, sz, qx, big);
    for (int i = 0; i < 2 * R; i += 2) {
      cost_fetch<1, true>(L, &q, crow, sx, rowb, sz, qx + 1.0f, big);
      use(p, i);
      qx += 2.0f;
      cost_fetch<2, true>(L, &p, crow, sx, rowb, sz, qx, big);
      use(q, i + 1);
    }
    use(p, 2 * R);
  } else {
    for (int i = 0; i <= 2 * R; ++i, qx += 1.0f) {
      cost_fetch<3, false>(L, &p, crow, sx, rowb, sz, qx, big);
      use(p, i);
    }
  }
}

// patch_eval_color_grad_weighted on tame images: cost_eval_cg's sums.  A
// tap that does not count gets weight 0, which leaves both sums as they
// are.
__device__ __forceinline__ float cost_cg_tame(const Lane& L, float4 s,
                                              bool active) {
  active = active && L.valid;
  if (!__any(active)) return 0.0f;
  const int R = L.R;
  const float big = vconst(0x1p127f), negw = vconst(-L.kw);
  // idle lanes sample a column that is inside
  const float sx = active ? s.x : 0.0f, sy = active ? s.y : 0.0f;
  const float sz = active ? s.z + 0.0f : L.safe;
  const int y0 = max(-R, -L.y), y1 = min(R, L.H - 1 - L.y);
  float ret = 0.0f, wsum = 0.0f;
  for (int dy = y0; dy <= y1; ++dy) {
    const int qy = L.y + dy;  // uniform
    const float rowb = sy * (float)qy;
    const char* __restrict__ crow = colour_row(L, qy);
    const char* __restrict__ grow = gradient_row(L, qy);
    const LdsRow trow = L.trow0 + (dy + R) * L.TW;
    const LdsRow wrow = L.wrow0 + (dy + R) * L.wstride;
    auto use = [&](auto inside, const CostTap& t, int i) {
      constexpr bool kIn = decltype(inside)::value;
      float4 G[2];
      window_gradients<2, kIn>(L, wrow, grow, t.t, t.m > 0.0f, G);
      const float4 t1 = lds_at(trow, i);
      const float4 g1 = lds_at(trow, L.GT + i);
      const float w = t.m * weight_tame(t1.x - L.tc.x, t1.y - L.tc.y,
                                        t1.z - L.tc.z, negw);
      const Rgb s2 = lerp_rgb(t.c0, t.c1, t.a);
      const float4 d2 = lerp4(G[0], G[1], t.a);
      const float sc = (fminf(fabsf(t1.x - s2.r), 0.05f) +
                        fminf(fabsf(t1.y - s2.g), 0.05f)) +
                       fminf(fabsf(t1.z - s2.b), 0.05f);
      const float sg = ((fminf(fabsf(g1.x - d2.x), 0.05f) +
                         fminf(fabsf(g1.y - d2.y), 0.05f)) +
                        fminf(fabsf(g1.z - d2.z), 0.05f)) +
                       fminf(fabsf(g1.w - d2.w), 0.05f);
      const float C = fmaf(0.05f, sc, (1.0f - 0.05f) * sg);
      wsum += w;
      ret = fmaf(w, C, ret);
    };
    if (row_inside(L, sx, rowb, sz, L.xf - (float)R))
      cost_row<true>(L, crow, sx, rowb, sz, big,
                     [&](const CostTap& t, int i) { use(Yes(), t, i); });
    else
      cost_row<false>(L, crow, sx, rowb, sz, big,
                      [&](const CostTap& t, int i) { use(No(), t, i); });
  }
  return ret / wsum;
}

// patch_eval_census on tame images: cost_eval's sums and row-wise exit.  The
// exact exit test divides; the product decides most rows: census < 0.999999
// bilw mincost implies census / bilw < mincost.
__device__ __forceinline__ float cost_census_tame(const Lane& L, float4 s,
                                                  float mincost, bool active,
                                                  float* quot) {
  const int R = L.R;
  bool live = active && L.valid;
  float res = 0.0f;
  if (live) {
    const float xp = transform(s, L.xf, L.yf);
    if (!(finite_f(s.x) && finite_f(s.y) && finite_f(s.z)) ||
        to_normal(s).z < kNormalZMin || xp < 0.0f || xp >= L.Wf) {
      res = 1e5f;
      live = false;
    }
  }
  if (!__any(live)) return res;
  const float big = vconst(0x1p127f);
  const float negw = vconst(-L.cw), twenty = vconst(20.0f);
  // idle lanes sample a column that is inside
  float sx = live ? s.x : 0.0f, sy = live ? s.y : 0.0f;
  float sz = live ? s.z + 0.0f : L.safe;
  const float below = 0.999999f * (L.bilw * mincost);
  const int y0 = max(-R, -L.y), y1 = min(R, L.H - 1 - L.y);
  float census = 0.0f, wsum = 0.0f;
  for (int dy = y0; dy <= y1; ++dy) {
    const int qy = L.y + dy;  // uniform
    const float rowb = sy * (float)qy;
    const char* __restrict__ crow = colour_row(L, qy);
    const char* __restrict__ grow = gradient_row(L, qy);
    const LdsRow trow = L.trow0 + (dy + R) * L.TW;
    const LdsRow wrow = L.wrow0 + (dy + R) * L.wstride;
    auto use = [&](auto inside, const CostTap& t, int i) {
      constexpr bool kIn = decltype(inside)::value;
      float4 G[2];
      window_gradients<2, kIn>(L, wrow, grow, t.t, t.m > 0.0f, G);
      const float4 t1 = lds_at(trow, i);
      const float w = t.m * weight_tame(t1.x - L.tc.x, t1.y - L.tc.y,
                                        t1.z - L.tc.z, negw);
      const Rgb s2 = lerp_rgb(t.c0, t.c1, t.a);
      const float4 d2 = lerp4(G[0], G[1], t.a);
      const float c0 = clamp20(s2.r - t1.x, twenty);
      const float c1 = clamp20(s2.g - t1.y, twenty);
      const float c2 = clamp20(s2.b - t1.z, twenty);
      const float cad = 0.33f * ((c0 + c1) + c2);
      const float cost =
          fmaf(0.02734375f, sign_mismatches8f(__float_as_uint(t1.w), d2),
               0.125f * cad);
      census = fmaf(w, cost, census);
      wsum += w;
    };
    if (row_inside(L, sx, rowb, sz, L.xf - (float)R))
      cost_row<true>(L, crow, sx, rowb, sz, big,
                     [&](const CostTap& t, int i) { use(Yes(), t, i); });
    else
      cost_row<false>(L, crow, sx, rowb, sz, big,
                      [&](const CostTap& t, int i) { use(No(), t, i); });
    if (live && !(census < below) && census / L.bilw >= mincost) {
      res = 1.0f;
      live = false;
      sx = sy = 0.0f;
      sz = L.safe;
    }
    if (!__any(live)) break;
  }
  if (live) res = (wsum <= 1.0f) ? 1.1f : census / wsum;
  if (quot) *quot = census / L.bilw;
  return res;
}

// one term of klt_pass_tame; k1 = w1 0.125 0.33, k2 = w1 0.875 / 32, the
// powers of two folded in (exact)
__device__ __forceinline__ float klt_term_tame(const Rgb& s, float4 grad,
                                               float v0, float v1, float v2,
                                               uint32_t ga, float k1, float k2,
                                               float twenty) {
  const float c0 = clamp20(s.r - v0, twenty);
  const float c1 = clamp20(s.g - v1, twenty);
  const float c2 = clamp20(s.b - v2, twenty);
  const float C = k1 * ((c0 + c1) + c2);
  return fmaf(k2, sign_mismatches8f(ga, grad), C);
}

__device__ float4 klt_solve(float4 s, const float (&J)[3], const float (&H)[6]);

// One KLT tap in flight: the colours of texels f - 1 .. f + 2, f =
// floor(xc), xc = x' clamped to [-1, W].
struct KltTap {
  Rgb c[4];
  float xc, fl;
  int f;
};

// x' clamped to [-1, W], NaN to W (med3 of a NaN is the minimum of the
// others); klt_pass_general explains the clamp.  kInside: x' needs none.
template <int kPlace, bool kInside>
__device__ __forceinline__ void klt_fetch(KltTap* t,
                                          const char* __restrict__ crow,
                                          float sx, float rowb, float sz,
                                          float px, float negW) {
  const float xq = fmaf(sx, px, rowb) + sz;
  t->xc = kInside ? xq : -__builtin_amdgcn_fmed3f(-xq, 1.0f, negW);
  t->fl = floorf(t->xc);
  t->f = (int)t->fl;
  // from the record of texel -2, the row's first pad
  const char* __restrict__ pad = crow - 12 * kTexPadL;
  const uint32_t off = __umul24((uint32_t)(t->f + (kTexPadL - 1)), 12u);
  const float4 u = load16(pad + off), v = load16(pad + off + 16u),
               w = load16(pad + off + 32u);
  t->c[0] = Rgb{u.x, u.y, u.z};
  t->c[1] = Rgb{u.w, v.x, v.y};
  t->c[2] = Rgb{v.z, v.w, w.x};
  t->c[3] = Rgb{w.y, w.z, w.w};
  asm volatile("; klt loads, place %0" : : "i"(kPlace) : "memory");
}

// patch_census_klt2 on tame images: klt_pass_general's sums.  dead: the
// plane is not finite and its candidate is known to be rejected, so only
// its being non-finite has to last; such a lane samples a column inside.
__device__ __forceinline__ float4 klt_pass_tame(const Lane& L, float4 s,
                                                bool dead) {
  const int R = L.R;
  dead = dead || !L.valid;
  const float sx = dead ? 0.0f : s.x, sy = dead ? 0.0f : s.y,
              sz = dead ? L.safe : s.z;
  float J[3] = {0.0f, 0.0f, 0.0f};
  float H[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  const float negw = vconst(-L.cw), twenty = vconst(20.0f);
  const float negW = vconst(-L.Wf);
  const int y0 = max(-R, -L.y), y1 = min(R, L.H - 1 - L.y);
  for (int dy = y0; dy <= y1; ++dy) {
    const int qy = L.y + dy;  // uniform
    const float py = (float)qy;
    const float rowb = sy * py;
    const char* __restrict__ crow = colour_row(L, qy);
    const char* __restrict__ grow = gradient_row(L, qy);
    const LdsRow trow = L.trow0 + (dy + R) * L.TW;
    const LdsRow wrow = L.wrow0 + (dy + R) * L.wstride;
    float px = L.xf - (float)R;
    // the tap at column px of the row
    auto use = [&](auto inside, const KltTap& t, float px, int i) {
      constexpr bool kIn = decltype(inside)::value;
      float4 G[4];
      window_gradients<4, kIn>(L, wrow, grow, t.f - 1, !dead, G);
      const float4 t1 = lds_at(trow, i);
      const float v0 = t1.x - L.tc.x, v1 = t1.y - L.tc.y, v2 = t1.z - L.tc.z;
      const uint32_t ga = __float_as_uint(t1.w);
      float w1 = weight_tame(v0, v1, v2, negw);
      if (L.edge) {
        asm volatile("");  // stays a scalar branch
        w1 = px >= 1.0f && px < L.Wf - 1.0f ? w1 : 0.0f;
      }
      const float k1 = w1 * (0.125f * 0.33f), k2 = w1 * 0.02734375f;
      const float a = t.xc - t.fl;
      // floor(xc + 1) is floor(xc) + 1 unless the sum rounds up to floor(xc)
      // + 2: then the sample is the last texel
      const float ap = (t.xc + 1.0f) - (t.fl + 1.0f);
      const float4 gm = lerp4(G[0], G[1], a), g0 = lerp4(G[1], G[2], a);
      float4 gp = lerp4(G[2], G[3], ap);
      const Rgb cm = lerp_rgb(t.c[0], t.c[1], a);
      const Rgb c0 = lerp_rgb(t.c[1], t.c[2], a);
      Rgb cp = lerp_rgb(t.c[2], t.c[3], ap);
      if (__builtin_expect(__any(ap >= 1.0f), 0)) {
        asm volatile("");  // stays a scalar branch
        if (ap >= 1.0f) {
          cp = t.c[3];
          gp = G[3];
        }
      }
      const float C = klt_term_tame(c0, g0, v0, v1, v2, ga, k1, k2, twenty);
      const float Cxp = klt_term_tame(cp, gp, v0, v1, v2, ga, k1, k2, twenty);
      const float Cxm = klt_term_tame(cm, gm, v0, v1, v2, ga, k1, k2, twenty);
      const float curv = fmaf(-2.0f, C, Cxp + Cxm);
      if (curv > 0.0f) {
        const float gj = (w1 * (Cxm - Cxp)) * 0.5f;
        J[0] = fmaf(gj, px, J[0]);
        J[1] = fmaf(gj, py, J[1]);
        J[2] = J[2] + gj;
        const float h = w1 * curv;
        H[0] = H[0] + h * (px * px);
        H[1] = H[1] + h * (px * py);
        H[2] = H[2] + h * px;
        H[3] = H[3] + h * (py * py);
        H[4] = H[4] + h * py;
        H[5] = H[5] + h;
      }
    };
    KltTap p;
    if (row_inside(L, sx, rowb, sz, px)) {
      // loads one tap ahead
      KltTap q;
      klt_fetch<0, true>(&p, crow, sx, rowb, sz, px, negW);
      for (int i = 0; i < 2 * R; i += 2) {
        klt_fetch<1, true>(&q, crow, sx, rowb, sz, px + 1.0f, negW);
        use(Yes(), p, px, i);
        px += 2.0f;
        klt_fetch<2, true>(&p, crow, sx, rowb, sz, px, negW);
        use(Yes(), q, px - 1.0f, i + 1);
      }
      use(Yes(), p, px, 2 * R);
    } else {
      for (int i = 0; i <= 2 * R; ++i, px += 1.0f) {
        klt_fetch<3, false>(&p, crow, sx, rowb, sz, px, negW);
        use(No(), p, px, i);
      }
    }
  }
  return klt_solve(s, J, H);
}

// ---------------------------------------------------------------------
// patch_eval_census (pmhstereo.cl:661-736), one plane per lane (lanes with
// active == false idle), patch rows wave-uniform.  The reference tests
// census/bilw >= mincost after every tap; the census terms are >= 0 and
// accumulate monotonically, so testing at the end of each row returns 1.0
// exactly when the per-tap test would.
// quot (optional): the whole sum over bilw, what the exit compares.
// kCount: count the taps the reference's per-tap test evaluates (the
// algorithmic work; used by an untimed counting pass only).
// ---------------------------------------------------------------------
template <bool kCount>
__device__ __forceinline__ float cost_eval(const Lane& L, float4 s,
                                           float mincost, bool active,
                                           uint32_t* ntaps,
                                           float* quot = nullptr) {
  const int R = L.R, W = L.W;
  bool live = active && L.valid;
  float res = 0.0f;
  if (live) {
    const float xp = transform(s, L.xf, L.yf);
    if (!(finite_f(s.x) && finite_f(s.y) && finite_f(s.z)) ||
        to_normal(s).z < kNormalZMin || xp < 0.0f || xp >= L.Wf) {
      res = 1e5f;
      live = false;
    }
  }
  const int dx0 = max(-R, -L.x), dx1 = min(R, W - 1 - L.x);
  float census = 0.0f, wsum = 0.0f;
  for (int dy = -R; dy <= R; ++dy) {
    if (!__any(live)) break;
    const int qy = L.y + dy;  // uniform
    if (qy < 0 || qy >= L.H) continue;
    if (!live) continue;
    const float rowb = s.y * (float)qy;  // transform(), b y per row
    const float4* __restrict__ srow = L.tex2 + (size_t)qy * L.TS;
    const LdsRow trow = L.trow0 + (dy + R) * L.TW + R;
    // tap column as a float, stepped by 1 (exact below 2^24)
    float qx = L.xf + (float)dx0;
    for (int dx = dx0; dx <= dx1; ++dx, qx += 1.0f) {
      const float xq = fmaf(s.x, qx, rowb) + s.z;
      if (xq < 0.0f || xq >= L.Wf) continue;
      const float4 t1 = lds_at(trow, dx);
      const uint32_t m1 = __float_as_uint(t1.w);
      const float w = support_weight(t1.x - L.tc.x, t1.y - L.tc.y,
                                     t1.z - L.tc.z, L.cw);
      // 0 <= xq < W: no coordinate clamp; the second texel of xq in
      // [W-1, W) is the right edge pad, a copy of texel W-1
      const float fq = floorf(xq);
      const float4* __restrict__ tq = srow + (int)fq;
      const Sample s2 =
          lerp_texels(texel_at(tq, L.GP), texel_at(tq + 1, L.GP), xq - fq);
      const float c0 = fminf(fabsf(s2.r - t1.x), 0.05f) * 20.0f;
      const float c1 = fminf(fabsf(s2.g - t1.y), 0.05f) * 20.0f;
      const float c2 = fminf(fabsf(s2.b - t1.z), 0.05f) * 20.0f;
      const float cad = 0.33f * ((c0 + c1) + c2);
      // cost = 0.125 cad, then cost += 0.875 * (0.25 n): both products
      // are exact, so one fma with 0.21875 n = (7/256) (8 n) rounds the
      // same sum
      const float cost = fmaf(0.02734375f,
                              (float)sign_mismatches8(m1, s2.grad),
                              0.125f * cad);
      census = fmaf(w, cost, census);
      wsum += w;
      if (kCount) {
        ++*ntaps;
        if (census / L.bilw >= mincost) break;
      }
    }
    if (census / L.bilw >= mincost) {
      res = 1.0f;
      live = false;
    }
  }
  if (live) res = (wsum <= 1.0f) ? 1.1f : census / wsum;
  if (quot) *quot = census / L.bilw;
  return res;
}

// patch_eval_color_grad_weighted (pmhstereo.cl:510-565), one plane per lane
// (lanes with active == false idle), patch rows wave-uniform:
// w = exp(-|dot(I1(p) - I1(q), gray)| * kw), C = 0.05 sum_3 min(|I1(q) -
// I2(x')|, 0.05) + 0.95 sum_4 min(|G1(q) - G2(x')|, 0.05), result
// sum(w C) / sum(w).  No early exit and no invalid-plane test: a tap counts
// when its own pixel is in the image and x' lies in [0, W) (a non-finite x'
// fails the test; the reference samples at it, which OpenCL leaves
// undefined).  No qualifying tap gives 0 / 0 = NaN, which the accept rule
// never takes.  Needs the gradient tile (block_setup<true>).
// kCount: count the taps evaluated.
template <bool kCount>
__device__ float cost_eval_cg(const Lane& L, float4 s, bool active,
                              uint32_t* ntaps) {
  const int R = L.R, W = L.W;
  const bool live = active && L.valid;
  const int dx0 = max(-R, -L.x), dx1 = min(R, W - 1 - L.x);
  float ret = 0.0f, wsum = 0.0f;
  for (int dy = -R; dy <= R; ++dy) {
    if (!__any(live)) break;
    const int qy = L.y + dy;  // uniform
    if (qy < 0 || qy >= L.H) continue;
    if (!live) continue;
    const float rowb = s.y * (float)qy;  // transform(), b y per row
    const float4* __restrict__ srow = L.tex2 + (size_t)qy * L.TS;
    const LdsRow trow = L.trow0 + (dy + R) * L.TW + R;
    const LdsRow grow = trow + L.GT;
    float qx = L.xf + (float)dx0;
    for (int dx = dx0; dx <= dx1; ++dx, qx += 1.0f) {
      const float xq = fmaf(s.x, qx, rowb) + s.z;
      if (!(xq >= 0.0f && xq < L.Wf)) continue;
      const float4 t1 = lds_at(trow, dx);
      const float4 g1 = lds_at(grow, dx);
      // dot(valcenter - val1, gray): the negated difference gives the
      // negated dot bit for bit, so |.| is the same
      const float w = support_weight(t1.x - L.tc.x, t1.y - L.tc.y,
                                     t1.z - L.tc.z, L.kw);
      const float fq = floorf(xq);
      const float4* __restrict__ tq = srow + (int)fq;
      const Sample s2 =
          lerp_texels(texel_at(tq, L.GP), texel_at(tq + 1, L.GP), xq - fq);
      const float sc = (fminf(fabsf(t1.x - s2.r), 0.05f) +
                        fminf(fabsf(t1.y - s2.g), 0.05f)) +
                       fminf(fabsf(t1.z - s2.b), 0.05f);
      const float sg = ((fminf(fabsf(g1.x - s2.grad.x), 0.05f) +
                         fminf(fabsf(g1.y - s2.grad.y), 0.05f)) +
                        fminf(fabsf(g1.z - s2.grad.z), 0.05f)) +
                       fminf(fabsf(g1.w - s2.grad.w), 0.05f);
      // alpha dot(.) + (1 - alpha) dot(.), the left product fused
      const float C = fmaf(0.05f, sc, (1.0f - 0.05f) * sg);
      wsum += w;
      ret = fmaf(w, C, ret);
      if (kCount) ++*ntaps;
    }
  }
  return ret / wsum;
}

// ---------------------------------------------------------------------
// Teams.  A small image has fewer pixels than the GPU needs lanes: 320 x 240
// is 1200 wavefronts for 1024 SIMDs, and a wavefront alone on its SIMD waits
// for every load and for every instruction before the next.  There four lanes
// (a quad) share a pixel: each takes every fourth tap of a patch row and
// forms the tap's terms, then all four add the quad's terms up in the order
// of the taps, each lane's broadcast by DPP, so that every lane holds the
// sums and the bits are those of one lane's.  A tap that does not count has
// terms of -0, which leave any sum as it is.
// Three iterations of 320 x 240, R = 5: 4.85 -> 3.01 ms; 451 x 333, R = 7,
// red-black: 17.8 -> 12.4.  Tried on top: the wide tile's window of gradients
// in LDS (3.12; 16.9, for the work-groups it keeps off a CU), one image row
// per work-group (no difference), all nine KLT sums in every lane (3.17;
// 13.0).
// ---------------------------------------------------------------------
constexpr int kTeamLanes = 4;

template <int kLane>
__device__ __forceinline__ float quad_lane(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v),
                                                 0x55 * kLane, 0xf, 0xf, true));
}

// add(term a, term b, tap of the quad) for the quad's four taps in order
template <typename Add>
__device__ __forceinline__ void quad_sum(float a, float b, Add add) {
  add(quad_lane<0>(a), quad_lane<0>(b), 0);
  add(quad_lane<1>(a), quad_lane<1>(b), 1);
  add(quad_lane<2>(a), quad_lane<2>(b), 2);
  add(quad_lane<3>(a), quad_lane<3>(b), 3);
}

// cost_eval and cost_eval_cg by a team; kTame: see "Tame images"
template <int kKind, bool kTame>
__device__ __forceinline__ float cost_team(const Lane& L, float4 s,
                                           float mincost, bool active,
                                           float* quot) {
  constexpr bool kGrad = kKind == kCostColorGrad;
  const int R = L.R, W = L.W;
  bool live = active && L.valid;
  float res = 0.0f;
  if (!kGrad && live) {
    const float xp = transform(s, L.xf, L.yf);
    if (!(finite_f(s.x) && finite_f(s.y) && finite_f(s.z)) ||
        to_normal(s).z < kNormalZMin || xp < 0.0f || xp >= L.Wf) {
      res = 1e5f;
      live = false;
    }
  }
  const float cw = kGrad ? L.kw : L.cw;
  const float negw = vconst(-cw), twenty = vconst(20.0f);
  float sum = 0.0f, wsum = 0.0f;
  for (int dy = -R; dy <= R; ++dy) {
    if (!__any(live)) break;
    const int qy = L.y + dy;  // uniform
    if (qy < 0 || qy >= L.H) continue;
    if (!live) continue;
    const float rowb = s.y * (float)qy;  // transform(), b y per row
    const float4* __restrict__ srow = L.tex2 + (size_t)qy * L.TS;
    const LdsRow trow = L.trow0 + (dy + R) * L.TW;
    for (int i0 = 0; i0 <= 2 * R; i0 += kTeamLanes) {
      const int i = i0 + L.sub, x = L.x + i - R;
      const float xq = fmaf(s.x, (float)x, rowb) + s.z;
      float w = -0.0f, C = 0.0f;
      if (i <= 2 * R && x >= 0 && x < W && xq >= 0.0f && xq < L.Wf) {
        const float4 t1 = lds_at(trow, i);
        const float dr = t1.x - L.tc.x, dg = t1.y - L.tc.y,
                    db = t1.z - L.tc.z;
        w = kTame ? weight_tame(dr, dg, db, negw)
                  : support_weight(dr, dg, db, cw);
        const float fq = floorf(xq);
        const float4* __restrict__ tq = srow + (int)fq;
        const Sample s2 =
            lerp_texels(texel_at(tq, L.GP), texel_at(tq + 1, L.GP), xq - fq);
        if (kGrad) {
          const float4 g1 = lds_at(trow, L.GT + i);
          const float sc = (fminf(fabsf(t1.x - s2.r), 0.05f) +
                            fminf(fabsf(t1.y - s2.g), 0.05f)) +
                           fminf(fabsf(t1.z - s2.b), 0.05f);
          const float sg = ((fminf(fabsf(g1.x - s2.grad.x), 0.05f) +
                             fminf(fabsf(g1.y - s2.grad.y), 0.05f)) +
                            fminf(fabsf(g1.z - s2.grad.z), 0.05f)) +
                           fminf(fabsf(g1.w - s2.grad.w), 0.05f);
          C = fmaf(0.05f, sc, (1.0f - 0.05f) * sg);
        } else {
          const uint32_t m1 = __float_as_uint(t1.w);
          float c0, c1, c2, n;
          if (kTame) {
            c0 = clamp20(s2.r - t1.x, twenty);
            c1 = clamp20(s2.g - t1.y, twenty);
            c2 = clamp20(s2.b - t1.z, twenty);
            n = sign_mismatches8f(m1, s2.grad);
          } else {
            c0 = fminf(fabsf(s2.r - t1.x), 0.05f) * 20.0f;
            c1 = fminf(fabsf(s2.g - t1.y), 0.05f) * 20.0f;
            c2 = fminf(fabsf(s2.b - t1.z), 0.05f) * 20.0f;
            n = (float)sign_mismatches8(m1, s2.grad);
          }
          C = fmaf(0.02734375f, n, 0.125f * (0.33f * ((c0 + c1) + c2)));
        }
      }
      quad_sum(w, C, [&](float wj, float Cj, int) {
        sum = fmaf(wj, Cj, sum);
        wsum += wj;
      });
    }
    if (!kGrad && sum / L.bilw >= mincost) {
      res = 1.0f;
      live = false;
    }
  }
  if (kGrad) return sum / wsum;
  if (live) res = (wsum <= 1.0f) ? 1.1f : sum / wsum;
  if (quot) *quot = sum / L.bilw;
  return res;
}

// the candidate cost the kernels' patch_eval selects
template <int kKind, bool kCount, bool kWin = false, int kTeam = 1>
__device__ __forceinline__ float cost_any(const Lane& L, float4 s,
                                          float mincost, bool active,
                                          uint32_t* ntaps,
                                          float* quot = nullptr) {
  if (kTeam > 1)
    return L.tame ? cost_team<kKind, true>(L, s, mincost, active, quot)
                  : cost_team<kKind, false>(L, s, mincost, active, quot);
  // the counting pass takes the general loops, which count
  const bool tame = kWin && !kCount && L.tame;  // uniform
  if (kKind == kCostColorGrad)
    return tame ? cost_cg_tame(L, s, active)
                : cost_eval_cg<kCount>(L, s, active, ntaps);
  return tame ? cost_census_tame(L, s, mincost, active, quot)
              : cost_eval<kCount>(L, s, mincost, active, ntaps, quot);
}

// one census term of patch_census_klt2 (pmhstereo.cl:360-392); v0..v2 is
// the centred colour I1(q) - I1(p) the reference compares against;
// k1 = (w1 * alpha) * 0.33, k2 = w1 * (1 - alpha)
__device__ __forceinline__ float klt_term(const Sample& s, float v0, float v1,
                                          float v2, uint32_t ga, float k1,
                                          float k2) {
  const float c0 = fminf(fabsf(s.r - v0), 0.05f) * 20.0f;
  const float c1 = fminf(fabsf(s.g - v1), 0.05f) * 20.0f;
  const float c2 = fminf(fabsf(s.b - v2), 0.05f) * 20.0f;
  const float C = k1 * ((c0 + c1) + c2);
  // C += w1 * (1 - alpha) * 0.25 * n, 0.25 a double literal
  // (pmhstereo.cl:370): 0.25 n = 0.03125 (8 n) is exact, one rounding
  return fmaf(k2, 0.03125f * (float)sign_mismatches8(ga, s.grad), C);
}

// patch_census_klt2 (pmhstereo.cl:326-410) + mat3f_lusolve
// (cvt/cl/kernel/Matrix3.cl:286-311), one plane per lane
__device__ float4 klt_pass_general(const Lane& L, float4 s) {
  const int R = L.R, W = L.W;
  float J0 = 0.0f, J1 = 0.0f, J2 = 0.0f;
  float H00 = 0.0f, H01 = 0.0f, H02 = 0.0f, H11 = 0.0f, H12 = 0.0f,
        H22 = 0.0f;
  // taps need 1 <= x+dx < W-1 (the test is on the tap, pmhstereo.cl:358)
  const int dx0 = max(-R, 1 - L.x), dx1 = min(R, W - 2 - L.x);
  if (L.valid) {
    for (int dy = -R; dy <= R; ++dy) {
      const int qy = L.y + dy;  // uniform
      if (qy < 0 || qy >= L.H) continue;
      const float py = (float)qy;
      const float rowb = s.y * py;  // transform(), b y per row
      const float4* __restrict__ srow = L.tex2 + (size_t)qy * L.TS;
      const LdsRow trow = L.trow0 + (dy + R) * L.TW + R;
      // texel window srow[kf - 1 .. kf + 2] of the previous tap; a slope
      // near 1 slides it by one texel per tap
      int kf = INT_MIN;
      Texel tw0, tw1, tw2, tw3;
      float px = L.xf + (float)dx0;  // stepped by 1, exact below 2^24
      for (int dx = dx0; dx <= dx1; ++dx, px += 1.0f) {
        const float4 t1 = lds_at(trow, dx);
        const float v0 = t1.x - L.tc.x, v1 = t1.y - L.tc.y,
                    v2 = t1.z - L.tc.z;
        const uint32_t ga = __float_as_uint(t1.w);
        const float w1 = support_weight(v0, v1, v2, L.cw);
        const float k1 = (w1 * 0.125f) * 0.33f, k2 = w1 * 0.875f;
        const float xq = fmaf(s.x, px, rowb) + s.z;
        // The samples at x'-1, x' and x'+1 read the four texels from
        // floor(xc)-1 on, xc = x' clamped to [-1, W] (a NaN x' clamps to W):
        //  - x'-1 is exact for x' >= 0.5 and shares the floor and fraction
        //    of x'; below that it and its neighbour both read texel 0 (the
        //    left pads), whatever the fraction;
        //  - past either edge every texel involved is a copy of the edge
        //    texel, which is what the clamped sampler returns;
        //  - x'+1 is rounded and has its own fraction; its floor is
        //    floor(xc)+1, or floor(xc)+2 when the sum rounded up to the
        //    next integer (xc < W, so texel floor(xc)+3 is at most the
        //    last right pad).
        const float xc = fmaxf(fminf(xq, L.Wf), -1.0f);
        const float xp1 = xc + 1.0f;
        const float fl = floorf(xc);
        const float flp = floorf(xp1);
        const float a = xc - fl;
        const float ap = xp1 - flp;
        const int f = (int)fl;  // -1 <= f <= W
        if (f != kf) {
          if (f == kf + 1) {
            tw0 = tw1;
            tw1 = tw2;
            tw2 = tw3;
          } else {
            tw0 = texel_at(srow + (f - 1), L.GP);
            tw1 = texel_at(srow + f, L.GP);
            tw2 = texel_at(srow + (f + 1), L.GP);
          }
          tw3 = texel_at(srow + (f + 2), L.GP);
          kf = f;
        }
        const Sample sm = lerp_texels(tw0, tw1, a);
        const Sample s0 = lerp_texels(tw1, tw2, a);
        Sample sp = lerp_texels(tw2, tw3, ap);
        if (flp != fl + 1.0f)
          sp = lerp_texels(tw3, texel_at(srow + (f + 3), L.GP), ap);
        const float C = klt_term(s0, v0, v1, v2, ga, k1, k2);
        const float Cxp = klt_term(sp, v0, v1, v2, ga, k1, k2);
        const float Cxm = klt_term(sm, v0, v1, v2, ga, k1, k2);
        // (Cxp + Cxm) - 2 C: the product is exact, so the fma rounds the
        // same difference
        const float curv = fmaf(-2.0f, C, Cxp + Cxm);
        if (curv > 0.0f) {
          // J = J + w1 (Cxm - Cxp) 0.5 p, the last product fused
          // (pmhstereo.cl:394)
          const float gj = (w1 * (Cxm - Cxp)) * 0.5f;
          J0 = fmaf(gj, px, J0);
          J1 = fmaf(gj, py, J1);
          J2 = J2 + gj;
          const float h = w1 * curv;
          H00 = H00 + h * (px * px);
          H01 = H01 + h * (px * py);
          H02 = H02 + h * (px * 1.0f);
          H11 = H11 + h * (py * py);
          H12 = H12 + h * (py * 1.0f);
          H22 = H22 + h * (1.0f * 1.0f);
        }
      }
    }
  }
  const float J[3] = {J0, J1, J2};
  const float H[6] = {H00, H01, H02, H11, H12, H22};
  return klt_solve(s, J, H);
}

// s - H^-1 J: LU without pivoting; H is symmetric (H10 = H01, ...)
__device__ float4 klt_solve(float4 s, const float (&J)[3],
                            const float (&H)[6]) {
  float m00 = H[0], m01 = H[1], m02 = H[2];
  float m10 = H[1], m11 = H[3], m12 = H[4];
  float m20 = H[2], m21 = H[4], m22 = H[5];
  m10 /= m00;
  m20 /= m00;
  // x -= a * b contracts to fma(-a, b, x); the built-in dot of two
  // components is fma(y0, y1, x0 * x1)
  m11 = fmaf(-m10, m01, m11);
  m12 = fmaf(-m10, m02, m12);
  m21 = fmaf(-m20, m01, m21);
  m22 = fmaf(-m20, m02, m22);
  m21 /= m11;
  m22 = fmaf(-m21, m12, m22);
  float b0 = J[0], b1 = J[1], b2 = J[2];
  b1 = fmaf(-m10, b0, b1);
  b2 -= fmaf(m21, b1, m20 * b0);
  const float r2 = b2 / m22;
  const float r1 = fmaf(-m12, r2, b1) / m11;
  const float r0 = (b0 - fmaf(m02, r2, m01 * r1)) / m00;
  return mk4(s.x - r0, s.y - r1, s.z - r2, s.w - 1e5f);
}

// klt_pass_general by a team.  The nine sums are spread over the quad: each
// lane keeps one of J, one of H00, H01, H02, H11 (A) and one of H12, H22 (B),
// its coefficients chosen by the constants u, v (c = u px + v, exact for u 0
// or 1).
template <bool kTame>
__device__ __forceinline__ float4 klt_team(const Lane& L, float4 s) {
  const int R = L.R, W = L.W;
  float J = 0.0f, A = 0.0f, B = 0.0f;
  const float negw = vconst(-L.cw), twenty = vconst(20.0f);
  const float ja = L.sub == 0 ? 1.0f : 0.0f;                // px | py | 1
  const float aa = L.sub == 3 ? 0.0f : 1.0f;                // px px px py
  const float ba = L.sub == 0 ? 1.0f : 0.0f;                // px py 1 py
  if (L.valid) {
    for (int dy = -R; dy <= R; ++dy) {
      const int qy = L.y + dy;  // uniform
      if (qy < 0 || qy >= L.H) continue;
      const float py = (float)qy;
      const float rowb = s.y * py;  // transform(), b y per row
      const float4* __restrict__ srow = L.tex2 + (size_t)qy * L.TS;
      const LdsRow trow = L.trow0 + (dy + R) * L.TW;
      const float jb = L.sub == 0 ? 0.0f : (L.sub == 1 ? py : 1.0f);
      const float ab = L.sub == 3 ? py : 0.0f;
      const float bb = L.sub == 0 ? 0.0f : (L.sub == 2 ? 1.0f : py);
      const float cB = L.sub == 0 ? py : 1.0f;              // py 1
      for (int i0 = 0; i0 <= 2 * R; i0 += kTeamLanes) {
        const int i = i0 + L.sub, x = L.x + i - R;
        float gj = -0.0f, h = -0.0f;
        if (i <= 2 * R && x >= 1 && x < W - 1) {
          const float xq = fmaf(s.x, (float)x, rowb) + s.z;
          const float xc = fmaxf(fminf(xq, L.Wf), -1.0f);
          const float xp1 = xc + 1.0f;
          const float fl = floorf(xc), flp = floorf(xp1);
          const float a = xc - fl, ap = xp1 - flp;
          const float4* __restrict__ tq = srow + (int)fl;
          const Texel tw0 = texel_at(tq - 1, L.GP), tw1 = texel_at(tq, L.GP),
                      tw2 = texel_at(tq + 1, L.GP),
                      tw3 = texel_at(tq + 2, L.GP);
          const Sample sm = lerp_texels(tw0, tw1, a);
          const Sample s0 = lerp_texels(tw1, tw2, a);
          Sample sp = lerp_texels(tw2, tw3, ap);
          if (flp != fl + 1.0f)
            sp = lerp_texels(tw3, texel_at(tq + 3, L.GP), ap);
          const float4 t1 = lds_at(trow, i);
          const float v0 = t1.x - L.tc.x, v1 = t1.y - L.tc.y,
                      v2 = t1.z - L.tc.z;
          const uint32_t ga = __float_as_uint(t1.w);
          const float w1 = kTame ? weight_tame(v0, v1, v2, negw)
                                 : support_weight(v0, v1, v2, L.cw);
          auto term = [&](const Sample& t) {
            if (kTame)
              return klt_term_tame(Rgb{t.r, t.g, t.b}, t.grad, v0, v1, v2, ga,
                                   w1 * (0.125f * 0.33f), w1 * 0.02734375f,
                                   twenty);
            return klt_term(t, v0, v1, v2, ga, (w1 * 0.125f) * 0.33f,
                            w1 * 0.875f);
          };
          const float C = term(s0), Cxp = term(sp), Cxm = term(sm);
          const float curv = fmaf(-2.0f, C, Cxp + Cxm);
          if (curv > 0.0f) {
            gj = (w1 * (Cxm - Cxp)) * 0.5f;
            h = w1 * curv;
          }
        }
        // a tap that counts has px >= 1; |px| keeps the others' terms -0
        const float px0 = L.xf + (float)(i0 - R);
        quad_sum(gj, h, [&](float g, float hj, int j) {
          const float px = fabsf(px0 + (float)j);
          J = fmaf(g, fmaf(px, ja, jb), J);
          A = A + hj * (fmaf(px, aa, ab) * fmaf(px, ba, bb));
          B = B + hj * cB;
        });
      }
    }
  }
  const float Js[3] = {quad_lane<0>(J), quad_lane<1>(J), quad_lane<2>(J)};
  const float Hs[6] = {quad_lane<0>(A), quad_lane<1>(A), quad_lane<2>(A),
                       quad_lane<3>(A), quad_lane<0>(B), quad_lane<1>(B)};
  return klt_solve(s, Js, Hs);
}

template <bool kWin, int kTeam>
__device__ __forceinline__ float4 klt_pass(const Lane& L, float4 s,
                                           bool dead) {
  if (kTeam > 1)
    return L.tame ? klt_team<true>(L, s) : klt_team<false>(L, s);
  return kWin && L.tame ? klt_pass_tame(L, s, dead) : klt_pass_general(L, s);
}

__device__ __forceinline__ bool finite_plane(float4 s) {
  return finite_f(s.x) && finite_f(s.y) && finite_f(s.z);
}

// ---------------------------------------------------------------------
// precompute: pmhstereo_bilateral_weight_to_alpha (pmhstereo.cl:1462-1498)
// and pmhstereo_gradxy (pmhstereo.cl:1549-1602) into one texel record,
// plus the gradient sign bits
// ---------------------------------------------------------------------
constexpr int kBX = 64, kBY = 4;  // simple per-pixel kernels

// whether a pixel keeps the image tame (see there): colours 0 or of a
// magnitude in [2^-60, lim], a finite alpha
__device__ __forceinline__ bool pixel_tame(float4 c, float lim) {
  const float v[3] = {c.x, c.y, c.z};
  bool ok = finite_f(c.w);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float m = fabsf(v[k]);
    ok = ok && ((m >= 0x1p-60f && m <= lim) || __float_as_uint(v[k]) == 0u);
  }
  return ok;
}

__device__ __forceinline__ void prepare_pixel(const float* __restrict__ img,
                                              int W, int H, int C, int stride,
                                              int R, float cw, float lim,
                                              float4* __restrict__ tex,
                                              uint8_t* __restrict__ sgn,
                                              int x, int y) {
  const size_t p = (size_t)y * W + x;
  const float4 c = fetch_rgba(img, C, stride, x, y);
  if (!pixel_tame(c, lim)) *wild_word(tex, tex_stride(W), H) = 1u;
  float wsum = 0.0f;
  for (int dy = -R; dy <= R; ++dy) {
    const int qy = y + dy;
    if (qy < 0 || qy >= H) continue;
    for (int dx = -R; dx <= R; ++dx) {
      const int qx = x + dx;
      if (qx < 0 || qx >= W) continue;
      const float4 q = fetch_rgba(img, C, stride, qx, qy);
      wsum += support_weight(q.x - c.x, q.y - c.y, q.z - c.z, cw);
    }
  }
  const float g = gray_at(img, W, H, C, stride, x, y);
  const float gxp = gray_at(img, W, H, C, stride, x + 1, y);
  const float gxm = gray_at(img, W, H, C, stride, x - 1, y);
  const float gyp = gray_at(img, W, H, C, stride, x, y + 1);
  const float gym = gray_at(img, W, H, C, stride, x, y - 1);
  const float4 grad = mk4(gxp - g, gyp - g, gxp - gxm, gyp - gym);
  const float4 col = mk4(c.x, c.y, c.z, wsum);
  const size_t gp = (size_t)tex_stride(W) * H;  // gradient plane offset
  float4* row = tex + (size_t)y * tex_stride(W) + kTexPadL;
  float* pc = packed_colours(tex, tex_stride(W), H) +
              ((size_t)y * tex_stride(W) + kTexPadL) * 3;
  row[x] = col;
  row[gp + x] = grad;
  pc[3 * x] = c.x;
  pc[3 * x + 1] = c.y;
  pc[3 * x + 2] = c.z;
  // edge pads: copies of the first and last texel of the row
  if (x == 0)
    for (int i = 1; i <= kTexPadL; ++i) {
      row[-i] = col;
      row[gp - i] = grad;
      pc[-3 * i] = c.x;
      pc[-3 * i + 1] = c.y;
      pc[-3 * i + 2] = c.z;
    }
  if (x == W - 1)
    for (int i = 1; i <= kTexPadR; ++i) {
      row[x + i] = col;
      row[gp + x + i] = grad;
      pc[3 * (x + i)] = c.x;
      pc[3 * (x + i) + 1] = c.y;
      pc[3 * (x + i) + 2] = c.z;
    }
  sgn[p] = (uint8_t)signmask4(grad);
}

__global__ void k_clear_wild(uint32_t* __restrict__ a,
                             uint32_t* __restrict__ b) {
  if (threadIdx.x == 0) *a = *b = 0u;
}

__global__ void k_costs_unknown(CostWords* cw, int view) {
  if (threadIdx.x == 0) cw->known[view] = 0u;
}

// The work-group that finishes last says that the field's costs are known.
// Every work-group has read the word by then, so all find the same.
__global__ void __launch_bounds__(256)
k_forget_costs(size_t npix, CostWords* cw, float4* __restrict__ left,
               float4* __restrict__ right) {
  const int view = blockIdx.y;
  if (cw->known[view]) return;
  float4* s = view ? right : left;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < npix;
       i += (size_t)gridDim.x * 256)
    s[i].w = NAN;
  __syncthreads();
  if (threadIdx.x != 0) return;
  if (atomicAdd(&cw->tickets[view], 1u) != gridDim.x - 1) return;
  cw->tickets[view] = 0u;
  cw->known[view] = 1u;
}

__global__ void __launch_bounds__(256)
k_prepare(const float* __restrict__ img, int W, int H, int C, int stride,
          int R, float cw, float lim, float4* __restrict__ tex,
          uint8_t* __restrict__ sgn) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  if (x >= W || y >= H) return;
  prepare_pixel(img, W, H, C, stride, R, cw, lim, tex, sgn, x, y);
}

// pmhstereo_init (pmhstereo.cl:755-773): RNG_init(p, 3), three draws; one
// tile block of 64 x kRows pixels, reached by every thread of the block
template <int kKind, int kRows>
__device__ __forceinline__ void init_block(const Geometry& g, ViewBufs self,
                                           ViewBufs other, float dmax, int lr,
                                           float4* __restrict__ states,
                                           float4* smem, int bx, int by) {
  const Lane L = block_setup_at<kKind == kCostColorGrad, false, kRows>(
      g, self, other, smem, bx * kTX, by * kRows, g.H);
  float4 s = mk4(0.0f, 0.0f, 0.0f, 0.0f);
  if (L.valid) {
    Mwc rng = mwc_jump((uint64_t)L.p * 3u);
    const float u0 = mwc_next(&rng), u1 = mwc_next(&rng), u2 = mwc_next(&rng);
    s = state_init(u0, u1, u2, L.xf, L.yf, lr, dmax);
  }
  const float w = cost_any<kKind, false>(L, s, 1e10f, true, nullptr);
  if (L.valid) {
    s.w = w;
    states[L.p] = s;
  }
}

template <int kKind>
__global__ void __launch_bounds__(256)
k_init(Geometry g, ViewBufs self, ViewBufs other, float dmax, int lr,
       float4* __restrict__ states) {
  extern __shared__ float4 smem[];
  int bx, by;
  xcd_block(&bx, &by);
  init_block<kKind, kTY>(g, self, other, dmax, lr, states, smem, bx, by);
}

// pmhstereo_disparity_to_normal (pmhstereo.cl:1604-1637)
__global__ void __launch_bounds__(256)
k_disparity_to_normal(int W, int H, const float* __restrict__ disp,
                      float4* __restrict__ normals) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  if (x >= W || y >= H) return;
  const size_t p = (size_t)y * W + x;
  const float d = disp[p];
  const float dxp = x + 1 < W ? disp[p + 1] : 0.0f;
  const float dyp = y + 1 < H ? disp[p + W] : 0.0f;
  const float dx = dxp - d, dy = dyp - d;
  float3 n = make_float3(0.0f * dy - dx * 1.0f, dx * 0.0f - 1.0f * dy,
                         1.0f * 1.0f - 0.0f * 0.0f);
  n = normalize3(n);
  normals[p] = mk4(n.x, n.y, n.z, 0.0f);
}

// pmhstereo_init_disparity_normal (pmhstereo.cl:802-828)
template <int kKind>
__global__ void __launch_bounds__(256)
k_init_prior(Geometry g, ViewBufs self, ViewBufs other, float dmax, int lr,
             const float* __restrict__ disp,
             const float4* __restrict__ normals, float4* __restrict__ states) {
  extern __shared__ float4 smem[];
  const Lane L = block_setup<kKind == kCostColorGrad>(g, self, other, smem);
  float4 s = mk4(0.0f, 0.0f, 0.0f, 0.0f);
  if (L.valid) {
    Mwc rng = mwc_jump((uint64_t)L.p * 3u);
    const float d = disp[L.p];
    if (d > 0.0f) {
      const float4 nn = normals[L.p];
      const float3 n = normalize3(make_float3(nn.x, nn.y, nn.z));
      s = from_disparity_normal(L.xf, L.yf, lr ? d : -d, n);
    } else {
      const float u0 = mwc_next(&rng), u1 = mwc_next(&rng),
                  u2 = mwc_next(&rng);
      s = state_init(u0, u1, u2, L.xf, L.yf, lr, dmax);
    }
  }
  const float w = cost_any<kKind, false>(L, s, 1e10f, true, nullptr);
  if (L.valid) {
    s.w = w;
    states[L.p] = s;
  }
}

// Init of a view from a plane proposal, with a per-pixel fallback: the
// proposed plane (disparity d = o.x * dscale and normal (o.y, o.z, o.w) at
// the pixel, from_disparity_normal as pmhstereo_init_disparity_normal
// builds it, pmhstereo.cl:802-828) competes with the random plane of
// pmhstereo_init (draws 3p..3p+2, pmhstereo.cl:755-773), and the random
// plane takes the pixel only when its cost is lower (a NaN cost never
// wins).  The right view's proposal (lr = 0) comes from the network's pass
// over the mirrored pair: it is read at column W - 1 - x, and its normal
// maps to (nx, -ny, nz) (the mirror flips the sign of the disparity's x
// slope, the right view's plane convention flips both slopes).  A
// non-finite or non-positive proposed disparity leaves the random plane.
template <int kKind>
__global__ void __launch_bounds__(256)
k_init_proposal(Geometry g, ViewBufs self, ViewBufs other, float dmax, int lr,
                const float* __restrict__ prop, int os, int Wp, float dscale,
                float4* __restrict__ states) {
  extern __shared__ float4 smem[];
  const Lane L = block_setup<kKind == kCostColorGrad>(g, self, other, smem);
  float4 q = mk4(0.0f, 0.0f, 0.0f, 0.0f), sp = q;
  bool have = false;
  if (L.valid) {
    Mwc rng = mwc_jump((uint64_t)L.p * 3u);
    const float u0 = mwc_next(&rng), u1 = mwc_next(&rng), u2 = mwc_next(&rng);
    q = state_init(u0, u1, u2, L.xf, L.yf, lr, dmax);
    const int xs = lr ? L.x : L.W - 1 - L.x;
    const float* o = prop + ((size_t)L.y * Wp + xs) * os;
    const float d = o[0] * dscale;
    float3 n = make_float3(o[1], lr ? o[2] : -o[2], o[3]);
    if (d > 0.0f && finite_f(d) && finite_f(n.x) && finite_f(n.y) &&
        finite_f(n.z)) {
      n = normalize3(n);
      sp = from_disparity_normal(L.xf, L.yf, lr ? d : -d, n);
      have = true;
    }
  }
  const float cq = cost_any<kKind, false>(L, q, 1e10f, true, nullptr);
  const float cp = cost_any<kKind, false>(L, sp, 1e10f, have, nullptr);
  if (L.valid) {
    q.w = cq;
    sp.w = cp;
    const bool keep = have && (cp <= cq || cq != cq);
    states[L.p] = keep ? sp : q;
  }
}

// The right view's start when only the left view is seeded
// (pm_setup_proposal_views, views = 1): at every pixel the nearest left
// surface the view scatter put there (slot key 0, the propagate's first
// view candidate, pmhstereo.cl:1007-1016) carried over by viewprop, else
// the random plane of pmhstereo_init (draws 3p..3p+2, pmhstereo.cl:
// 755-773).  No cost is evaluated: the cost channel is NaN, and every
// propagate re-costs its own planes before it uses them
// (pmhstereo.cl:940).
__global__ void __launch_bounds__(256)
k_init_from_view(int W, int H, float dmax,
                 const unsigned long long* __restrict__ slots,
                 const float4* __restrict__ src, float4* __restrict__ states) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  if (x >= W || y >= H) return;
  const size_t p = (size_t)y * W + x;
  const uint32_t k0 = (uint32_t)(slots[p] & 0xFFFFFFFFull);
  float4 s;
  if (k0 != kSlotEmpty) {
    // the left view's key is W - 1 - x (slot_insert's order: nearest first)
    s = viewprop(src[(size_t)y * W + (W - 1 - (int)k0)]);
  } else {
    Mwc rng = mwc_jump((uint64_t)p * 3u);
    const float u0 = mwc_next(&rng), u1 = mwc_next(&rng), u2 = mwc_next(&rng);
    s = state_init(u0, u1, u2, (float)x, (float)y, 0, dmax);
  }
  s.w = __int_as_float(0x7fc00000);
  states[p] = s;
}

__global__ void __launch_bounds__(256)
k_viewbuf_clear(size_t n, unsigned long long* __restrict__ vbuf,
                CostWords* cw) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) vbuf[i] = ~0ull;
  if (cw && i == 0) *cw = CostWords{{1u, 1u}, {0u, 0u}};
}

// ---------------------------------------------------------------------
// pmhstereo_propagate_view (pmhstereo.cl:880-1071), Jacobi schedule
// ---------------------------------------------------------------------
struct PropCtx {
  float dmax, theta;
  int lr;
  float4 smooth;
};

// a propagate's candidates by index: the view's own plane (re-costed), the
// smooth proposal, the random neighbours, the random plane, the other
// view's planes, the refinement, the KLT step
constexpr int kCandSelf = 0, kCandSmooth = 1, kCandNeighbour = 2,
              kCandRandom = kCandNeighbour + kNumRndSample,
              kCandView = kCandRandom + 1,
              kCandRefine = kCandView + kViewSamples,
              kCandidates = kCandRefine + 2;

// keep the two smallest keys of a slot: the two nearest surfaces win the
// view scatter, independent of the order of arrival (the reference's
// atomic_inc race, pmhstereo.cl:1057-1067, keeps an arbitrary two)
__device__ __forceinline__ void slot_insert(unsigned long long* slot,
                                            uint32_t key) {
  unsigned long long old = *reinterpret_cast<volatile unsigned long long*>(slot);
  while (true) {
    const uint32_t k0 = (uint32_t)(old & 0xFFFFFFFFull);
    const uint32_t k1 = (uint32_t)(old >> 32);
    unsigned long long nw;
    if (key < k0)
      nw = ((unsigned long long)k0 << 32) | key;
    else if (key < k1)
      nw = ((unsigned long long)key << 32) | k0;
    else
      return;
    const unsigned long long prev = atomicCAS(slot, old, nw);
    if (prev == old) return;
    old = prev;
  }
}

// view scatter of a final state (pmhstereo.cl:1060-1067): slot at
// rte(x') of the other view when the integer disparity is > 0
__device__ __forceinline__ void scatter(float4 self, int x, int y, int W,
                                        int lr,
                                        unsigned long long* viewout) {
  const float xf = (float)x, yf = (float)y;
  const float xs = transform(self, xf, yf);
  const float xr = rintf(xs);
  const float disp = (xs - xf) * (lr ? -1.0f : 1.0f);
  if (xr >= 0.0f && xr < (float)W && disp >= 1.0f) {
    const uint32_t key = (uint32_t)(lr ? W - 1 - x : x);
    slot_insert(&viewout[(size_t)y * W + (int)xr], key);
  }
}

// One tile block of pmhstereo_propagate_view: the pixels of the block
// (bx, by) of 64 x kRows tiles (kRB: of 128 x kRows, one colour).  Must be
// reached by every thread of the block.
// kCount: accumulate the cost taps (counters[0]) and KLT taps
// (counters[1]) this block evaluates; the results are identical.
// kRB: one pass of the red-black schedule (g.color); pass 1 reads the
// neighbours of colour 0 from a.fresh, the planes pass 0 just wrote.
// kTeam: lanes per pixel, all of which hold its planes and costs.
template <int kKind, bool kCount, bool kRB, int kRows, int kWX, bool kWin,
          int kTeam = 1>
__device__ __forceinline__ void propagate_block(
    const Geometry& g, const PropagateArgs& a, unsigned long long* counters,
    float4* smem, int x0, int y0, int row_end, Window win) {
  const Lane L =
      block_setup_at<kKind == kCostColorGrad, kRB, kRows, kWX, kWin, kTeam>(
          g, a.self, a.other, smem, x0, y0, row_end, win);
  if (!__any(L.valid)) return;  // no barrier follows
  const int W = g.W, H = g.H;
  uint32_t ncost = 0;
  uint32_t* nc = kCount ? &ncost : nullptr;
  PropCtx c;
  c.dmax = a.dmax;
  c.theta = a.theta;
  c.lr = a.lr;
  float4 sm = mk4(0.0f, 0.0f, 0.0f, 0.0f);
  float4 self = sm;
  if (L.valid) {
    if (a.smooth) sm = a.smooth[L.p];
    self = a.old[L.p];
  }
  sm.w = fminf(fmaxf(sm.w, 0.0f), 1.0f) * a.dmax;
  c.smooth = sm;

  Mwc rng = mwc_jump(prop_draw_start(L.p, a.iter));
  uint32_t keys[2] = {kSlotEmpty, kSlotEmpty};
  if (a.viewin && L.valid) {
    const unsigned long long slot = a.viewin[L.p];
    keys[0] = (uint32_t)(slot & 0xFFFFFFFFull);
    keys[1] = (uint32_t)(slot >> 32);
  }
  const bool plain = a.smooth == nullptr && c.theta == 0.0f;

  // The candidates in the reference's order, one rolled loop: the cost
  // loops are in the code once, not once per candidate.
  for (int k = 0; k < kCandidates; ++k) {
    asm volatile("" : "+s"(k));  // not unrolled or specialised by k
    float4 cand = self;
    bool active = L.valid;
    if (k == kCandSelf) {
      // The old plane's cost.  The cost channel holds it as an evaluation
      // without an early exit gives it, and only the values that do not
      // settle it are evaluated again: NaN (no cost yet, or a
      // colour+gradient patch without a tap) and the 1.0 of the census
      // early exit.
      if (!kCount) {
        active = active && (self.w != self.w ||
                            (kKind != kCostColorGrad && self.w == 1.0f));
        if (!__any(active)) continue;
      }
    } else if (k == kCandSmooth) {
      // smooth proposal (pmhstereo.cl:968-976)
      cand = from_disparity_normal(
          L.xf, L.yf, sm.w * (a.lr ? -1.0f : 1.0f),
          normalize3(make_float3(sm.x, sm.y, sm.z)));
      if (!a.lr) cand = viewprop(cand);
    } else if (k < kCandRandom) {
      // random neighbours (pmhstereo.cl:981-991), x offset drawn first
      const float ux = mwc_next(&rng);
      const float uy = mwc_next(&rng);
      const int ox = (int)fmaf((ux - 0.5f) * 2.0f, kRndSampleRadius, 0.5f);
      const int oy = (int)fmaf((uy - 0.5f) * 2.0f, kRndSampleRadius, 0.5f);
      if (L.valid) {
        const int nx = clampi(L.x + ox, 0, W - 1),
                  ny = clampi(L.y + oy, 0, H - 1);
        const float4* src = a.old;
        if (kRB && g.color == 1 && ((nx + ny) & 1) == 0) src = a.fresh;
        cand = src[(size_t)ny * W + nx];
      }
    } else if (k == kCandRandom || k == kCandRefine) {
      const float u0 = mwc_next(&rng), u1 = mwc_next(&rng),
                  u2 = mwc_next(&rng);
      // random plane (pmhstereo.cl:996-1002); randomized refinement
      // (pmhstereo.cl:1021-1028)
      if (k == kCandRandom)
        cand = state_init(u0, u1, u2, L.xf, L.yf, a.lr, a.dmax);
      else
        cand = state_refine(u0, u1, u2, self, L.xf, L.yf, a.dmax, a.lr);
    } else if (k < kCandRefine) {
      // other view (pmhstereo.cl:1007-1016)
      const uint32_t key = k == kCandView ? keys[0] : keys[1];
      active = active && keys[0] != kSlotEmpty && key != kSlotEmpty;
      if (active) {
        const int xs = a.lr ? (int)key : W - 1 - (int)key;
        cand = viewprop(a.src_other[(size_t)L.y * W + xs]);
      }
    } else {
      // KLT step (pmhstereo.cl:1034-1053).  A pass that meets a singular
      // system leaves a plane that is not finite, and so do the passes
      // after it.  Its cost is NaN (colour+gradient: no tap counts), which
      // is never accepted, or 1e5 (census), accepted only by a plane that
      // costs as much.
      bool sure = kKind == kCostColorGrad;
      if (kKind != kCostColorGrad) {
        float v = self.w;
        if (!plain)
          v = fmaf(c.theta,
                   smooth_dist(self, c.smooth, L.xf, L.yf, c.dmax, c.lr), v);
        sure = v < 9e4f;
      }
      for (int it = 0; it < kKltPasses; ++it) {
        const bool dead = sure && !finite_plane(cand);
        if (!__any(L.valid && !dead)) break;
        cand = klt_pass<kWin, kTeam>(L, cand, dead);
      }
    }
    // minimalCost (pmhstereo.cl:873-877).  With theta = 0 and no smooth
    // field it is the current cost, unless a distance is infinite or NaN,
    // which needs an |x'| whose square overflows.
    float ds = 0.0f, dc = 0.0f, mincost = 1e10f;
    if (k != kCandSelf) {
      mincost = self.w;
      const bool near =
          plain && fabsf(transform(cand, L.xf, L.yf)) < 1e15f &&
          fabsf(transform(self, L.xf, L.yf)) < 1e15f;
      if (__any(active && !near) && active) {
        ds = smooth_dist(self, c.smooth, L.xf, L.yf, c.dmax, c.lr);
        dc = smooth_dist(cand, c.smooth, L.xf, L.yf, c.dmax, c.lr);
        mincost = fmaf(-c.theta, dc, fmaf(c.theta, ds, self.w));
      }
    }
    // The smooth proposal of a cleared field is one plane for all iterations
    // of the call: costed in full by the first, kept for the others.  The
    // census exit returns 1.0 exactly when the whole sum reaches mincost
    // (the row sums only grow, and so do their quotients).
    const bool flat = !kCount && k == kCandSmooth && a.flat_cost;
    float w = 0.0f, q = 0.0f;
    if (!(flat && a.flat_known))
      w = cost_any<kKind, kCount, kWin, kTeam>(
          L, cand, flat ? 1e10f : mincost, active, nc, &q);
    if (flat && active) {
      float* fc = a.flat_cost + L.p * kFlatCosts;
      if (a.flat_known) {
        w = fc[0];
        if (kKind != kCostColorGrad) q = fc[1];
      } else {
        fc[0] = w;
        if (kKind != kCostColorGrad) fc[1] = q;
      }
      if (kKind != kCostColorGrad && w != 1e5f && q >= mincost) w = 1.0f;
    }
    if (active) {
      // the select rule (pmhstereo.cl:976)
      cand.w = w;
      if (k == kCandSelf ||
          fmaf(c.theta, dc, cand.w) <= fmaf(c.theta, ds, self.w))
        self = cand;
    }
  }
  if (!L.valid || L.sub) return;
  if (a.viewout) scatter(self, L.x, L.y, W, a.lr, a.viewout);
  a.out[L.p] = self;
  if (kCount) {
    // KLT taps: rows in the image times columns with 1 <= x+dx < W-1
    const int R = g.R;
    const int rows = min(R, H - 1 - L.y) - max(-R, -L.y) + 1;
    const int cols = min(R, W - 2 - L.x) - max(-R, 1 - L.x) + 1;
    const unsigned long long nklt =
        cols > 0 ? (unsigned long long)rows * cols * kKltPasses : 0ull;
    atomicAdd(&counters[0], (unsigned long long)ncost);
    atomicAdd(&counters[1], nklt);
  }
}

// The single-image launch: one tile block per work-group.  kEu: wavefronts
// per SIMD the kernel is built for (see saves_a_round).
template <int kKind, bool kCount, bool kRB, int kRows, int kWX, bool kWin,
          int kTeam, int kEu>
__global__ void __launch_bounds__(64 * kWX * kRows)
__attribute__((amdgpu_waves_per_eu(kEu, kEu)))
k_propagate(Geometry g, PropagateArgs a, unsigned long long* counters,
            Window win) {
  extern __shared__ float4 smem[];
  int bx, by;
  xcd_block(&bx, &by);
  const int row0 = g.band0 * kBandRows;
  propagate_block<kKind, kCount, kRB, kRows, kWX, kWin, kTeam>(
      g, a, counters, smem, bx * (kRB ? 2 : 1) * kTX * kWX / kTeam,
      row0 + by * kRows, g.row_end(), win);
}

// view scatter alone, from a stored field: rebuilds the buffer the field's
// last propagate left behind
__global__ void __launch_bounds__(256)
k_scatter(int W, int H, const float4* __restrict__ states, int lr,
          unsigned long long* __restrict__ viewout) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  if (x >= W || y >= H) return;
  scatter(states[(size_t)y * W + x], x, y, W, lr, viewout);
}

template <int kKind>
__global__ void __launch_bounds__(256)
k_cost_field(Geometry g, ViewBufs self, ViewBufs other,
             const float4* __restrict__ planes, float* __restrict__ cost) {
  extern __shared__ float4 smem[];
  const Lane L = block_setup<kKind == kCostColorGrad>(g, self, other, smem);
  const float4 s = L.valid ? planes[L.p] : mk4(0.0f, 0.0f, 0.0f, 0.0f);
  const float w = cost_any<kKind, false>(L, s, 1e10f, true, nullptr);
  if (L.valid) cost[L.p] = w;
}

__global__ void __launch_bounds__(256)
k_klt_field(Geometry g, ViewBufs self, ViewBufs other,
            const float4* __restrict__ planes, int passes,
            float4* __restrict__ out) {
  extern __shared__ float4 smem[];
  const Lane L = block_setup<false>(g, self, other, smem);
  float4 s = L.valid ? planes[L.p] : mk4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int i = 0; i < passes; ++i) s = klt_pass<false, 1>(L, s, false);
  if (L.valid) out[L.p] = s;
}

// pmhstereo_consistency (pmhstereo.cl:1095-1129) at pixel (x, y)
__device__ __forceinline__ void consistency_pixel(
    int W, const float4* __restrict__ left, const float4* __restrict__ right,
    float maxdispdiff, float maxdeg, float4* __restrict__ out, int x, int y) {
  const size_t p = (size_t)y * W + x;
  const float athr = maxdeg / 180.0f;
  const float4 sl = left[p];
  const float xf = (float)x, yf = (float)y;
  const float x2 = transform(sl, xf, yf);
  float4 val = mk4(0.0f, 0.0f, 0.0f, -1.0f);
  const float fl = floorf(x2), ce = ceilf(x2);
  if (ce >= 0.0f && fl < (float)W) {
    const int i0 = clampi((int)fl, 0, W - 1), i1 = clampi((int)ce, 0, W - 1);
    const float4 r1 = right[(size_t)y * W + i0];
    const float4 r2 = right[(size_t)y * W + i1];
    const float3 nl = to_normal(sl);
    const float3 n1 = to_normal(viewprop(r1));
    const float3 n2 = to_normal(viewprop(r2));
    const float nd1 = fmaf(nl.z, n1.z, fmaf(nl.y, n1.y, nl.x * n1.x));
    const float nd2 = fmaf(nl.z, n2.z, fmaf(nl.y, n2.y, nl.x * n2.x));
    const float dm1 = fabsf(xf - transform(r1, x2, yf));
    const float dm2 = fabsf(xf - transform(r2, x2, yf));
    const float a1 = acospi_f(fminf(fmaxf(nd1, -1.0f), 1.0f));
    const float a2 = acospi_f(fminf(fmaxf(nd2, -1.0f), 1.0f));
    if (!(dm1 >= maxdispdiff || a1 >= athr) ||
        !(dm2 >= maxdispdiff || a2 >= athr))
      val = sl;
  }
  out[p] = val;
}

__global__ void __launch_bounds__(256)
k_consistency(int W, int H, const float4* __restrict__ left,
              const float4* __restrict__ right, float maxdispdiff,
              float maxdeg, float4* __restrict__ out) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  if (x >= W || y >= H) return;
  consistency_pixel(W, left, right, maxdispdiff, maxdeg, out, x, y);
}

// pmhstereo_to_disparity (pmhstereo.cl:1232-1257) at pixel (x, y)
__device__ __forceinline__ void to_disparity_pixel(
    int W, const float4* __restrict__ states, float scale, int lr,
    float* __restrict__ disp, int x, int y) {
  const size_t p = (size_t)y * W + x;
  const float4 s = states[p];
  const float d = (transform(s, (float)x, (float)y) - (float)x) *
                  (lr ? -1.0f : 1.0f);
  float val;
  if (len3(s) < 1e-4f || d < 0.0f || d > (float)W)
    val = 0.0f;
  else
    val = fmaxf(d, 0.0f);
  disp[p] = val * scale;
}

__global__ void __launch_bounds__(256)
k_to_disparity(int W, int H, const float4* __restrict__ states, float scale,
               int lr, float* __restrict__ disp) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  if (x >= W || y >= H) return;
  to_disparity_pixel(W, states, scale, lr, disp, x, y);
}

// row scans of pmhstereo_fill_depthmap / pmhstereo_fill_normalmap
__device__ __forceinline__ void row_fill_pair(const float4* __restrict__ in,
                                              int W, int x, int y, float4* l,
                                              float4* r) {
  const float4* row = in + (size_t)y * W;
  float4 a = mk4(0.0f, 0.0f, 0.0f, 0.0f), b = a;
  for (int i = x - 1; len3(a) < 1e-1f && i >= 0; --i) a = row[i];
  for (int i = x + 1; len3(b) < 1e-1f && i < W; ++i) b = row[i];
  if (len3(a) < 1e-1f) a.x = a.y = a.z = -1e5f;
  if (len3(b) < 1e-1f) b.x = b.y = b.z = -1e5f;
  const float xf = (float)x, yf = (float)y;
  a.w = -(transform(a, xf, yf) - xf);
  b.w = -(transform(b, xf, yf) - xf);
  *l = a;
  *r = b;
}

// pmhstereo_fill_depthmap (pmhstereo.cl:1187-1230) at pixel (x, y)
__device__ __forceinline__ void fill_depthmap_pixel(
    int W, const float4* __restrict__ states, float scale,
    float* __restrict__ disp, int x, int y) {
  const size_t p = (size_t)y * W + x;
  const float4 s = states[p];
  float val;
  if (len3(s) < 1e-4f) {
    float4 l, r;
    row_fill_pair(states, W, x, y, &l, &r);
    val = fminf(l.w, r.w);
  } else {
    val = fabsf(transform(s, (float)x, (float)y) - (float)x);
  }
  disp[p] = val * scale;
}

__global__ void __launch_bounds__(256)
k_fill_depthmap(int W, int H, const float4* __restrict__ states, float scale,
                float* __restrict__ disp) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  if (x >= W || y >= H) return;
  fill_depthmap_pixel(W, states, scale, disp, x, y);
}

// pmhstereo_fill_normalmap (pmhstereo.cl:1259-1305)
__global__ void __launch_bounds__(256)
k_fill_normalmap(int W, int H, const float4* __restrict__ states,
                 float4* __restrict__ normals) {
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  if (x >= W || y >= H) return;
  const size_t p = (size_t)y * W + x;
  const float4 s = states[p];
  float3 n;
  if (len3(s) < 1e-1f) {
    float4 l, r;
    row_fill_pair(states, W, x, y, &l, &r);
    n = (l.w < r.w) ? to_normal(l) : to_normal(r);
  } else {
    n = to_normal(s);
  }
  normals[p] = mk4(n.x, n.y, n.z, 0.0f);
}

// Disparity::evaluateError (cvt/vision/Disparity.cpp:201-233) on the
// device: over the pixels with gt > 0, counts[2] += 1, counts[1] += 1 when
// the estimate is > 0, counts[0] += 1 when |gt - est| > abs_thres and
// |gt - est| / |gt| > rel_thres.  A block sums its pixels' counts, one
// atomic per counter.
// Called by every lane of the wavefront (pixels outside the image count
// nothing).
__device__ __forceinline__ void eval_error_pixel(
    const float* __restrict__ disp, int sd, const float* __restrict__ gt,
    int sg, int W, int H, float abs_thres, float rel_thres,
    unsigned long long* __restrict__ counts, int x, int y) {
  unsigned e = 0, v = 0, a = 0;
  if (x < W && y < H) {
    const float g = gt[(size_t)y * sg + x];
    if (g > 0.0f) {
      const float d = disp[(size_t)y * sd + x];
      const float diff = fabsf(g - d);
      e = (diff > abs_thres && diff / fabsf(g) > rel_thres) ? 1u : 0u;
      v = d > 0.0f ? 1u : 0u;
      a = 1u;
    }
  }
  // wave sums by ballot, then one atomic per wave and counter
  const unsigned long long be = __ballot(e), bv = __ballot(v),
                           ba = __ballot(a);
  if ((threadIdx.x & 63) == 0) {
    if (be) atomicAdd(&counts[0], (unsigned long long)__popcll(be));
    if (bv) atomicAdd(&counts[1], (unsigned long long)__popcll(bv));
    if (ba) atomicAdd(&counts[2], (unsigned long long)__popcll(ba));
  }
}

__global__ void __launch_bounds__(256)
k_eval_error(const float* __restrict__ disp, int sd, const float* __restrict__ gt,
             int sg, int W, int H, float abs_thres, float rel_thres,
             unsigned long long* __restrict__ counts) {
  eval_error_pixel(disp, sd, gt, sg, W, H, abs_thres, rel_thres, counts,
                   blockIdx.x * kBX + threadIdx.x,
                   blockIdx.y * kBY + threadIdx.y);
}

__global__ void k_zero_u64(unsigned long long* __restrict__ p, int n) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0ull;
}

// draws [k + 16 t, k + 16 t + 16) by one jump and sixteen steps
__global__ void __launch_bounds__(256)
k_draws(uint64_t k, int n, float* __restrict__ out) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  const int i0 = t * 16;
  if (i0 >= n) return;
  Mwc s = mwc_jump(k + (uint64_t)i0);
  for (int j = 0; j < 16 && i0 + j < n; ++j) out[i0 + j] = mwc_next(&s);
}

// plain streaming copy of n float4: the known-size workload that the HBM
// byte counters are calibrated with
__global__ void __launch_bounds__(256)
k_copy_probe(const float4* __restrict__ src, float4* __restrict__ dst,
             size_t n) {
  const size_t stride = (size_t)gridDim.x * 256;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride)
    dst[i] = src[i];
}

__global__ void __launch_bounds__(256)
k_math(const float* __restrict__ in, int n, float* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float x = in[i];
  float s, c;
  sincos_f(x, &s, &c);
  out[5 * i + 0] = exp_f(x);
  out[5 * i + 1] = s;
  out[5 * i + 2] = c;
  out[5 * i + 3] = acospi_f(x);
  out[5 * i + 4] = sqrtf(x);
}

// ---------------------------------------------------------------------
// batches of pairs of uneven sizes (BatchPair descriptors in device
// memory).  The tile kernels number the tile blocks of all pairs in one
// sequence, pair after pair, row-major within a pair; the per-pixel
// kernels take the pair (and view) from the grid's z index.
// ---------------------------------------------------------------------

// Persistent walk over the tile blocks: the sequence is cut into kXcds
// contiguous eighths, and the work-groups of XCD k (hardware ids congruent
// to k, dispatched round-robin) take the k-th eighth with a stride of
// their number, so each XCD's L2 serves a contiguous run of rows.  Each
// work-group calls body(pair, bx, by) for its blocks in increasing order;
// every block of [0, nitems) is visited exactly once for any grid of at
// least kXcds work-groups.  The barrier before each block keeps the
// previous block's LDS tile intact until every wavefront is done with it.
// kWide: the blocks are wide tiles.
template <bool kWide, typename Body>
__device__ __forceinline__ void batch_walk(const BatchPair* __restrict__ pairs,
                                           int npairs, long long nitems,
                                           Body body) {
  const int G = (int)gridDim.x, w = (int)blockIdx.x;
  const int xcd = w % kXcds, j = w / kXcds;
  const int g8 = (G - xcd + kXcds - 1) / kXcds;
  const long long i0 = nitems * xcd / kXcds, i1 = nitems * (xcd + 1) / kXcds;
  int pi = 0;
  for (long long it = i0 + j; it < i1; it += g8) {
    __syncthreads();
    while (pi + 1 < npairs &&
           (kWide ? pairs[pi + 1].wide0 : pairs[pi + 1].item0) <= it)
      ++pi;
    const BatchPair& P = pairs[pi];
    const long long li = it - (kWide ? P.wide0 : P.item0);
    const int nbx = kWide ? (P.g.W + kWideCols - 1) / kWideCols : P.nbx;
    body(P, (int)(li % nbx), (int)(li / nbx));
  }
}

template <int kKind, int kRows>
__global__ void __launch_bounds__(64 * kRows)
k_init_batch(const BatchPair* __restrict__ pairs, int npairs,
             long long nitems, int view) {
  extern __shared__ float4 smem[];
  batch_walk<false>(pairs, npairs, nitems,
                    [&](const BatchPair& P, int bx, int by) {
    init_block<kKind, kRows>(P.g, P.v[view], P.v[1 - view], P.dmax,
                             view == 0 ? 1 : 0, P.state[view][0], smem, bx,
                             by);
  });
}

// one view's propagate over all pairs: the single-image launch's
// arguments (one_iteration in pm_capi.cpp) from each pair's descriptor
__device__ __forceinline__ PropagateArgs batch_args(const BatchPair& P,
                                                    int view, int cur,
                                                    int iter) {
  PropagateArgs a;
  a.self = P.v[view];
  a.other = P.v[1 - view];
  a.old = P.state[view][cur];
  a.out = P.state[view][1 - cur];
  a.smooth = nullptr;
  a.viewin = P.vbuf[1 - view];
  a.viewout = P.vbuf[view];
  // the left view reads the right view's field of the previous iteration,
  // the right view the left view's new one
  a.src_other = view == 0 ? P.state[1][cur] : P.state[0][1 - cur];
  a.dmax = P.dmax;
  a.theta = 0.0f;
  a.lr = view == 0 ? 1 : 0;
  a.iter = iter;
  a.flat_cost = P.flat[view];
  a.flat_known = iter > 0;
  return a;
}

template <int kKind, int kRows, int kEu>
__global__ void __launch_bounds__(64 * kRows)
__attribute__((amdgpu_waves_per_eu(kEu, kEu)))
k_propagate_batch(const BatchPair* __restrict__ pairs, int npairs,
                  long long nitems, int view, int cur, int iter) {
  extern __shared__ float4 smem[];
  batch_walk<false>(pairs, npairs, nitems,
                    [&](const BatchPair& P, int bx, int by) {
    propagate_block<kKind, false, false, kRows, 1, false>(
        P.g, batch_args(P, view, cur, iter), nullptr, smem, bx * kTX,
        by * kRows, P.g.H, Window());
  });
}

template <int kKind>
__global__ void __launch_bounds__(kWideCols * kWideRows)
__attribute__((amdgpu_waves_per_eu(4, 4)))
k_propagate_batch_wide(const BatchPair* __restrict__ pairs, int npairs,
                       long long nitems, int view, int cur, int iter) {
  extern __shared__ float4 smem[];
  batch_walk<true>(pairs, npairs, nitems,
                   [&](const BatchPair& P, int bx, int by) {
    propagate_block<kKind, false, false, kWideRows, kWideCols / kTX, true>(
        P.g, batch_args(P, view, cur, iter), nullptr, smem, bx * kWideCols,
        by * kWideRows, P.g.H,
        window_of(P.g.R, P.dmax, view == 0 ? 1 : 0));
  });
}

__global__ void __launch_bounds__(256)
k_prepare_batch(const BatchPair* __restrict__ pairs, int R, float cw,
                float lim) {
  const BatchPair& P = pairs[blockIdx.z >> 1];
  const int view = blockIdx.z & 1;
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  if (x >= P.g.W || y >= P.g.H) return;
  prepare_pixel(P.img[view], P.g.W, P.g.H, P.channels, P.stride, R, cw, lim,
                P.v[view].tex, P.v[view].sgn, x, y);
}

__global__ void __launch_bounds__(256)
k_clear_wild_batch(const BatchPair* __restrict__ pairs, int npairs) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= 2 * npairs) return;
  const BatchPair& P = pairs[i >> 1];
  *wild_word(P.v[i & 1].tex, P.g.TS, P.g.H) = 0u;
}

__global__ void __launch_bounds__(256)
k_viewbuf_clear_batch(const BatchPair* __restrict__ pairs, int view) {
  const BatchPair& P = pairs[blockIdx.z];
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  if (x >= P.g.W || y >= P.g.H) return;
  P.vbuf[view][(size_t)y * P.g.W + x] = ~0ull;
}

__global__ void __launch_bounds__(256)
k_consistency_batch(const BatchPair* __restrict__ pairs, int cur,
                    float maxdispdiff, float maxdeg) {
  const BatchPair& P = pairs[blockIdx.z];
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  if (x >= P.g.W || y >= P.g.H) return;
  consistency_pixel(P.g.W, P.state[0][cur], P.state[1][cur], maxdispdiff,
                    maxdeg, P.checked, x, y);
}

// pp 0: the left field's disparity; 1: the LR-checked field's; 2: the
// LR-checked field's, holes filled
__global__ void __launch_bounds__(256)
k_disparity_batch(const BatchPair* __restrict__ pairs, int cur, int pp) {
  const BatchPair& P = pairs[blockIdx.z];
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  if (x >= P.g.W || y >= P.g.H) return;
  if (pp == 2)
    fill_depthmap_pixel(P.g.W, P.checked, 1.0f, P.disp, x, y);
  else
    to_disparity_pixel(P.g.W, pp == 1 ? P.checked : P.state[0][cur], 1.0f,
                       1, P.disp, x, y);
}

__global__ void __launch_bounds__(256)
k_zero_counts_batch(const BatchPair* __restrict__ pairs, int npairs) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < 3 * npairs && pairs[i / 3].counts) pairs[i / 3].counts[i % 3] = 0ull;
}

__global__ void __launch_bounds__(256)
k_eval_error_batch(const BatchPair* __restrict__ pairs, float abs_thres,
                   float rel_thres) {
  const BatchPair& P = pairs[blockIdx.z];
  if (!P.gt || !P.counts) return;   // uniform over the work-group
  const int x = blockIdx.x * kBX + threadIdx.x;
  const int y = blockIdx.y * kBY + threadIdx.y;
  eval_error_pixel(P.disp, P.g.W, P.gt, P.gt_stride, P.g.W, P.g.H, abs_thres,
                   rel_thres, P.counts, x, y);
}

// ---------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------
// Launches and returns the launch's own error.  The runtime's last-error
// slot is cleared first: an earlier failed call, already returned to its
// caller, is not reported again here.
#define PM_LAUNCH(kernel, grid, block, lds, st, ...)                \
  do {                                                              \
    (void)hipGetLastError();                                        \
    hipLaunchKernelGGL(kernel, grid, block, lds, st, __VA_ARGS__);  \
    return hipGetLastError();                                       \
  } while (0)

static const dim3 kBlock2D(kBX, kBY);
static const dim3 kBlockTile(kTX, kTY);

// dynamic LDS above 64 KiB has to be allowed per kernel
template <typename K>
static hipError_t allow_lds(K kernel, size_t bytes) {
  if (bytes <= 65536) return hipSuccess;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                             hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)bytes);
}

#define PM_LAUNCH_TILE(kernel, kind, g, st, ...)                        \
  do {                                                                  \
    const size_t lds_ = tile_lds_bytes((g).R, kind, kTX, kTY, 0);       \
    hipError_t e_ = allow_lds(kernel, lds_);                            \
    if (e_ != hipSuccess) return e_;                                    \
    PM_LAUNCH(kernel, grid_for(g), kBlockTile, lds_, st,                \
              __VA_ARGS__);                                             \
  } while (0)

// largest colour magnitude of a tame image: |gray difference| <= 2 lim, so
// the exponent of a support weight stays above -80
static float tame_limit(float color_weight, int cost_kind,
                        float cost_weight) {
  const float w = cost_kind == kCostColorGrad
                      ? std::max(color_weight, cost_weight)
                      : color_weight;
  return w > 39e-4f ? 39.0f / w : 1e4f;
}

hipError_t launch_clear_wild(hipStream_t st, const Geometry& g, ViewBufs a,
                             ViewBufs b) {
  PM_LAUNCH(k_clear_wild, dim3(1), dim3(64), 0, st, wild_word(a.tex, g.TS, g.H),
            wild_word(b.tex, g.TS, g.H));
}

hipError_t launch_costs_unknown(hipStream_t st, CostWords* cw, int view) {
  PM_LAUNCH(k_costs_unknown, dim3(1), dim3(64), 0, st, cw, view);
}

hipError_t launch_forget_costs(hipStream_t st, size_t npix, CostWords* cw,
                               float4* left, float4* right) {
  const unsigned blocks =
      (unsigned)std::min<size_t>((npix + 255) / 256, 256);
  PM_LAUNCH(k_forget_costs, dim3(blocks, 2), dim3(256), 0, st, npix, cw, left,
            right);
}

hipError_t launch_prepare(hipStream_t st, const Geometry& g, const float* img,
                          int channels, int stride, ViewBufs v) {
  const dim3 grid((g.W + kBX - 1) / kBX, (g.H + kBY - 1) / kBY);
  PM_LAUNCH(k_prepare, grid, kBlock2D, 0, st, img, g.W, g.H, channels, stride,
            g.R, g.color_weight,
            tame_limit(g.color_weight, g.cost_kind, g.cost_weight), v.tex,
            v.sgn);
}

hipError_t launch_init(hipStream_t st, const Geometry& g, ViewBufs self,
                       ViewBufs other, float dmax, int lr, float4* states) {
  if (g.cost_kind == kCostColorGrad)
    PM_LAUNCH_TILE(k_init<kCostColorGrad>, kCostColorGrad, g, st, g, self,
                   other, dmax, lr, states);
  PM_LAUNCH_TILE(k_init<kCostCensus>, kCostCensus, g, st, g, self, other,
                 dmax, lr, states);
}

hipError_t launch_disparity_to_normal(hipStream_t st, const Geometry& g,
                                      const float* disp, float4* normals) {
  PM_LAUNCH(k_disparity_to_normal,
            dim3((g.W + kBX - 1) / kBX, (g.H + kBY - 1) / kBY), kBlock2D, 0,
            st, g.W, g.H, disp, normals);
}

hipError_t launch_init_prior(hipStream_t st, const Geometry& g, ViewBufs self,
                             ViewBufs other, float dmax, int lr,
                             const float* disp, const float4* normals,
                             float4* states) {
  if (g.cost_kind == kCostColorGrad)
    PM_LAUNCH_TILE(k_init_prior<kCostColorGrad>, kCostColorGrad, g, st, g,
                   self, other, dmax, lr, disp, normals, states);
  PM_LAUNCH_TILE(k_init_prior<kCostCensus>, kCostCensus, g, st, g, self,
                 other, dmax, lr, disp, normals, states);
}

hipError_t launch_init_proposal(hipStream_t st, const Geometry& g,
                                ViewBufs self, ViewBufs other, float dmax,
                                int lr, const float* prop, int os, int Wp,
                                float dscale, float4* states) {
  if (g.cost_kind == kCostColorGrad)
    PM_LAUNCH_TILE(k_init_proposal<kCostColorGrad>, kCostColorGrad, g, st, g,
                   self, other, dmax, lr, prop, os, Wp, dscale, states);
  PM_LAUNCH_TILE(k_init_proposal<kCostCensus>, kCostCensus, g, st, g, self,
                 other, dmax, lr, prop, os, Wp, dscale, states);
}

hipError_t launch_viewbuf_clear_rows(hipStream_t st, const Geometry& g,
                                     unsigned long long* vbuf, int row0,
                                     int rows) {
  if (row0 < 0 || rows < 0 || row0 + rows > g.H) return hipErrorInvalidValue;
  const size_t n = (size_t)rows * g.W;
  if (n == 0) return hipSuccess;
  const unsigned blocks = (unsigned)((n + 255) / 256);
  PM_LAUNCH(k_viewbuf_clear, dim3(blocks), dim3(256), 0, st, n,
            vbuf + (size_t)row0 * g.W, (CostWords*)nullptr);
}

hipError_t launch_viewbuf_clear(hipStream_t st, const Geometry& g,
                                unsigned long long* vbuf, CostWords* cw) {
  const unsigned blocks = (unsigned)((g.npix + 255) / 256);
  PM_LAUNCH(k_viewbuf_clear, dim3(blocks), dim3(256), 0, st, g.npix, vbuf, cw);
}

template <int kKind, bool kCount, bool kRB, int kRows, int kWX, bool kWin,
          int kTeam = 1, int kEu = 4>
static hipError_t launch_propagate_tile(hipStream_t st, const Geometry& g,
                                        const PropagateArgs& a,
                                        unsigned long long* counters,
                                        size_t lds, Window win) {
  const int cols = (kRB ? 2 : 1) * kTX * kWX / kTeam;
  const int rows = g.row_end() - g.band0 * kBandRows;
  const dim3 grid((unsigned)((g.W + cols - 1) / cols),
                  (unsigned)((rows + kRows - 1) / kRows));
  constexpr auto kernel =
      k_propagate<kKind, kCount, kRB, kRows, kWX, kWin, kTeam, kEu>;
  const hipError_t e = allow_lds(kernel, lds);
  if (e != hipSuccess) return e;
  PM_LAUNCH(kernel, grid, dim3(kTX * kWX, kRows), lds, st, g, a, counters, win);
}

// Five wavefronts per SIMD, at 96 registers and some spills, are 1 to 7 %
// slower than four while either fills the GPU, but a launch with nothing
// beside it (a batch's, a red-black pass) that is a little more than one or
// a few rounds of four takes a round less with five (from six rounds on it is
// all one).  Batches by work-groups of 64 x 4 pixels (1024 to a round of four,
// 1280 to one of five), the time with four and with five against a kernel of
// five whose candidates were unrolled:
//   900  1050  1092  1200  1272  1320  1800  2000  2100  2208  2400  3180  3600
//   .94   .82   .98  1.15  1.08   .98   .92   .88  1.02  1.03   .93   .97   .92
//   .95   .95   .95   .94   .95   .94   .99   .95   .93   .94   .94   .95   .94
static bool saves_a_round(long long workgroups, int waves, size_t lds) {
  if (20 % waves || 20 / waves * lds > kLdsPerCu) return false;
  const long long four = 4 * kCus * 4, five = 5 * kCus * 4;
  const long long n = workgroups * waves;
  const long long over = n - 128;  // 3 % more fit into a round's end
  return n < 6 * four &&
         (over + four - 1) / four > (n + five - 1) / five &&
         (over - 1) % four < 1920;
}

size_t wide_lds_bytes(int R, int cost_kind, float dmax) {
  return tile_lds_bytes(R, cost_kind, kWideCols, kWideRows,
                        window_of(R, dmax, 1).cols);
}

// The wide tile pays when the image has enough of them and they cover it
// without much more padding than 64 x 4 tiles: a CU holds one, so an image of
// 260 tiles takes two rounds with the second nearly empty, a tile whose
// second half lies beyond the right border keeps the CU for the first, and
// the smaller the patch the less the window saves per tile staged.  Time
// against the 64 x 4 tiles (teams, where those are taken), plain PatchMatch,
// by padding (wide pixels over narrow ones) and tiles:
//   padding   1.00                1.06  1.07  1.09  1.11  1.14  1.20  1.33
//   tiles      260   320   480    700   700   700   700   700   700   700
//   R = 2     1.11  1.03   .99   1.05  1.02  1.02  1.07  1.10  1.08  1.16
//   R = 4     1.09   .98   .93    .95   .97   .96  1.02  1.05  1.03  1.16
//   R = 5     1.07   .97   .91    .95   .97   .96  1.01  1.03  1.02  1.12
// (widths 640, 1030, 900, 700, 520, 390, 300, 140); R = 4 at 320 tiles and
// 1.06 to 1.09 1.02 to 1.03.  Uneven batches of 1.03 and 1.06, R = 4: .94 and
// .98.
//   A launch with nothing beside it (alone: a batch's; an image's bands and
// iterations overlap) also ends with a round that has to be half full, the
// sooner the fewer rounds there are.  Of 110 batches of 128 to 896 columns,
// the wide tiles' time against the better of the others at tiles
//   250-325    1.0-1.5    (one round of 256, almost or just over)
//   330-488    .74-1.0
//   490-610    1.0-1.25
//   620-750     .83-1.0
//   756-836     .94-1.1
//   880-1000    .85-.97
//   1064-1130   .95-1.0    (from there on .88-.98)
bool wide_pays(int R, long long tiles, long long narrow, bool alone) {
  const long long wide = tiles * (kWideCols * kWideRows);
  if (alone && tiles < 1130 && (tiles + 24 + kCus - 1) % kCus + 1 < 130)
    return false;
  const bool tight = 50 * wide <= 51 * narrow;
  if (tiles < 448) return R >= 4 && tiles >= 300 && tight;
  return R >= 4 ? 10 * wide <= 11 * narrow : tight;
}

bool wide_fits(int R, int cost_kind, float dmax, int maxW) {
  return dmax < 4096.0f && maxW < (1 << 23) &&
         wide_lds_bytes(R, cost_kind, dmax) <= kLdsPerCu;
}
long long wide_tiles(int W, int H) {
  return (long long)((W + kWideCols - 1) / kWideCols) *
         ((H + kWideRows - 1) / kWideRows);
}
long long narrow_pixels(int W, int H) {
  return (long long)((W + kTX - 1) / kTX * kTX) *
         ((H + kTY - 1) / kTY * kTY);
}

// Teams pay while the image is too small to fill the GPU with one lane per
// pixel.  The work of a team is its slots, 4 ceil((2 R + 1) / 4) a patch row,
// so the line is on pixels times slots per tap; below R = 3 what all four
// lanes do alike weighs more.  Time with teams against without, census,
// Jacobi (red-black):
//   R                1     2     3     4     5     6     7
//   160 x 120            .67         .53   .45
//   400 x 300     1.00  1.00   .78   .82   .69   .74   .66
//                 (.82) (.81) (.61) (.65) (.53) (.55) (.47)
//   512 x 384     1.25  1.21   .90   .95   .79   .85   .75
//                (1.18)(1.17) (.88) (.94) (.79) (.85) (.75)
//   560 x 416     1.43  1.41  1.06  1.13   .94  1.01   .90
//                (1.21)(1.16) (.87) (.93) (.77) (.83) (.73)
// Beside PM-Huber smoothing, which takes CUs itself, the line lies lower.
// depthMap (disparityMap is alike), 4 iterations, teams against without:
//   pixels      30000  50700  76800  108300  145200  187500
//   R = 1         .92    .96   1.01    1.06
//   R = 2         .81    .92   1.00
//   R = 3         .63    .78    .87     .97     .98    1.08
//   R = 4         .59    .76    .90    1.02    1.03    1.15
//   R = 5         .46    .67    .79     .90     .90    1.02
// and the work-groups ask for no more LDS than they use: with the floor that
// makes room for the smoothing beside 64 x 4 tiles, 50700 pixels take 2 to 9
// % more time, 187500 pixels 7 %.
static bool team_pays(int R, int W, int H, bool smoothing) {
  const long long taps = 2 * R + 1;
  const long long slots = (taps + kTeamLanes - 1) / kTeamLanes * kTeamLanes;
  const long long line = smoothing ? (R < 3 ? 90000 : 163840)
                                   : (R < 3 ? 150000 : 262144);
  return (long long)W * H * slots <= taps * line;
}

template <int kKind, bool kRB>
static hipError_t launch_propagate_kind(hipStream_t st, const Geometry& g,
                                        const PropagateArgs& a,
                                        unsigned long long* counters,
                                        size_t lds_floor) {
  const size_t lds = std::max(
      tile_lds_bytes(g.R, kKind, (kRB ? 2 : 1) * kTX, kTY, 0), lds_floor);
  if (counters)
    return launch_propagate_tile<kKind, true, kRB, kTY, 1, false>(
        st, g, a, counters, lds, Window());
  // (a radius whose 64 x 4 tile does not fit is refused below)
  if (lds <= kLdsPerCu && team_pays(g.R, g.W, g.H, a.smooth != nullptr))
    return launch_propagate_tile<kKind, false, kRB, kTY, 1, false, kTeamLanes>(
        st, g, a, counters,
        tile_lds_bytes(g.R, kKind, (kRB ? 2 : 1) * kTX / kTeamLanes, kTY, 0),
        Window());
  if (!kRB && wide_fits(g.R, kKind, a.dmax, g.W) &&
      wide_pays(g.R, wide_tiles(g.W, g.H), narrow_pixels(g.W, g.H), false))
    return launch_propagate_tile<kKind, false, false, kWideRows,
                                 kWideCols / kTX, true>(
        st, g, a, counters, wide_lds_bytes(g.R, kKind, a.dmax),
        window_of(g.R, a.dmax, a.lr));
  // The build for five: beside smoothing, three work-groups a CU whichever it
  // is, from radius 4 on for the registers it leaves (radius 5, 620 x 465:
  // depthMap 20.5 ms with the build for four, 18.3 with it; 1 to 2 % more where
  // the smoothing fits beside either, as it always did at radius 2 and 3), and
  // in red-black's passes, in its first round only (640 x 960, R = 4: 1.00 with
  // four, .96 with five; 1280 x 960 .92 and .95).
  const long long blocks = (long long)((g.W + 2 * kTX - 1) / (2 * kTX)) *
                           ((g.H + kTY - 1) / kTY);
  if (a.smooth ? g.R >= 4
               : kRB && blocks <= 5 * kCus && saves_a_round(blocks, kTY, lds))
    return launch_propagate_tile<kKind, false, kRB, kTY, 1, false, 1, 5>(
        st, g, a, counters, lds, Window());
  return launch_propagate_tile<kKind, false, kRB, kTY, 1, false>(
      st, g, a, counters, lds, Window());
}

hipError_t launch_propagate(hipStream_t st, const Geometry& g,
                            const PropagateArgs& a,
                            unsigned long long* counters, size_t lds_floor) {
  if (g.color != -1 && g.color != 0 && g.color != 1)
    return hipErrorInvalidValue;
  if (g.color >= 0 && g.color == 1 && !a.fresh) return hipErrorInvalidValue;
  const bool rb = g.color >= 0;
  if (g.cost_kind == kCostColorGrad)
    return rb ? launch_propagate_kind<kCostColorGrad, true>(st, g, a, counters,
                                                           lds_floor)
              : launch_propagate_kind<kCostColorGrad, false>(st, g, a,
                                                            counters,
                                                            lds_floor);
  return rb ? launch_propagate_kind<kCostCensus, true>(st, g, a, counters,
                                                      lds_floor)
            : launch_propagate_kind<kCostCensus, false>(st, g, a, counters,
                                                       lds_floor);
}

hipError_t launch_init_from_view(hipStream_t st, const Geometry& g,
                                 float dmax,
                                 const unsigned long long* slots,
                                 const float4* src, float4* states) {
  PM_LAUNCH(k_init_from_view,
            dim3((g.W + kBX - 1) / kBX, (g.H + kBY - 1) / kBY), kBlock2D, 0,
            st, g.W, g.H, dmax, slots, src, states);
}

hipError_t launch_scatter(hipStream_t st, const Geometry& g,
                          const float4* states, int lr,
                          unsigned long long* viewout) {
  PM_LAUNCH(k_scatter, dim3((g.W + kBX - 1) / kBX, (g.H + kBY - 1) / kBY),
            kBlock2D, 0, st, g.W, g.H, states, lr, viewout);
}

hipError_t launch_cost_field(hipStream_t st, const Geometry& g, ViewBufs self,
                             ViewBufs other, const float4* planes,
                             float* cost) {
  if (g.cost_kind == kCostColorGrad)
    PM_LAUNCH_TILE(k_cost_field<kCostColorGrad>, kCostColorGrad, g, st, g,
                   self, other, planes, cost);
  PM_LAUNCH_TILE(k_cost_field<kCostCensus>, kCostCensus, g, st, g, self,
                 other, planes, cost);
}

hipError_t launch_klt_field(hipStream_t st, const Geometry& g, ViewBufs self,
                            ViewBufs other, const float4* planes, int passes,
                            float4* out) {
  PM_LAUNCH_TILE(k_klt_field, kCostCensus, g, st, g, self, other, planes,
                 passes, out);
}

hipError_t launch_consistency(hipStream_t st, const Geometry& g,
                              const float4* left, const float4* right,
                              float maxdispdiff, float maxdeg, float4* out) {
  PM_LAUNCH(k_consistency, dim3((g.W + kBX - 1) / kBX, (g.H + kBY - 1) / kBY),
            kBlock2D, 0, st, g.W, g.H, left, right, maxdispdiff, maxdeg, out);
}

hipError_t launch_to_disparity(hipStream_t st, const Geometry& g,
                               const float4* states, float scale, int lr,
                               float* disp) {
  PM_LAUNCH(k_to_disparity,
            dim3((g.W + kBX - 1) / kBX, (g.H + kBY - 1) / kBY), kBlock2D, 0,
            st, g.W, g.H, states, scale, lr, disp);
}

hipError_t launch_fill_depthmap(hipStream_t st, const Geometry& g,
                                const float4* states, float scale,
                                float* disp) {
  PM_LAUNCH(k_fill_depthmap,
            dim3((g.W + kBX - 1) / kBX, (g.H + kBY - 1) / kBY), kBlock2D, 0,
            st, g.W, g.H, states, scale, disp);
}

hipError_t launch_fill_normalmap(hipStream_t st, const Geometry& g,
                                 const float4* states, float4* normals) {
  PM_LAUNCH(k_fill_normalmap,
            dim3((g.W + kBX - 1) / kBX, (g.H + kBY - 1) / kBY), kBlock2D, 0,
            st, g.W, g.H, states, normals);
}

hipError_t launch_eval_error(hipStream_t st, const float* disp, int sd,
                             const float* gt, int sg, int W, int H,
                             float abs_thres, float rel_thres,
                             unsigned long long* counts) {
  (void)hipGetLastError();
  hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, st, counts, 3);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  PM_LAUNCH(k_eval_error, dim3((W + kBX - 1) / kBX, (H + kBY - 1) / kBY),
            kBlock2D, 0, st, disp, sd, gt, sg, W, H, abs_thres, rel_thres,
            counts);
}

// ---------------------------------------------------------------------
// batch launchers
// ---------------------------------------------------------------------
size_t batch_lds_bytes(int R, int cost_kind, int rows) {
  return tile_lds_bytes(R, cost_kind, kTX, rows, 0);
}

static dim3 batch_pixel_grid(int maxW, int maxH, int z) {
  return dim3((unsigned)((maxW + kBX - 1) / kBX),
              (unsigned)((maxH + kBY - 1) / kBY), (unsigned)z);
}

// persistent grid: at least one work-group per XCD (batch_walk's
// requirement), at most one per tile block
static unsigned batch_tile_grid(long long nitems, BatchShape shape) {
  long long g = shape.workgroups > 0 ? shape.workgroups : nitems;
  g = std::min(g, nitems);
  return (unsigned)std::max<long long>(g, kXcds);
}

hipError_t launch_prepare_batch(hipStream_t st, const BatchPair* pairs,
                                int npairs, int maxW, int maxH, int R,
                                float cw, int cost_kind, float kw) {
  if (npairs < 1) return hipSuccess;
  (void)hipGetLastError();
  hipLaunchKernelGGL(k_clear_wild_batch,
                     dim3((unsigned)((2 * npairs + 255) / 256)), dim3(256), 0,
                     st, pairs, npairs);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  PM_LAUNCH(k_prepare_batch, batch_pixel_grid(maxW, maxH, 2 * npairs),
            kBlock2D, 0, st, pairs, R, cw, tame_limit(cw, cost_kind, kw));
}

hipError_t launch_viewbuf_clear_batch(hipStream_t st, const BatchPair* pairs,
                                      int npairs, int maxW, int maxH,
                                      int view) {
  if (npairs < 1) return hipSuccess;
  PM_LAUNCH(k_viewbuf_clear_batch, batch_pixel_grid(maxW, maxH, npairs),
            kBlock2D, 0, st, pairs, view);
}

template <int kKind, int kRows>
static hipError_t init_batch_rows(hipStream_t st, const BatchPair* pairs,
                                  int npairs, long long nitems, int view,
                                  size_t lds, BatchShape shape) {
  const hipError_t e = allow_lds(k_init_batch<kKind, kRows>, lds);
  if (e != hipSuccess) return e;
  PM_LAUNCH((k_init_batch<kKind, kRows>), dim3(batch_tile_grid(nitems, shape)),
            dim3(kTX, kRows), lds, st, pairs, npairs, nitems, view);
}

template <int kKind>
static hipError_t init_batch_kind(hipStream_t st, const BatchPair* pairs,
                                  int npairs, long long nitems, int view,
                                  size_t lds, BatchShape shape) {
  switch (shape.rows) {
    case 2:
      return init_batch_rows<kKind, 2>(st, pairs, npairs, nitems, view, lds,
                                       shape);
    case 4:
      return init_batch_rows<kKind, 4>(st, pairs, npairs, nitems, view, lds,
                                       shape);
    case 8:
      return init_batch_rows<kKind, 8>(st, pairs, npairs, nitems, view, lds,
                                       shape);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_init_batch(hipStream_t st, const BatchPair* pairs,
                             int npairs, long long nitems, int view,
                             int cost_kind, size_t lds, BatchShape shape) {
  if (nitems < 1) return hipSuccess;
  if (cost_kind == kCostColorGrad)
    return init_batch_kind<kCostColorGrad>(st, pairs, npairs, nitems, view,
                                           lds, shape);
  return init_batch_kind<kCostCensus>(st, pairs, npairs, nitems, view, lds,
                                      shape);
}

template <int kKind, int kRows, int kEu>
static hipError_t propagate_batch_built(hipStream_t st,
                                        const BatchPair* pairs, int npairs,
                                        long long nitems, int view, int cur,
                                        int iter, size_t lds,
                                        BatchShape shape) {
  constexpr auto kernel = k_propagate_batch<kKind, kRows, kEu>;
  const hipError_t e = allow_lds(kernel, lds);
  if (e != hipSuccess) return e;
  PM_LAUNCH(kernel, dim3(batch_tile_grid(nitems, shape)), dim3(kTX, kRows),
            lds, st, pairs, npairs, nitems, view, cur, iter);
}

// (8 rows: five per SIMD would be two and a half work-groups a CU)
template <int kKind, int kRows>
static hipError_t propagate_batch_rows(hipStream_t st, const BatchPair* pairs,
                                       int npairs, long long nitems, int view,
                                       int cur, int iter, size_t lds,
                                       BatchShape shape) {
  if (kRows < 8 && shape.workgroups == 0 && saves_a_round(nitems, kRows, lds))
    return propagate_batch_built<kKind, kRows, kRows < 8 ? 5 : 4>(
        st, pairs, npairs, nitems, view, cur, iter, lds, shape);
  return propagate_batch_built<kKind, kRows, 4>(
      st, pairs, npairs, nitems, view, cur, iter, lds, shape);
}

template <int kKind>
static hipError_t propagate_batch_kind(hipStream_t st, const BatchPair* pairs,
                                       int npairs, long long nitems, int view,
                                       int cur, int iter, size_t lds,
                                       BatchShape shape) {
  switch (shape.rows) {
    case 2:
      return propagate_batch_rows<kKind, 2>(st, pairs, npairs, nitems, view,
                                            cur, iter, lds, shape);
    case 4:
      return propagate_batch_rows<kKind, 4>(st, pairs, npairs, nitems, view,
                                            cur, iter, lds, shape);
    case 8:
      return propagate_batch_rows<kKind, 8>(st, pairs, npairs, nitems, view,
                                            cur, iter, lds, shape);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_propagate_batch(hipStream_t st, const BatchPair* pairs,
                                  int npairs, long long nitems, int view,
                                  int cur, int iter, int cost_kind,
                                  size_t lds, BatchShape shape) {
  if (nitems < 1) return hipSuccess;
  if (cost_kind == kCostColorGrad)
    return propagate_batch_kind<kCostColorGrad>(st, pairs, npairs, nitems,
                                                view, cur, iter, lds, shape);
  return propagate_batch_kind<kCostCensus>(st, pairs, npairs, nitems, view,
                                           cur, iter, lds, shape);
}

hipError_t launch_propagate_batch_wide(hipStream_t st, const BatchPair* pairs,
                                       int npairs, long long nitems, int view,
                                       int cur, int iter, int cost_kind,
                                       size_t lds, int workgroups) {
  if (nitems < 1) return hipSuccess;
  BatchShape shape;
  shape.workgroups = workgroups;
  const dim3 grid(batch_tile_grid(nitems, shape));
  const dim3 block(kWideCols, kWideRows);
  if (cost_kind == kCostColorGrad) {
    const hipError_t e = allow_lds(k_propagate_batch_wide<kCostColorGrad>, lds);
    if (e != hipSuccess) return e;
    PM_LAUNCH(k_propagate_batch_wide<kCostColorGrad>, grid, block, lds, st,
              pairs, npairs, nitems, view, cur, iter);
  }
  const hipError_t e = allow_lds(k_propagate_batch_wide<kCostCensus>, lds);
  if (e != hipSuccess) return e;
  PM_LAUNCH(k_propagate_batch_wide<kCostCensus>, grid, block, lds, st, pairs,
            npairs, nitems, view, cur, iter);
}

hipError_t batch_allow_wide(int cost_kind, size_t lds) {
  return cost_kind == kCostColorGrad
             ? allow_lds(k_propagate_batch_wide<kCostColorGrad>, lds)
             : allow_lds(k_propagate_batch_wide<kCostCensus>, lds);
}

template <int kKind, int kRows>
static hipError_t resident_rows(size_t lds, int* out) {
  hipError_t e = hipSuccess;
  if (kRows < 8)  // before a capture, as the one the occupancy is asked of
    e = allow_lds(k_propagate_batch<kKind, kRows, kRows < 8 ? 5 : 4>, lds);
  if (e == hipSuccess) e = allow_lds(k_propagate_batch<kKind, kRows, 4>, lds);
  if (e != hipSuccess) return e;
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(
      out, k_propagate_batch<kKind, kRows, 4>, kTX * kRows, lds);
}

hipError_t batch_resident_per_cu(int cost_kind, int rows, size_t lds,
                                 int* out) {
  const bool cg = cost_kind == kCostColorGrad;
  switch (rows) {
    case 2:
      return cg ? resident_rows<kCostColorGrad, 2>(lds, out)
                : resident_rows<kCostCensus, 2>(lds, out);
    case 4:
      return cg ? resident_rows<kCostColorGrad, 4>(lds, out)
                : resident_rows<kCostCensus, 4>(lds, out);
    case 8:
      return cg ? resident_rows<kCostColorGrad, 8>(lds, out)
                : resident_rows<kCostCensus, 8>(lds, out);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_postprocess_batch(hipStream_t st, const BatchPair* pairs,
                                    int npairs, int maxW, int maxH, int cur,
                                    int pp, float maxdispdiff, float maxdeg) {
  if (npairs < 1) return hipSuccess;
  if (pp < 0 || pp > 2) return hipErrorInvalidValue;
  const dim3 grid = batch_pixel_grid(maxW, maxH, npairs);
  if (pp != 0) {
    (void)hipGetLastError();
    hipLaunchKernelGGL(k_consistency_batch, grid, kBlock2D, 0, st, pairs,
                       cur, maxdispdiff, maxdeg);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  PM_LAUNCH(k_disparity_batch, grid, kBlock2D, 0, st, pairs, cur, pp);
}

hipError_t launch_eval_error_batch(hipStream_t st, const BatchPair* pairs,
                                   int npairs, int maxW, int maxH,
                                   float abs_thres, float rel_thres) {
  if (npairs < 1) return hipSuccess;
  (void)hipGetLastError();
  hipLaunchKernelGGL(k_zero_counts_batch,
                     dim3((unsigned)((3 * npairs + 255) / 256)), dim3(256), 0,
                     st, pairs, npairs);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  PM_LAUNCH(k_eval_error_batch, batch_pixel_grid(maxW, maxH, npairs),
            kBlock2D, 0, st, pairs, abs_thres, rel_thres);
}

hipError_t launch_draws(hipStream_t st, uint64_t k, int n, float* out) {
  const int threads = (n + 15) / 16;
  PM_LAUNCH(k_draws, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0,
            st, k, n, out);
}

hipError_t launch_copy_probe(hipStream_t st, const float4* src, float4* dst,
                             size_t n) {
  PM_LAUNCH(k_copy_probe, dim3(4096), dim3(256), 0, st, src, dst, n);
}

hipError_t launch_math(hipStream_t st, const float* in, int n, float* out) {
  PM_LAUNCH(k_math, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, in,
            n, out);
}

}  // namespace pm
