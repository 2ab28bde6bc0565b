// The ionosphere warm-start network on the device: a 4-level U-Net (32 base
// channels) whose 3x3 convolutions, their input and weight gradients run as
// implicit GEMMs on the matrix cores (bf16 operands, fp32 accumulation,
// v_mfma_f32_16x16x16_bf16). Everything between two convolutions is part of
// their operand loads or epilogues: bias and ReLU, pooling, the decoder's
// upsample + concatenation, the 1x1 head, and in the backward pass the ReLU
// mask and the sums over pooled, upsampled and skipped gradients. A forward
// pass is 14 launches, a backward pass 18; gradients are deterministic.
//
// H = colatitude rows (zero padding beyond the pole and the low-latitude
// edge), W = longitude columns (periodic). The network is defined layer by
// layer in kLayers; the numpy statement of the same network is the oracle the
// tests compare with.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "gcs_device.hpp"
#include "gcs_unet.hpp"

namespace gcs {
namespace unet {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kT = 256;

// float -> bf16, round to nearest even (NaN stays NaN)
__device__ __host__ inline uint16_t to_bf16(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ inline float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ inline uint32_t pack2(float a, float b) {
  return (uint32_t)to_bf16(a) | ((uint32_t)to_bf16(b) << 16);
}

__device__ inline long gtid() { return blockIdx.x * (long)blockDim.x + threadIdx.x; }

// D(16x16) += A(16x16) B(16x16). Lane l supplies A[l%16][4(l/16)+0..3] and
// B[4(l/16)+0..3][l%16]; it holds D[4(l/16)+i][l%16] in element i.
__device__ inline f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
// Eight products per lane as two of these, in the order of the channels. (The
// 16 x 16 x 32 instruction takes them at once, but the convolutions are not
// bound by the matrix cores.)
__device__ inline f32x4 mfma32(u32x4 a, u32x4 b, f32x4 c) {
  c = mfma16(__builtin_bit_cast(bf16x4, u32x2{a[0], a[1]}),
             __builtin_bit_cast(bf16x4, u32x2{b[0], b[1]}), c);
  return mfma16(__builtin_bit_cast(bf16x4, u32x2{a[2], a[3]}),
                __builtin_bit_cast(bf16x4, u32x2{b[2], b[3]}), c);
}

// ---- tensors -------------------------------------------------------------------
//
// Activations and masked gradients exist twice. NHWC (channels innermost) is
// what a convolution reads, with each 32 channels in the order of a
// wavefront's results and operands: quarter q of the lanes holds channels 4q ..
// 4q + 3 and 16 + 4q .. 16 + 4q + 3, which lie together as 16 bytes. Planar
// [channel][sample][row][padded row of pixels] is what a weight gradient reads:
// its sum runs over pixels, and eight consecutive pixels of a channel are one
// lane's operand. Both are written by the epilogue that has the values in
// registers. Planar rows are padded to a multiple of
// eight pixels; the first pad element repeats pixel 0 (longitude is
// periodic), the others stay zero, and gradients are zero in the whole pad.
struct Grid {
  int N, H, W;      // samples, rows, columns
  int wp, batches;  // planar row pitch and samples per channel
  __device__ int pixel(int n, int y, int x) const { return (n * H + y) * W + x; }
  __device__ long plane(int c, int n, int y) const {
    return (((long)c * batches + n) * H + y) * wp;
  }
};

// The input of a convolution: channels [0, c0) from src0 (at half resolution,
// read with nearest upsampling), channels [c0, c0 + c1) from src1, NHWC; or
// fp32 features (the network's input), rounded to bf16 as they are read.
struct ConvIn {
  const uint16_t *src0 = nullptr, *src1 = nullptr;
  const float *f32 = nullptr;
  const uint16_t *zero = nullptr;  // what rows outside the grid read: 64 zero bytes
  int c0 = 0, c1 = 0;
};

// What a convolution does with its sums.
enum Epilogue {
  EP_FORWARD,  // + bias, ReLU, store; optionally the 2 x 2 mean pool and the 1 x 1 head
  EP_PLAIN,    // input gradient of a plain layer: mask by act > 0, store
  EP_POOL,     // of a layer that reads a pooled activation: spread over 2 x 2 fine
               // pixels, add the skip's gradient, mask, store at the fine grid
  EP_CAT       // of a decoder input: sum 2 x 2 into the coarse activation (channels
               // < c0: mask, store) or keep the skip's gradient (fp32)
};
struct ConvOut {
  Grid g;                       // of `out` (EP_POOL: fine, EP_CAT: coarse)
  uint16_t *out = nullptr, *planar = nullptr;
  const float *bias = nullptr;  // EP_FORWARD
  Grid gp;                      // pooled grid
  uint16_t *pooled = nullptr, *pooled_planar = nullptr;
  const float *head_w = nullptr, *head_b = nullptr;
  float *head_out = nullptr;
  const uint16_t *act = nullptr;  // NHWC activation whose ReLU masks the gradient
  float *skip = nullptr;          // EP_POOL: read; EP_CAT: written; NHWC
  int c0 = 0;                     // EP_CAT: channels of the upsampled part
};

// The lane's eight channels (quarter q of the 32 from c on) of pixel (n, y, x).
__device__ inline void store8(const Grid &g, uint16_t *nhwc, uint16_t *planar, int C, int n, int y,
                              int x, int c, int q, u32x4 v, bool wrap) {
  *(u32x4 *)(nhwc + (long)g.pixel(n, y, x) * C + c + 8 * q) = v;
  const long step = (long)g.batches * g.H * g.wp;
  uint16_t *p = planar + g.plane(c + 4 * q, n, y);
  for (int i = 0; i < 8; ++i) {
    const uint16_t e = (uint16_t)(i & 1 ? v[i >> 1] >> 16 : v[i >> 1]);
    uint16_t *at = p + (i < 4 ? i : 12 + i) * step;
    at[x] = e;
    if (wrap && x == 0 && g.W < g.wp) at[g.W] = e;
  }
}
// Element i of a packed operand, widened.
__device__ inline float element(u32x4 v, int i) {
  return from_bf16((uint16_t)(i & 1 ? v[i >> 1] >> 16 : v[i >> 1]));
}
__device__ inline u32x4 pack8(const float z[8]) {
  return u32x4{pack2(z[0], z[1]), pack2(z[2], z[3]), pack2(z[4], z[5]), pack2(z[6], z[7])};
}

// The value of the neighbouring lane (l ^ 1).
__device__ inline float lane_xor1(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xb1, 0xf, 0xf, true));
}

// 3x3 convolution as an implicit GEMM on 32 output channels x 32 pixels (two
// rows of 16, so that a wavefront holds whole 2 x 2 blocks) per wavefront:
// rows = output channels (weights packed in operand order, k_pack_weights),
// columns = pixels, k = (tap, input channel) in steps of 32 channels. Operands
// come straight from L1 / L2 as 16-byte loads, four loads per four MFMAs, the
// loads of kAhead steps in flight. A tile's sum is one chain: another order
// flips the rounding and the ReLU of values near a tie, and the network and
// its training carry that on (with the deep layers' input gradients split into
// four, 20 training steps took 10.9 instead of 11.2 ms but ended up to 1e-2
// away; now they end as near as two runs that add gradients in another order).
// What bounds it is the latency of a launch and of the loads at the small
// grids, L2 traffic (16 flops a byte) at the large ones. Measured with the
// kernel before, which gathered 8 bytes per lane and MFMA: the 14 layers of
// 2 x 128 x 256, 930 -> 174 us (130 TFLOP/s); a layer of 8 x 32 x 64, 60 -> 11.
constexpr int kAhead = 4;

struct ConvWork {
  ConvIn in;
  Grid g;
  int cout;
  const uint16_t *w;
  ConvOut o;
};

template <int EP, bool F32, bool CAT>
__device__ inline void conv_block(const ConvWork &job, int block) {
  const ConvIn &in = job.in;
  const Grid &g = job.g;
  const ConvOut &o = job.o;
  const uint16_t *__restrict__ w = job.w;
  const int cout = job.cout;
  const int cin = in.c0 + in.c1, spt = cin >> 5, steps = 9 * spt;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int ctiles = cout >> 5, xt = (g.W + 15) >> 4, yt = (g.H + 1) >> 1;
  const int tiles = ctiles * xt * yt * g.N;
  const int tile = block * (int)(blockDim.x >> 6) + wave;
  const bool live = tile < tiles;
  int r = live ? tile : 0;
  const int ct = r % ctiles;
  r /= ctiles;
  const int tx = r % xt;
  r /= xt;
  const int y0 = 2 * (r % yt), n = r / yt;
  const int col = lane & 15, q = lane >> 4;
  const int x = 16 * tx + col, xc = min(x, g.W - 1);
  f32x4 acc[2][2];  // [16 channels][row of pixels]
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint16_t *wt = w + ((long)(2 * ct) * steps * 64 + lane) * 8;
  const long wnext = (long)steps * 64 * 8;
  // One step's operands as loaded: nothing touches a loaded value before its
  // use, and every step loads (the last ones again, past the end), so that the
  // wait before a product leaves the loads of the steps ahead in flight.
  struct Step {
    u32x4 a[2], b[2], b2[F32 ? 2 : 1];
  };
  // The next step to load: its tap's pixels (a row outside the grid reads
  // zeros, whatever the channel) and its first channel.
  int ls = 0, tap = 0, lc = 0;
  const uint16_t *px[2], *px0[2];
  int inside[2];  // all ones, or zero
  auto set_tap = [&]() {
    const int ky = tap / 3, kx = tap - 3 * ky;
    int xx = xc + kx - 1;
    xx = xx < 0 ? g.W - 1 : xx >= g.W ? 0 : xx;
    for (int t = 0; t < 2; ++t) {
      const int yy = y0 + t + ky - 1;
      const bool in_grid = yy >= 0 && yy < g.H;
      inside[t] = in_grid ? -1 : 0;
      const int at = g.pixel(n, yy, xx);
      if (F32)
        px[t] = in_grid ? (const uint16_t *)(in.f32 + (long)at * cin + 4 * q) : in.zero;
      else
        px[t] = in_grid ? in.src1 + (long)at * in.c1 + 8 * q : in.zero;
      if (CAT) {
        const int up = (n * (g.H >> 1) + (yy >> 1)) * (g.W >> 1) + (xx >> 1);
        px0[t] = in_grid ? in.src0 + (long)up * in.c0 + 8 * q : in.zero;
      }
    }
  };
  set_tap();
  auto load = [&](Step &o) {
    const uint16_t *ws = wt + (long)min(ls, steps - 1) * 512;
    const int c = lc * 32;
    for (int t = 0; t < 2; ++t) {
      o.a[t] = *(const u32x4 *)(ws + t * wnext);
      if (F32) {
        o.b[t] = *(const u32x4 *)px[t];
        o.b2[t] = *(const u32x4 *)(px[t] + (32 & inside[t]));  // 16 floats on
      } else if (CAT && c < in.c0) {
        o.b[t] = *(const u32x4 *)(px0[t] + (c & inside[t]));
      } else {
        o.b[t] = *(const u32x4 *)(px[t] + ((c - in.c0) & inside[t]));
      }
    }
    ++ls;
    if (++lc == spt) {
      lc = 0;
      if (tap < 8) ++tap;
      set_tap();
    }
  };
  auto operand = [&](const Step &o, int v) {
    if (!F32) return o.b[v];
    const f32x4 lo = __builtin_bit_cast(f32x4, o.b[v]),
                hi = __builtin_bit_cast(f32x4, o.b2[F32 ? v : 0]);
    return u32x4{pack2(lo[0], lo[1]), pack2(lo[2], lo[3]), pack2(hi[0], hi[1]),
                 pack2(hi[2], hi[3])};
  };
  if (live) {
    Step ahead[kAhead];
#pragma unroll
    for (int p = 0; p < kAhead; ++p) load(ahead[p]);
    auto use = [&](const Step &o) {
      for (int v = 0; v < 2; ++v) {
        const u32x4 b = operand(o, v);
        for (int t = 0; t < 2; ++t) acc[t][v] = mfma32(o.a[t], b, acc[t][v]);
      }
    };
    int left = steps;
    for (; left >= kAhead; left -= kAhead) {
#pragma unroll
      for (int p = 0; p < kAhead; ++p) {
        use(ahead[p]);
        load(ahead[p]);
      }
    }
#pragma unroll
    for (int p = 0; p < kAhead - 1; ++p)
      if (p < left) use(ahead[p]);
  }
  if (!live) return;
  // lane: channels c + 4q + 0..3 and c + 16 + 4q + 0..3 of pixels (y0 + v, x)
  const bool xin = x < g.W;
  const int c = 32 * ct;
  float sum[2][8];
  for (int v = 0; v < 2; ++v)
    for (int i = 0; i < 8; ++i) sum[v][i] = acc[i >> 2][v][i & 3];
  if (EP == EP_FORWARD) {
    const f32x4 b0 = *(const f32x4 *)(o.bias + c + 4 * q),
                b1 = *(const f32x4 *)(o.bias + c + 16 + 4 * q);
    u32x4 z[2];
    for (int v = 0; v < 2; ++v) {
      for (int i = 0; i < 8; ++i)
        sum[v][i] = fmaxf(sum[v][i] + (i < 4 ? b0[i & 3] : b1[i & 3]), 0.f);
      z[v] = pack8(sum[v]);
      if (xin && y0 + v < g.H) store8(o.g, o.out, o.planar, cout, n, y0 + v, x, c, q, z[v], true);
    }
    if (o.pooled != nullptr) {
      // mean of the stored (rounded) values, in the order (0,0) (0,1) (1,0) (1,1)
      float m[8];
      for (int i = 0; i < 8; ++i) {
        const float top = element(z[0], i), low = element(z[1], i);
        const float top1 = lane_xor1(top), low1 = lane_xor1(low);
        m[i] = 0.25f * (((top + top1) + low) + low1);
      }
      if (xin && !(col & 1))
        store8(o.gp, o.pooled, o.pooled_planar, cout, n, y0 >> 1, x >> 1, c, q, pack8(m), true);
    }
    if (o.head_out != nullptr) {
      const f32x4 h0 = *(const f32x4 *)(o.head_w + 4 * q),
                  h1 = *(const f32x4 *)(o.head_w + 16 + 4 * q);
      for (int v = 0; v < 2; ++v) {
        // in the order of the channels (32 are one tile): a quarter adds four
        // and hands the sum to the next
        float s = 0.f;
        for (int h = 0; h < 8; ++h) {
          const int first = h < 4 ? 0 : 4;
          for (int i = first; i < first + 4; ++i)
            s += element(z[v], i) * (i < 4 ? h0[i & 3] : h1[i & 3]);
          s = __shfl(s, 16 * (h & 3) + col, 64);
        }
        if (q == 0 && xin && y0 + v < g.H) o.head_out[g.pixel(n, y0 + v, x)] = s + o.head_b[0];
      }
    }
  } else if (EP == EP_PLAIN) {
    for (int v = 0; v < 2; ++v) {
      if (!xin || y0 + v >= g.H) continue;
      const u32x4 m = *(const u32x4 *)(o.act + (long)g.pixel(n, y0 + v, x) * cout + c + 8 * q);
      for (int i = 0; i < 8; ++i) sum[v][i] = element(m, i) > 0.f ? sum[v][i] : 0.f;
      store8(o.g, o.out, o.planar, cout, n, y0 + v, x, c, q, pack8(sum[v]), false);
    }
  } else if (EP == EP_POOL) {
    for (int v = 0; v < 2; ++v) {
      if (!xin || y0 + v >= g.H) continue;
      for (int f = 0; f < 4; ++f) {
        const int fy = 2 * (y0 + v) + (f >> 1), fx = 2 * x + (f & 1);
        const long p = (long)o.g.pixel(n, fy, fx) * cout + c + 8 * q;
        const f32x4 s0 = *(const f32x4 *)(o.skip + p), s1 = *(const f32x4 *)(o.skip + p + 4);
        const u32x4 m = *(const u32x4 *)(o.act + p);
        float z[8];
        for (int i = 0; i < 8; ++i)
          z[i] = element(m, i) > 0.f ? (i < 4 ? s0[i & 3] : s1[i & 3]) + 0.25f * sum[v][i] : 0.f;
        store8(o.g, o.out, o.planar, cout, n, fy, fx, c, q, pack8(z), false);
      }
    }
  } else if (c < o.c0) {  // EP_CAT, upsampled part
    float z[8];
    for (int i = 0; i < 8; ++i) {
      const float top1 = lane_xor1(sum[0][i]), low1 = lane_xor1(sum[1][i]);
      z[i] = ((sum[0][i] + top1) + sum[1][i]) + low1;
    }
    if (xin && !(col & 1)) {
      const u32x4 m =
          *(const u32x4 *)(o.act + (long)o.g.pixel(n, y0 >> 1, x >> 1) * o.c0 + c + 8 * q);
      for (int i = 0; i < 8; ++i)
        if (!(element(m, i) > 0.f)) z[i] = 0.f;
      store8(o.g, o.out, o.planar, o.c0, n, y0 >> 1, x >> 1, c, q, pack8(z), false);
    }
  } else if (xin) {  // EP_CAT, skip part, kept in the same channel order
    for (int v = 0; v < 2; ++v)
      if (y0 + v < g.H) {
        float *p = o.skip + (long)g.pixel(n, y0 + v, x) * (cout - o.c0) + (c - o.c0) + 8 * q;
        *(f32x4 *)p = f32x4{sum[v][0], sum[v][1], sum[v][2], sum[v][3]};
        *(f32x4 *)(p + 4) = f32x4{sum[v][4], sum[v][5], sum[v][6], sum[v][7]};
      }
  }
}

// A forward layer. One wavefront to a block up to 1024 tiles (four a CU), so that a deep
// layer's few long sums have a CU's load path each and neighbouring XCDs read
// different weights, else four (forward pass of 2 x 32 x 64: 236 us as blocks
// of four, 197 so; of 2 x 128 x 256: 521, 493).
template <bool F32, bool CAT>
__global__ void __launch_bounds__(256) k_conv(ConvWork job) {
  conv_block<EP_FORWARD, F32, CAT>(job, blockIdx.x);
}

// Weight and bias gradients: gw[co][tap][ci] += sum over pixels of gz[co] x
// input[ci, shifted by the tap]. Rows = 32 output channels, columns = 16
// input channels, the reduction over pixels in steps of 32 (four groups of
// eight consecutive pixels of a row, one group per quarter of the wavefront).
// The three taps of a kernel row differ by one pixel, so a lane loads its
// eight pixels and one on each side once and shifts them in registers: eleven
// loads feed 18 MFMAs. A block's four wavefronts take `per_wave` steps each
// and add up in LDS; the blocks' slices of the pixels are added by k_grad_sum
// in their order, so that gradients are the same in every run. Blocks of input
// tile 0 also sum gz itself (a product with ones) for the bias. What bounds it
// is the latency of its few steps at the small grids, the loads' L2 traffic at
// the large ones. Per layer, 8 x 128 x 256: 296 -> 39 us, 8 x 32 x 64: 66 -> 11
// (before: 2-byte gathers, atomics).
struct GradIn {
  const uint16_t *src0 = nullptr, *src1 = nullptr;  // planar; src0 at half resolution
  Grid g0;                                           // of src0
  int c0 = 0, c1 = 0;
};

constexpr int kGradLds = 18 * 256 + 32;  // floats of a block

struct GradWork {
  GradIn in;
  Grid g;
  const uint16_t *gz;  // planar
  int cout, per_wave, blocks;
  float *part;         // [slice][weights, bias] partial sums
};

__device__ inline void wgrad_block(const GradWork &job, int block, float *s_sum) {
  const GradIn &in = job.in;
  const Grid &g = job.g;
  const uint16_t *__restrict__ gz = job.gz;
  const int per_wave = job.per_wave;
  const int cin = in.c0 + in.c1;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, q = lane >> 4;
  const int ctiles = cin / 16, tile = block % (ctiles * (job.cout / 32));
  const int slice = block / (ctiles * (job.cout / 32));
  const int ci0 = (tile % ctiles) * 16, co0 = (tile / ctiles) * 32;
  const int xg_n = g.wp >> 3, groups = g.N * g.H * xg_n;
  const int step0 = (slice * 4 + wave) * per_wave;
  const bool up = ci0 < in.c0;  // a tile lies in one part
  const int ci = ci0 + col;
  f32x4 acc[2][9], bsum[2];
  for (int t = 0; t < 2; ++t) {
    bsum[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < 9; ++k) acc[t][k] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // this quarter's group of eight pixels: (n, y, xg)
  int gi = step0 * 4 + q;
  int xg = gi % xg_n, y = (gi / xg_n) % g.H, n = gi / (xg_n * g.H);
  const u32x4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
  for (int s = 0; s < per_wave; ++s, gi += 4) {
    if (4 * (step0 + s) >= groups) break;  // uniform
    const bool in_range = gi < groups;
    const u32x4 zero = {0u, 0u, 0u, 0u};
    u32x4 a[2] = {zero, zero}, mid[3] = {zero, zero, zero};
    uint32_t left[3] = {0u, 0u, 0u}, right[3] = {0u, 0u, 0u};
    if (in_range) {
      for (int t = 0; t < 2; ++t)
        a[t] = *(const u32x4 *)(gz + g.plane(co0 + 16 * t + col, n, y) + 8 * xg);
      const bool last = 8 * xg + 8 >= g.W;  // right neighbour wraps (or is pad)
      for (int ky = 0; ky < 3; ++ky) {
        const int yy = y + ky - 1;
        if (yy < 0 || yy >= g.H) continue;
        if (up) {
          const uint16_t *p = in.src0 + in.g0.plane(ci, n, yy >> 1);
          const u32x2 e = *(const u32x2 *)(p + 4 * xg);
          mid[ky] = u32x4{(e[0] & 0xffffu) * 0x10001u, (e[0] >> 16) * 0x10001u,
                          (e[1] & 0xffffu) * 0x10001u, (e[1] >> 16) * 0x10001u};
          left[ky] = p[xg == 0 ? in.g0.W - 1 : 4 * xg - 1];
          right[ky] = p[last ? 0 : 4 * xg + 4];
        } else {
          const uint16_t *p = in.src1 + g.plane(ci - in.c0, n, yy);
          mid[ky] = *(const u32x4 *)(p + 8 * xg);
          left[ky] = p[xg == 0 ? g.W - 1 : 8 * xg - 1];
          right[ky] = p[last ? 0 : 8 * xg + 8];
        }
      }
    }
    if (ci0 == 0)
      for (int t = 0; t < 2; ++t) bsum[t] = mfma32(a[t], ones, bsum[t]);
    for (int ky = 0; ky < 3; ++ky) {
      const u32x4 m = mid[ky];
      const uint32_t m01 = __builtin_amdgcn_alignbit(m[1], m[0], 16),
                     m12 = __builtin_amdgcn_alignbit(m[2], m[1], 16),
                     m23 = __builtin_amdgcn_alignbit(m[3], m[2], 16);
      const u32x4 b[3] = {u32x4{(m[0] << 16) | left[ky], m01, m12, m23}, m,
                          u32x4{m01, m12, m23, (m[3] >> 16) | (right[ky] << 16)}};
      for (int kx = 0; kx < 3; ++kx)
        for (int t = 0; t < 2; ++t)
          acc[t][3 * ky + kx] = mfma32(a[t], b[kx], acc[t][3 * ky + kx]);
    }
    xg += 4;
    while (xg >= xg_n) {
      xg -= xg_n;
      if (++y == g.H) {
        y = 0;
        ++n;
      }
    }
  }
  // element i of a sum: output channel 16 t + 4 q + i, input channel col; the
  // wavefronts add theirs in turn
  for (int turn = 0; turn < 4; ++turn) {
    if (wave == turn) {
      for (int t = 0; t < 2; ++t)
        for (int k = 0; k < 9; ++k)
          for (int i = 0; i < 4; ++i) {
            float *e = &s_sum[((16 * t + 4 * q + i) * 9 + k) * 16 + col];
            *e = turn == 0 ? acc[t][k][i] : *e + acc[t][k][i];
          }
      if (col == 0)
        for (int t = 0; t < 2; ++t)
          for (int i = 0; i < 4; ++i) {
            float *e = &s_sum[18 * 256 + 16 * t + 4 * q + i];
            *e = turn == 0 ? bsum[t][i] : *e + bsum[t][i];
          }
    }
    __syncthreads();
  }
  const long weights = 9L * cin * job.cout;
  float *part = job.part + slice * (weights + job.cout);
  for (int t = threadIdx.x; t < 18 * 256; t += 256) {
    const int co = co0 + t / 144, k = (t / 16) % 9;
    part[((long)co * 9 + k) * cin + ci0 + (t & 15)] = s_sum[t];
  }
  if (ci0 == 0 && threadIdx.x < 32) part[weights + co0 + threadIdx.x] = s_sum[18 * 256 + threadIdx.x];
}

__global__ void __launch_bounds__(256) k_wgrad(GradWork job) {
  __shared__ float lds[kGradLds];
  wgrad_block(job, blockIdx.x, lds);
}

// Both products of a layer's backward pass, which need only the masked
// gradient of its output, in one launch: the weight gradient's blocks first,
// then the input gradient's convolution (20 training steps of 8 x 32 x 64:
// 13.3 -> 11.1 ms against two launches, 8 x 128 x 256 the same within 1 %).
template <int EP>
__global__ void __launch_bounds__(256) k_backward(GradWork grad, ConvWork conv) {
  __shared__ float lds[kGradLds];
  if ((int)blockIdx.x < grad.blocks)
    wgrad_block(grad, blockIdx.x, lds);
  else
    conv_block<EP, false, false>(conv, blockIdx.x - grad.blocks);
}

// gradients = the slices' partial sums of every convolution parameter, in the
// slices' order (the head's are k_head_sum's).
struct SliceTable {
  int begin[kLayerCount + 1];     // the layers' first parameters
  int slices[kLayerCount];
  long part[kLayerCount];         // their partial sums
};
__global__ void __launch_bounds__(256) k_grad_sum(const float *part, SliceTable table,
                                                  float *grads) {
  const int t = (int)gtid();
  if (t >= table.begin[kLayerCount]) return;
  int l = 0;
  while (l + 1 < kLayerCount && t >= table.begin[l + 1]) ++l;
  const int size = table.begin[l + 1] - table.begin[l];
  const float *p = part + table.part[l] + (t - table.begin[l]);
  float s = 0.f;
  for (int q = 0; q < table.slices[l]; ++q) s += p[(long)q * size];
  grads[t] = s;
}

// fp32 features to the planar bf16 input (the first layer's weight gradient):
// a block transposes 64 pixels of a row through LDS.
__global__ void __launch_bounds__(256) k_planar_input(const float *in, Grid g, uint16_t *out) {
  __shared__ uint16_t s[64][kInChannels + 2];
  const int xt = (g.W + 63) / 64;
  const int x0 = (blockIdx.x % xt) * 64, row = blockIdx.x / xt;  // row = n H + y
  const int nx = min(64, g.W - x0);
  for (int t = threadIdx.x; t < nx * kInChannels; t += 256)
    s[t / kInChannels][t % kInChannels] =
        to_bf16(in[((long)row * g.W + x0) * kInChannels + t]);
  __syncthreads();
  const int n = row / g.H, y = row % g.H, x = threadIdx.x & 63;
  if (x >= nx) return;
  for (int c = threadIdx.x >> 6; c < kInChannels; c += 4) {
    uint16_t *p = out + g.plane(c, n, y);
    p[x0 + x] = s[x][c];
    if (x0 + x == 0 && g.W < g.wp) p[g.W] = s[x][c];
  }
}

__global__ void k_fill(float *p, long count, float v) {
  const long t = gtid();
  if (t < count) p[t] = v;
}

// Head backward: gz = bf16(g w, masked by act > 0), gw[c] += sum g act[c], gb
// += sum g. Four threads per pixel, eight channels each.
// Each block leaves its 33 sums in part and k_head_sum adds them up: 256 blocks'
// atomics on 33 neighbouring words took 86 us.
__global__ void __launch_bounds__(256) k_head_back(const uint16_t *act, const float *gout, Grid g,
                                                   const float *w, uint16_t *gz,
                                                   uint16_t *gz_planar, float *part) {
  // wavefront q of the block: channels 4q .. + 3 and 16 + 4q .. + 3
  const int q = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int M = g.N * g.H * g.W;
  float sum[8], total = 0.f, hw[8];
  for (int i = 0; i < 8; ++i) {
    sum[i] = 0.f;
    hw[i] = w[(i < 4 ? i : 12 + i) + 4 * q];
  }
  for (int m = blockIdx.x * 64 + lane; m < M; m += gridDim.x * 64) {
    const float gm = gout[m];
    const u32x4 v = *(const u32x4 *)(act + (long)m * kHeadIn + 8 * q);
    float z[8];
    for (int i = 0; i < 8; ++i) {
      const float a = element(v, i);
      sum[i] += gm * a;
      z[i] = a > 0.f ? gm * hw[i] : 0.f;
    }
    total += gm;
    const int x = m % g.W, y = (m / g.W) % g.H, n = m / (g.W * g.H);
    store8(g, gz, gz_planar, kHeadIn, n, y, x, 0, q, pack8(z), false);
  }
  for (int i = 0; i < 8; ++i) {
    float s = sum[i];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if (lane == 0) part[blockIdx.x * (kHeadIn + 1) + (i < 4 ? i : 12 + i) + 4 * q] = s;
  }
  if (q == 0) {
    for (int off = 32; off > 0; off >>= 1) total += __shfl_down(total, off, 64);
    if (lane == 0) part[blockIdx.x * (kHeadIn + 1) + kHeadIn] = total;
  }
}

// gw and gb follow each other in the parameters' order: one wavefront each.
__global__ void __launch_bounds__(64) k_head_sum(const float *part, int blocks, float *gw) {
  float s = 0.f;
  for (int b = threadIdx.x; b < blocks; b += 64) s += part[b * (kHeadIn + 1) + blockIdx.x];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if (threadIdx.x == 0) gw[blockIdx.x] = s;
}

// Mean square error: loss += sum (out - target)^2 / M; g = 2 (out - target) / M.
__global__ void k_mse(const float *out, const float *target, int M, float *g, float *loss) {
  __shared__ float red[kT];
  const long m = gtid();
  float d = 0.f;
  if (m < M) {
    d = out[m] - target[m];
    g[m] = 2.f * d / (float)M;
  }
  red[threadIdx.x] = d * d / (float)M;
  __syncthreads();
  for (int s = kT / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, red[0]);
}

// Mean square of each sample's target (one block per sample).
__global__ void k_sample_energy(const float *target, int P, float *energy) {
  __shared__ float red[kT];
  const float *t = target + (long)blockIdx.x * P;
  float s = 0.f;
  for (int m = threadIdx.x; m < P; m += kT) s += t[m] * t[m];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = kT / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) energy[blockIdx.x] = fmaxf(red[0] / (float)P, 1e-30f);
}

// Relative error: loss += mean over samples of mean_pixels (out - t)^2 /
// energy_b; g = 2 (out - t) / (B P energy_b).
__global__ void k_mse_rel(const float *out, const float *target, int B, int P,
                          const float *energy, float *g, float *loss) {
  __shared__ float red[kT];
  const long m = gtid();
  float d2 = 0.f;
  if (m < (long)B * P) {
    const float e = energy[m / P];
    const float d = out[m] - target[m];
    g[m] = 2.f * d / ((float)B * (float)P * e);
    d2 = d * d / ((float)B * (float)P * e);
  }
  red[threadIdx.x] = d2;
  __syncthreads();
  for (int s = kT / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, red[0]);
}

// Where each convolution's weights live: [cout][9][cin] at w in the
// parameters, and at `packed` in the two bf16 copies in operand order.
struct PackTable {
  int w[kLayerCount], packed[kLayerCount], cin[kLayerCount], cout[kLayerCount];
};

// bf16 copies of parameter t (a convolution weight) in the order k_conv reads:
// [16 output channels][step of 32 k][lane][8], k = (tap, input channel), lane
// l holding output channel l % 16 and input channels 4q .. + 3 and 16 + 4q .. +
// 3 of the step's 32, q = l / 16. `back` is the
// input gradient's convolution: channels exchanged, taps reversed.
__device__ inline void pack_weight(const PackTable &p, int t, float v, uint16_t *fwd,
                                   uint16_t *back) {
  int l = 0;
  while (l + 1 < kLayerCount && t >= p.w[l + 1]) ++l;
  const int cin = p.cin[l], cout = p.cout[l], r = t - p.w[l];
  if (r >= cout * 9 * cin) return;  // a bias
  const int ci = r % cin, tap = (r / cin) % 9, co = r / (9 * cin);
  const uint16_t b = to_bf16(v);
  auto at = [](int row, int tp, int c, int channels) {
    const int spt = channels >> 5, step = tp * spt + (c >> 5);
    const int lane = (row & 15) + 16 * ((c >> 2) & 3), e = (c & 3) + 4 * ((c >> 4) & 1);
    return (((row >> 4) * 9 * spt + step) * 64 + lane) * 8 + e;
  };
  fwd[p.packed[l] + at(co, tap, ci, cin)] = b;
  back[p.packed[l] + at(ci, 8 - tap, co, cout)] = b;
}

__global__ void k_adam(float *p, const float *g, float *mo, float *ve, long count, float lr,
                       float b1, float b2, float c1, float c2, float eps, PackTable table,
                       uint16_t *fwd, uint16_t *back) {
  const long t = gtid();
  if (t >= count) return;
  const float gt = g[t];
  const float m = b1 * mo[t] + (1.f - b1) * gt;
  const float v = b2 * ve[t] + (1.f - b2) * gt * gt;
  mo[t] = m;
  ve[t] = v;
  const float w = p[t] - lr * (m / c1) / (sqrtf(v / c2) + eps);
  p[t] = w;
  pack_weight(table, (int)t, w, fwd, back);
}

__global__ void k_pack_weights(const float *p, long count, PackTable table, uint16_t *fwd,
                               uint16_t *back) {
  const long t = gtid();
  if (t < count) pack_weight(table, (int)t, p[t], fwd, back);
}

// GEMM check of the MFMA operand layout: C[M][N] = A[M][K] B[K][N], bf16 in
// fp32 out, one 16x16 tile per wave (M, N, K multiples of 16).
__global__ void k_gemm_check(const uint16_t *A, const uint16_t *B, int M, int N, int K,
                             float *C) {
  const int lane = threadIdx.x & 63;
  const int row = lane & 15, kq = (lane >> 4) * 4;
  const int m0 = blockIdx.x * 16, n0 = blockIdx.y * 16;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += 16) {
    bf16x4 a, b;
    for (int i = 0; i < 4; ++i) {
      a[i] = (short)A[(long)(m0 + row) * K + k0 + kq + i];
      b[i] = (short)B[(long)(k0 + kq + i) * N + n0 + row];
    }
    acc = mfma16(a, b, acc);
  }
  for (int i = 0; i < 4; ++i) C[(long)(m0 + kq + i) * N + n0 + row] = acc[i];
}

// Wavefronts of a weight-gradient launch over all its tiles: fewer leave the
// chip idle, more write and read more partial sums (8 samples of 128 x 256,
// loss and gradients with transfers: 512 3.65 ms, 1024 3.48, 2048 3.62, 4096
// 3.80; of 32 x 64: 1.09, 1.07, 1.12, 1.11).
constexpr int kGradWaves = 1024;
constexpr int kHeadBlocks = 512;  // most blocks of k_head_back

unsigned nb(long n, int t = kT) { return (unsigned)((n + t - 1) / t); }

}  // namespace

// ---- the network --------------------------------------------------------------

// (cin, cout, input kind, source activations); activations are numbered
// 0 = x, 1 + l = output of layer l.
const LayerSpec kLayers[kLayerCount] = {
    {"e0a", kInChannels, 32, IN_PLAIN, 0, -1},
    {"e0", 32, 32, IN_PLAIN, 1, -1},
    {"e1a", 32, 64, IN_POOL, 2, -1},
    {"e1", 64, 64, IN_PLAIN, 3, -1},
    {"e2a", 64, 128, IN_POOL, 4, -1},
    {"e2", 128, 128, IN_PLAIN, 5, -1},
    {"e3a", 128, 256, IN_POOL, 6, -1},
    {"e3", 256, 256, IN_PLAIN, 7, -1},
    {"d2a", 384, 128, IN_CAT, 8, 6},
    {"d2", 128, 128, IN_PLAIN, 9, -1},
    {"d1a", 192, 64, IN_CAT, 10, 4},
    {"d1", 64, 64, IN_PLAIN, 11, -1},
    {"d0a", 96, 32, IN_CAT, 12, 2},
    {"d0", 32, 32, IN_PLAIN, 13, -1},
};

// Level (0 = full grid) of each activation.
static int act_level(int a) {
  static const int lv[kActs] = {0, 0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0, 0};
  return lv[a];
}
static int act_channels(int a) { return a == 0 ? kInChannels : kLayers[a - 1].cout; }

static Grid grid_of(const Net &n, int level, int batch) {
  Grid g;
  g.N = batch;
  g.H = n.H >> level;
  g.W = n.W >> level;
  g.wp = (g.W + 7) / 8 * 8;
  g.batches = n.max_batch;
  return g;
}

static PackTable pack_table(const Net &n) {
  PackTable t;
  for (int l = 0; l < kLayerCount; ++l) {
    t.w[l] = (int)n.w_off[l];
    t.packed[l] = (int)n.wbf_off[l];
    t.cin[l] = kLayers[l].cin;
    t.cout[l] = kLayers[l].cout;
  }
  return t;
}

Net::~Net() {
  for (void *p : allocations) (void)hipFree(p);
}

// Device allocation recorded in net.allocations (a failed one as nullptr,
// which create() checks for).
template <typename T>
static T *dalloc(Net &net, size_t count) {
  void *p = nullptr;
  if (hipMalloc(&p, count * sizeof(T)) != hipSuccess) p = nullptr;
  net.allocations.push_back(p);
  return (T *)p;
}

// The pixel slices of a layer's weight gradient: blocks of four wavefronts of
// per_wave steps, about kGradWaves wavefronts over all tiles of the layer.
static int grad_slices(const Net &n, int l, int batch, int &per_wave) {
  const LayerSpec &L = kLayers[l];
  const Grid g = grid_of(n, act_level(l + 1), batch);
  const int tiles = (L.cin / 16) * (L.cout / 32);
  const int steps = (g.N * g.H * (g.wp / 8) + 3) / 4;
  const int waves = std::max(4, kGradWaves / tiles);  // per tile
  per_wave = std::max(2, (steps + waves - 1) / waves);
  return (steps + 4 * per_wave - 1) / (4 * per_wave);
}

// Zero bf16 values (an even number of them, in memory of whole words).
static void fill_zero(Net &n, uint16_t *p, long count) {
  k_fill<<<nb(count / 2), kT, 0, n.stream>>>((float *)p, count / 2, 0.f);
}

Net *create(int H, int W, int max_batch, uint64_t seed) {
  if (H <= 0 || W <= 0 || max_batch <= 0 || H % 8 != 0 || W % 8 != 0) {
    set_error("warm-start network: grid must be a positive multiple of 8 in both axes");
    return nullptr;
  }
  Net *net = new Net();
  Net &n = *net;
  n.H = H;
  n.W = W;
  n.max_batch = max_batch;
  // parameter layout: per layer w [cout][9][cin] then b [cout]; head w, b
  size_t off = 0;
  for (int l = 0; l < kLayerCount; ++l) {
    n.w_off[l] = off;
    off += (size_t)kLayers[l].cout * 9 * kLayers[l].cin;
    n.b_off[l] = off;
    off += kLayers[l].cout;
  }
  n.head_w_off = off;
  off += kHeadIn;
  n.head_b_off = off;
  off += 1;
  n.param_count = off;
  n.params = dalloc<float>(n, off);
  n.grads = dalloc<float>(n, off);
  n.adam_m = dalloc<float>(n, off);
  n.adam_v = dalloc<float>(n, off);
  size_t wcount = 0;
  for (int l = 0; l < kLayerCount; ++l) wcount += (size_t)kLayers[l].cout * 9 * kLayers[l].cin;
  n.wbf = dalloc<uint16_t>(n, wcount);
  n.wflip = dalloc<uint16_t>(n, wcount);
  size_t wo = 0;
  for (int l = 0; l < kLayerCount; ++l) {
    n.wbf_off[l] = wo;
    wo += (size_t)kLayers[l].cout * 9 * kLayers[l].cin;
  }
  // activations and masked gradients, NHWC and planar (with zeroed pads);
  // activation 0, the input, has no gradient and no NHWC copy
  for (int a = 0; a < kActs; ++a) {
    const Grid g = grid_of(n, act_level(a), max_batch);
    const long pix = (long)max_batch * g.H * g.W * act_channels(a);
    const long planar = (long)max_batch * g.H * g.wp * act_channels(a);
    n.act_planar[a] = dalloc<uint16_t>(n, planar);
    n.planar_count[a] = planar;
    if (a == 0) continue;
    n.act[a] = dalloc<uint16_t>(n, pix);
    n.gz[a] = dalloc<uint16_t>(n, pix);
    n.gz_planar[a] = dalloc<uint16_t>(n, planar);
  }
  for (int p = 0; p < 3; ++p) {
    const Grid g = grid_of(n, p + 1, max_batch);
    const int ch = kLayers[2 * p + 1].cout;
    n.pooled[p] = dalloc<uint16_t>(n, (long)max_batch * g.H * g.W * ch);
    n.pooled_planar[p] = dalloc<uint16_t>(n, (long)max_batch * g.H * g.wp * ch);
    n.skip[p] = dalloc<float>(n, (long)max_batch * 4 * g.H * g.W * ch);
  }
  const long pix0 = (long)max_batch * H * W;
  n.out = dalloc<float>(n, pix0);
  n.gout = dalloc<float>(n, pix0);
  n.target = dalloc<float>(n, pix0);
  n.input = dalloc<float>(n, pix0 * kInChannels);
  long part = 0;
  for (int l = 0; l < kLayerCount; ++l) {
    const long size = (long)kLayers[l].cout * (9 * kLayers[l].cin + 1);
    int most = 0, per_wave;
    for (int b = 1; b <= max_batch; ++b) most = std::max(most, grad_slices(n, l, b, per_wave));
    n.part_off[l] = part;
    part += size * most;
  }
  n.grad_part = dalloc<float>(n, part);
  n.zero = dalloc<uint16_t>(n, 32);
  n.head_part = dalloc<float>(n, kHeadBlocks * (kHeadIn + 1));
  n.loss = dalloc<float>(n, 1);
  n.energy = dalloc<float>(n, max_batch);
  for (void *p : n.allocations)
    if (p == nullptr) {
      set_error("warm-start network: device allocation failed");
      delete net;
      return nullptr;
    }
  if (hipStreamCreateWithFlags(&n.stream, hipStreamNonBlocking) != hipSuccess) {
    set_error("warm-start network: stream creation failed");
    delete net;
    return nullptr;
  }
  n.stage.make();
  for (int a = 0; a < kActs; ++a) {
    fill_zero(n, n.act_planar[a], n.planar_count[a]);
    if (a > 0) fill_zero(n, n.gz_planar[a], n.planar_count[a]);
  }
  for (int p = 0; p < 3; ++p) {
    const Grid g = grid_of(n, p + 1, max_batch);
    fill_zero(n, n.pooled_planar[p], (long)max_batch * g.H * g.wp * kLayers[2 * p + 1].cout);
  }
  fill_zero(n, n.zero, 32);
  // He-normal conv weights, zero biases, a small head
  std::mt19937_64 rng(seed);
  std::normal_distribution<float> normal(0.f, 1.f);
  std::vector<float> host(n.param_count, 0.f);
  for (int l = 0; l < kLayerCount; ++l) {
    const float sd = std::sqrt(2.f / (9.f * kLayers[l].cin));
    const size_t cnt = (size_t)kLayers[l].cout * 9 * kLayers[l].cin;
    for (size_t i = 0; i < cnt; ++i) host[n.w_off[l] + i] = normal(rng) * sd;
  }
  for (int c = 0; c < kHeadIn; ++c) host[n.head_w_off + c] = normal(rng) * 0.01f;
  if (set_params(n, host.data(), host.size()) != 0) {
    delete net;
    return nullptr;
  }
  return net;
}

void destroy(Net *net) {
  if (net == nullptr) return;
  if (net->stream) (void)hipStreamDestroy(net->stream);
  delete net;
}

static int prep_weights(Net &n) {
  k_pack_weights<<<nb((long)n.param_count), kT, 0, n.stream>>>(
      n.params, (long)n.param_count, pack_table(n), n.wbf, n.wflip);
  GCS_HIP(hipGetLastError());
  return 0;
}

int set_params(Net &n, const float *host, size_t count) {
  if (count != n.param_count) {
    set_error("warm-start network: parameter count mismatch");
    return -1;
  }
  if (stage_up(n.stage, n.stream, host, n.params, count * sizeof(float)) != 0) return -1;
  k_fill<<<nb((long)count), kT, 0, n.stream>>>(n.adam_m, (long)count, 0.f);
  k_fill<<<nb((long)count), kT, 0, n.stream>>>(n.adam_v, (long)count, 0.f);
  n.adam_t = 0;
  if (prep_weights(n) != 0) return -1;
  GCS_HIP(hipStreamSynchronize(n.stream));
  return 0;
}

int get_array(Net &n, int which, float *host, size_t count) {
  if (count != n.param_count) {
    set_error("warm-start network: parameter count mismatch");
    return -1;
  }
  return stage_down(n.stage, n.stream, which == 0 ? n.params : n.grads, host,
                    count * sizeof(float));
}

static ConvIn layer_input(const Net &n, int l) {
  const LayerSpec &L = kLayers[l];
  ConvIn in;
  if (l == 0) {
    in.f32 = n.input;
    in.c1 = L.cin;
  } else if (L.kind == IN_PLAIN) {
    in.src1 = n.act[L.src];
    in.c1 = L.cin;
  } else if (L.kind == IN_POOL) {
    in.src1 = n.pooled[(l - 2) / 2];
    in.c1 = L.cin;
  } else {
    in.src0 = n.act[L.src];
    in.c0 = act_channels(L.src);
    in.src1 = n.act[L.src2];
    in.c1 = act_channels(L.src2);
  }
  return in;
}

static int conv_tiles(const ConvWork &job) {
  return (job.cout / 32) * ((job.g.W + 15) / 16) * ((job.g.H + 1) / 2) * job.g.N;
}

static ConvWork conv_work(const ConvIn &in, const uint16_t *zero, const Grid &g, int cout,
                          const uint16_t *w, const ConvOut &o) {
  ConvWork job;
  job.in = in;
  job.in.zero = zero;
  job.g = g;
  job.cout = cout;
  job.w = w;
  job.o = o;
  return job;
}

// Forward pass over `batch` samples whose fp32 input features are already
// in n.input ([N][H][W][kInChannels]); output in n.out.
int forward_device(Net &n, int batch) {
  for (int l = 0; l < kLayerCount; ++l) {
    const LayerSpec &L = kLayers[l];
    const int lv = act_level(l + 1);
    const ConvIn in = layer_input(n, l);
    ConvOut o;
    o.g = grid_of(n, lv, batch);
    o.out = n.act[l + 1];
    o.planar = n.act_planar[l + 1];
    o.bias = n.params + n.b_off[l];
    if (l + 1 < kLayerCount && kLayers[l + 1].kind == IN_POOL) {
      o.gp = grid_of(n, lv + 1, batch);
      o.pooled = n.pooled[lv];
      o.pooled_planar = n.pooled_planar[lv];
    }
    if (l == kLayerCount - 1) {
      o.head_w = n.params + n.head_w_off;
      o.head_b = n.params + n.head_b_off;
      o.head_out = n.out;
    }
    const ConvWork job = conv_work(in, n.zero, o.g, L.cout, n.wbf + n.wbf_off[l], o);
    const int waves = conv_tiles(job) <= 1024 ? 1 : 4;
    const int blocks = (conv_tiles(job) + waves - 1) / waves, threads = 64 * waves;
    if (l == 0)
      k_conv<true, false><<<blocks, threads, 0, n.stream>>>(job);
    else if (L.kind == IN_CAT)
      k_conv<false, true><<<blocks, threads, 0, n.stream>>>(job);
    else
      k_conv<false, false><<<blocks, threads, 0, n.stream>>>(job);
  }
  GCS_HIP(hipGetLastError());
  return 0;
}

// Weight and bias gradient of layer l from gz of its output.
static GradWork grad_work(const Net &n, int l, int batch) {
  const LayerSpec &L = kLayers[l];
  const int lv = act_level(l + 1);
  const Grid g = grid_of(n, lv, batch);
  GradIn in;
  if (L.kind == IN_CAT) {
    in.src0 = n.act_planar[L.src];
    in.c0 = act_channels(L.src);
    in.g0 = grid_of(n, lv + 1, batch);
    in.src1 = n.act_planar[L.src2];
    in.c1 = act_channels(L.src2);
  } else {
    in.src1 = L.kind == IN_POOL ? n.pooled_planar[(l - 2) / 2] : n.act_planar[L.src];
    in.c1 = L.cin;
  }
  GradWork job;
  job.in = in;
  job.g = g;
  job.gz = n.gz_planar[l + 1];
  job.cout = L.cout;
  const int slices = grad_slices(n, l, batch, job.per_wave);
  job.blocks = slices * (L.cin / 16) * (L.cout / 32);
  job.part = n.grad_part + n.part_off[l];
  return job;
}

// Backward pass from n.gout (fp32, d loss / d out) of the last forward pass;
// gradients in n.grads.
int backward_device(Net &n, int batch) {
  hipStream_t s = n.stream;
  const Grid g0 = grid_of(n, 0, batch);
  k_planar_input<<<(unsigned)(batch * n.H * ((n.W + 63) / 64)), 256, 0, s>>>(n.input, g0,
                                                                            n.act_planar[0]);
  const unsigned head_blocks = std::min((unsigned)kHeadBlocks, nb((long)batch * n.H * n.W, 64));
  k_head_back<<<head_blocks, 256, 0, s>>>(n.act[kActs - 1], n.gout, g0, n.params + n.head_w_off,
                                          n.gz[kActs - 1], n.gz_planar[kActs - 1], n.head_part);
  k_head_sum<<<kHeadIn + 1, 64, 0, s>>>(n.head_part, (int)head_blocks, n.grads + n.head_w_off);
  for (int l = kLayerCount - 1; l >= 0; --l) {
    const LayerSpec &L = kLayers[l];
    const int lv = act_level(l + 1);
    const GradWork grad = grad_work(n, l, batch);
    if (l == 0) {  // no gradient for the input features
      k_wgrad<<<grad.blocks, 256, 0, s>>>(grad);
      break;
    }
    // input gradient = conv of gz with the flipped, transposed weights; its
    // epilogue leaves the masked gradient of layer l - 1's output
    const Grid g = grid_of(n, lv, batch);
    ConvIn gin;
    gin.src1 = n.gz[l + 1];
    gin.c1 = L.cout;
    ConvOut o;
    o.out = n.gz[L.src];
    o.planar = n.gz_planar[L.src];
    o.act = n.act[L.src];
    if (L.kind == IN_PLAIN) {
      o.g = g;
    } else if (L.kind == IN_POOL) {
      o.g = grid_of(n, lv - 1, batch);
      o.skip = n.skip[lv - 1];  // kept by the decoder layer of the fine grid
    } else {
      o.g = grid_of(n, lv + 1, batch);
      o.skip = n.skip[lv];
      o.c0 = act_channels(L.src);
    }
    ConvWork conv = conv_work(gin, n.zero, g, L.cin, n.wflip + n.wbf_off[l], o);
    const unsigned all = (unsigned)(grad.blocks + (conv_tiles(conv) + 3) / 4);
    if (L.kind == IN_PLAIN)
      k_backward<EP_PLAIN><<<all, 256, 0, s>>>(grad, conv);
    else if (L.kind == IN_POOL)
      k_backward<EP_POOL><<<all, 256, 0, s>>>(grad, conv);
    else
      k_backward<EP_CAT><<<all, 256, 0, s>>>(grad, conv);
  }
  SliceTable table;
  for (int l = 0; l < kLayerCount; ++l) {
    int per_wave;
    table.begin[l] = (int)n.w_off[l];
    table.slices[l] = grad_slices(n, l, batch, per_wave);
    table.part[l] = n.part_off[l];
  }
  table.begin[kLayerCount] = (int)n.head_w_off;
  k_grad_sum<<<nb((long)n.head_w_off), 256, 0, s>>>(n.grad_part, table, n.grads);
  GCS_HIP(hipGetLastError());
  return 0;
}

// Loss of n.out against n.target and its gradient into n.gout.
int loss_device(Net &n, int batch) {
  const long pix0 = (long)batch * n.H * n.W;
  k_fill<<<1, 64, 0, n.stream>>>(n.loss, 1, 0.f);
  k_mse<<<nb(pix0), kT, 0, n.stream>>>(n.out, n.target, (int)pix0, n.gout, n.loss);
  GCS_HIP(hipGetLastError());
  return 0;
}

// Per-sample relative error of n.out against n.target (training loss).
int loss_relative_device(Net &n, int batch) {
  const int P = n.H * n.W;
  k_fill<<<1, 64, 0, n.stream>>>(n.loss, 1, 0.f);
  k_sample_energy<<<batch, kT, 0, n.stream>>>(n.target, P, n.energy);
  k_mse_rel<<<nb((long)batch * P), kT, 0, n.stream>>>(n.out, n.target, batch, P, n.energy,
                                                      n.gout, n.loss);
  GCS_HIP(hipGetLastError());
  return 0;
}

int adam_device(Net &n, float lr) {
  const float b1 = 0.9f, b2 = 0.999f;
  ++n.adam_t;
  const float c1 = 1.f - std::pow(b1, (float)n.adam_t);
  const float c2 = 1.f - std::pow(b2, (float)n.adam_t);
  k_adam<<<nb((long)n.param_count), kT, 0, n.stream>>>(
      n.params, n.grads, n.adam_m, n.adam_v, (long)n.param_count, lr, b1, b2, c1, c2, 1e-8f,
      pack_table(n), n.wbf, n.wflip);
  GCS_HIP(hipGetLastError());
  return 0;
}

int check_batch(const Net &n, int batch) {
  if (batch <= 0 || batch > n.max_batch) {
    set_error("warm-start network: batch outside [1, max_batch]");
    return -1;
  }
  return 0;
}

int gemm_check(const uint16_t *A, const uint16_t *B, int M, int N, int K, float *C) {
  if (M % 16 || N % 16 || K % 16 || M <= 0 || N <= 0 || K <= 0) {
    set_error("gemm check: sizes must be positive multiples of 16");
    return -1;
  }
  uint16_t *dA = nullptr, *dB = nullptr;
  float *dC = nullptr;
  GCS_HIP(hipMalloc(&dA, (size_t)M * K * 2));
  GCS_HIP(hipMalloc(&dB, (size_t)K * N * 2));
  GCS_HIP(hipMalloc(&dC, (size_t)M * N * 4));
  GCS_HIP(hipMemcpy(dA, A, (size_t)M * K * 2, hipMemcpyHostToDevice));
  GCS_HIP(hipMemcpy(dB, B, (size_t)K * N * 2, hipMemcpyHostToDevice));
  k_gemm_check<<<dim3(M / 16, N / 16), 64>>>(dA, dB, M, N, K, dC);
  GCS_HIP(hipGetLastError());
  GCS_HIP(hipMemcpy(C, dC, (size_t)M * N * 4, hipMemcpyDeviceToHost));
  (void)hipFree(dA);
  (void)hipFree(dB);
  (void)hipFree(dC);
  return 0;
}

}  // namespace unet
}  // namespace gcs
