// rtm_cnn.hip -- a small image-domain deblurring network for migrated images
// (not in the reference): 3x3 convolutions with bias and ReLU, a residual
// connection from input channel 0, trained with Adam on mean-squared error.
// Layers may be dilated (tap offsets times the layer's dilation), which
// widens the receptive field at the same cost.
// Convolutions run on gfx950's matrix cores: operands in BF16, accumulation
// in FP32 (v_mfma_f32_16x16x32_bf16, K = 32 per instruction); master
// weights, Adam state, loss and gradient reductions stay FP32 / FP64.
//
// Layouts.  Activations are NHWC in BF16 with the channel count padded to a
// multiple of 8 (Cp), so the eight consecutive K values a lane feeds the
// MFMA are one 16-byte load.  Convolution as an implicit GEMM: M = 16 output
// channels, N = 16 consecutive pixels of one row, K = 9 taps x Cp
// input channels (k = tap*Cp + ci, padded to a multiple of 32).  The MFMA
// lane layout: A[m][k] at lane m + 16*(k/8), element k%8; B[k][n] at lane
// n + 16*(k/8), element k%8; D[m][n] at lane n + 16*(m/4), element m%4.
//
//   forward      z = conv(a, W) + b; hidden layers store relu(z) in BF16,
//                the last layer y = z + x0 in FP32
//   input grad   dz_prev = conv(dz, W flipped and transposed) * (a > 0)
//   weight grad  dW[tap][co][ci] = sum_pix dz[pix][co] * a[pix + tap][ci]:
//                M = co, N = ci, K = pixels, transposed on the way out of LDS;
//                each workgroup accumulates a range of rows and writes one
//                partial, a reduction kernel adds the partials in a fixed
//                order (FP64), so the result does not depend on scheduling.
// Channel counts above 16 run in blocks of 16 (two blocks of output channels
// per convolution wave; four 16 x 16 blocks per weight-gradient workgroup).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <new>
#include <string>
#include <vector>

#include "../../include/rtm_cnn.h"

namespace {

typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef unsigned short bf16;

constexpr int MAXC = 32;                    // channels per layer (two blocks of 16)
constexpr int MAXL = 16;                    // layers
constexpr int WG_STRIDE = 9 * MAXC * MAXC + MAXC;  // weight-grad partials per workgroup
constexpr int WG_GROUPS = 1024;             // most workgroups of one weight-gradient launch
constexpr int WG_LEVEL1 = 32;               // groups of the reduction
// Byte offsets into an activation (MAX_PIXELS x 32 channels x 2 bytes) stay
// below 2^31, the range of a buffer load's offset.
constexpr long long MAX_PIXELS = 1LL << 25;

__device__ __forceinline__ bf16 to_bf16(float f) {  // round to nearest even
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}
__device__ __forceinline__ float from_bf16(bf16 h) { return __uint_as_float(((unsigned)h) << 16); }


// Buffer resources: a load whose offset is out of range (kDrop) returns zero,
// which is the convolution's zero padding without a branch around the load.
typedef __amdgpu_buffer_rsrc_t Rsrc;
constexpr unsigned kDrop = 0x80000000u;
__device__ __forceinline__ Rsrc rsrc(const void* base, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ u32x4 bld16(Rsrc r, unsigned vo) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, (int)vo, 0, 0);
}

// mode 0: hidden layer (bias, ReLU, BF16 NHWC out); mode 1: last layer (bias
// + residual, FP32 out channel 0); mode 2: input gradient (mask by act > 0).
struct ConvArgs {
  const bf16* in;     // NHWC, cin_p channels
  const bf16* wt;     // [MAXC][kpad]
  const float* bias;  // [MAXC] (modes 0, 1)
  bf16* out;          // NHWC, cout_p channels (modes 0, 2)
  float* out32;       // [n][h][w] (mode 1)
  const float* resid; // [n][h][w] (mode 1)
  const bf16* mask;   // NHWC, cout_p channels (mode 2)
  int n, h, w, cin_p, kpad, cout_p, mode;
  int ncob;           // blocks of 16 output channels
  int ch;             // k_conv_rows: output rows of a strip
  int dil;            // dilation: tap (ky, kx) reads (y + (ky-1)*dil, x + (kx-1)*dil)
};

// The weights are the first MFMA operand and the pixels the second, so a lane
// ends with four consecutive channels of one pixel: D[channel 4 kg + j][pixel
// lane & 15], stored as 8 bytes (one channel a lane and 2-byte stores bound the
// convolution before: 94 us a 32 x 32 layer at 256 x 64 x 64).
template <int NCOB>
struct ConvOut {
  float bias[NCOB][4];
  __device__ __forceinline__ void load(const ConvArgs& a, int kg) {
#pragma unroll
    for (int cb = 0; cb < NCOB; ++cb)
#pragma unroll
      for (int j = 0; j < 4; ++j) bias[cb][j] = a.mode == 2 ? 0.0f : a.bias[cb * 16 + 4 * kg + j];
  }
  // What a tile's epilogue reads besides the accumulators, fetched a tile ahead:
  // the activations that mask an input gradient, or the residual.
  struct Extra {
    u32x2 mk[NCOB];
    float res;
  };
  // px: pixel of the row; p: its index in the batch
  static __device__ __forceinline__ void fetch(const ConvArgs& a, int kg, bool ok, unsigned p,
                                               Extra& e) {
    if (a.mode == 2) {
#pragma unroll
      for (int cb = 0; cb < NCOB; ++cb) {
        const int co = cb * 16 + 4 * kg;
        if (ok && co < a.cout_p)
          e.mk[cb] = *reinterpret_cast<const u32x2*>(a.mask + (size_t)p * a.cout_p + co);
      }
    } else if (a.mode == 1) {
      if (ok && kg == 0) e.res = a.resid[p];
    }
  }
  __device__ __forceinline__ void store(const ConvArgs& a, const f4* acc, int kg, int px, unsigned p,
                                        const Extra& e) const {
    if (px >= a.w) return;
    if (a.mode == 1) {
      if (kg == 0) a.out32[p] = (acc[0][0] + bias[0][0]) + e.res;
      return;
    }
#pragma unroll
    for (int cb = 0; cb < NCOB; ++cb) {
      const int co = cb * 16 + 4 * kg;
      if (co >= a.cout_p) continue;
      bf16 v[4];
      if (a.mode == 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = to_bf16(fmaxf(acc[cb][j] + bias[cb][j], 0.0f));
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          v[j] = to_bf16(from_bf16((bf16)(e.mk[cb][j >> 1] >> (16 * (j & 1)))) > 0.0f ? acc[cb][j]
                                                                                     : 0.0f);
      }
      *reinterpret_cast<u32x2*>(a.out + (size_t)p * a.cout_p + co) =
          u32x2{(unsigned)v[0] | ((unsigned)v[1] << 16), (unsigned)v[2] | ((unsigned)v[3] << 16)};
    }
  }
};

// Weight-stationary convolution of narrow inputs (8, 16 or 24 channels): a wave
// holds its weights (all NK K-steps of NCOB blocks of 16 output channels) in
// registers and walks 16-pixel row tiles, the next tile's inputs in flight where
// there is one (the addresses of one that is not there cost a wave with a single
// tile: five layers of 16 channels at 32 x 64 x 64 0.195 ms a call, 0.183 without).
// K-step ks covers k = 32 ks .. 32 ks + 31; lane group kg feeds k = 32 ks +
// 8 kg .. +7, eight consecutive channels of one tap (cin_p is a multiple of 8).
template <int NK, int NCOB>
__global__ __launch_bounds__(256) void k_conv(const ConvArgs a) {
  const int lane = threadIdx.x & 63;
  const int m = lane & 15, kg = lane >> 4;
  b8 wv[NCOB][NK];
#pragma unroll
  for (int cb = 0; cb < NCOB; ++cb)
#pragma unroll
    for (int ks = 0; ks < NK; ++ks)
      wv[cb][ks] = *reinterpret_cast<const b8*>(a.wt + (cb * 16 + m) * a.kpad + ks * 32 + 8 * kg);
  ConvOut<NCOB> co;
  co.load(a, kg);
  int tdy[NK], tdx[NK], tci[NK];
  bool tok[NK];
#pragma unroll
  for (int ks = 0; ks < NK; ++ks) {
    const int k = ks * 32 + 8 * kg, tap = k / a.cin_p;
    tok[ks] = tap < 9;
    tdy[ks] = (tap / 3 - 1) * a.dil;
    tdx[ks] = (tap % 3 - 1) * a.dil;
    tci[ks] = k - tap * a.cin_p;
  }
  const unsigned hw = (unsigned)(a.h * a.w);
  const Rsrc RI = rsrc(a.in, (unsigned)a.n * hw * (unsigned)a.cin_p * 2u);
  const unsigned segs = (unsigned)(a.w + 15) >> 4;
  const unsigned tiles = (unsigned)(a.n * a.h) * segs;
  const unsigned step = gridDim.x * 4u;
  auto fetch = [&](unsigned t, b8* av, typename ConvOut<NCOB>::Extra& e) {
    const unsigned row = t / segs, seg = t - row * segs;
    const unsigned nn = row / (unsigned)a.h;
    const int y = (int)(row - nn * (unsigned)a.h), x = (int)seg * 16 + m;
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      const int yy = y + tdy[ks], xx = x + tdx[ks];
      const bool ok = t < tiles && tok[ks] && yy >= 0 && yy < a.h && xx >= 0 && xx < a.w;
      const unsigned vo =
          ok ? ((nn * hw + (unsigned)(yy * a.w + xx)) * (unsigned)a.cin_p + (unsigned)tci[ks]) * 2u
             : kDrop;
      av[ks] = __builtin_bit_cast(b8, bld16(RI, vo));
    }
    ConvOut<NCOB>::fetch(a, kg, t < tiles && x < a.w, row * (unsigned)a.w + (unsigned)x, e);
  };
  unsigned t = blockIdx.x * 4u + (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  b8 av[NK], nx[NK];
  typename ConvOut<NCOB>::Extra e{}, en{};
  fetch(t, av, e);
  for (; t < tiles; t += step) {
    if (t + step < tiles) fetch(t + step, nx, en);
    f4 acc[NCOB];
#pragma unroll
    for (int cb = 0; cb < NCOB; ++cb) acc[cb] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < NK; ++ks)
#pragma unroll
      for (int cb = 0; cb < NCOB; ++cb)
        acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[cb][ks], av[ks], acc[cb], 0, 0, 0);
    const unsigned row = t / segs;
    const int px = (int)(t - row * segs) * 16 + m;
    co.store(a, acc, kg, px, row * (unsigned)a.w + (unsigned)px, e);
    e = en;
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) av[ks] = nx[ks];
  }
}

// Convolution of 32-channel inputs: a tap is one K-step, so the three
// column-shifted operands of an input row serve the output rows above, on and
// below it.  A wave marches down a strip of 16 columns and `ch` output rows
// (rows dil apart), loading three operands a row instead of nine; the rows in
// use and three rows of look-ahead sit in a circular register buffer.  Bound by
// memory: at 256 x 64 x 64 and 32 x 32 channels 41 us a launch (104 us with nine
// loads a tile and 2-byte stores), against 25 us for its 134 MB (37 us for an
// input gradient, which reads the mask) at the streaming rate.  Three waves per
// SIMD and two rows of look-ahead measured 42 us, two waves with two rows 53.
template <int NCOB>
__global__ __launch_bounds__(256, 2) void k_conv_rows(const ConvArgs a) {
  constexpr int NB = 6;  // rows i-1, i, i+1 and three in flight
  const int lane = threadIdx.x & 63;
  const int m = lane & 15, kg = lane >> 4;
  const int wvi = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  b8 wv[NCOB][9];
#pragma unroll
  for (int cb = 0; cb < NCOB; ++cb)
#pragma unroll
    for (int t = 0; t < 9; ++t)
      wv[cb][t] = *reinterpret_cast<const b8*>(a.wt + (cb * 16 + m) * a.kpad + t * 32 + 8 * kg);
  ConvOut<NCOB> co;
  co.load(a, kg);
  const int d = a.dil, segs = (a.w + 15) >> 4;
  const int per = (a.h + d - 1) / d, chunks = (per + a.ch - 1) / a.ch;  // rows of a residue class
  const unsigned hw = (unsigned)(a.h * a.w);
  const Rsrc RI = rsrc(a.in, (unsigned)a.n * hw * 64u);
  const unsigned strips = (unsigned)(a.n * d * chunks * segs);
  for (unsigned s = blockIdx.x * 4u + (unsigned)wvi; s < strips; s += gridDim.x * 4u) {
    const unsigned q = s / (unsigned)segs, q2 = q / (unsigned)chunks, nn = q2 / (unsigned)d;
    const int x = (int)(s - q * (unsigned)segs) * 16 + m;
    const int i0 = (int)(q - q2 * (unsigned)chunks) * a.ch, r = (int)(q2 - nn * (unsigned)d);
    const int i1 = min(i0 + a.ch, (a.h - r + d - 1) / d);
    unsigned vo[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int xx = x + (k - 1) * d;
      vo[k] = xx >= 0 && xx < a.w ? ((unsigned)xx * 32u + 8u * (unsigned)kg) * 2u : kDrop;
    }
    b8 buf[NB][3];
    auto fetch = [&](int i, b8* row) {  // row r + d*i of image nn, zero outside it
      const int y = r + d * i;
      const bool ok = i <= i1 && y >= 0 && y < a.h;
      const unsigned so = ok ? (nn * hw + (unsigned)(y * a.w)) * 64u : 0u;
#pragma unroll
      for (int k = 0; k < 3; ++k)
        row[k] = __builtin_bit_cast(
            b8, __builtin_amdgcn_raw_buffer_load_b128(RI, (int)(ok ? vo[k] : kDrop), (int)so, 0));
    };
    const auto pix = [&](int i) { return nn * hw + (unsigned)((r + d * i) * a.w + x); };
    typename ConvOut<NCOB>::Extra e{}, en{};
    ConvOut<NCOB>::fetch(a, kg, i0 < i1 && x < a.w, pix(i0), e);
#pragma unroll
    for (int b = 0; b < NB - 1; ++b) fetch(i0 - 1 + b, buf[b]);
    for (int base = i0; base < i1; base += NB) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int i = base + j;
        if (i >= i1) break;
        ConvOut<NCOB>::fetch(a, kg, i + 1 < i1 && x < a.w, pix(i + 1), en);
        fetch(i + NB - 2, buf[(j + NB - 1) % NB]);
        __builtin_amdgcn_sched_barrier(0);  // the look-ahead is issued before the products
        f4 acc[NCOB];
#pragma unroll
        for (int cb = 0; cb < NCOB; ++cb) acc[cb] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
          for (int cb = 0; cb < NCOB; ++cb)
            acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[cb][t], buf[(j + t / 3) % NB][t % 3],
                                                              acc[cb], 0, 0, 0);
        co.store(a, acc, kg, x, pix(i), e);
        e = en;
      }
    }
  }
}

// Weight / bias gradient partials of a range of image rows per workgroup.
struct WgradArgs {
  const bf16* dz;   // NHWC, dz_p channels
  const bf16* act;  // NHWC, act_p channels (the layer input)
  float* part;      // [groups][WG_STRIDE]
  int n, h, w, dz_p, act_p, dil;
  int rows_per;     // image rows (over n*h) of one workgroup
  int pw;           // pixels of a staged panel of a row (a multiple of 32)
};

// dW[tap][co][ci] = sum_pix dz[pix][co] act[pix + tap][ci] as MFMAs with
// M = co, N = ci, K = 32 pixels of one row.  Both operands need eight
// consecutive pixels of one channel per lane where memory holds the channels of
// a pixel together: rows are staged as they are and read with the transposing
// LDS load (ds_read_b64_tr_b16: of 16 lanes, lanes 4i .. 4i+3 address the 16
// channels of pixel i and lane l receives channel l of the four pixels), which
// serves all nine taps from one copy, each at its own pixel offset.
//
// A workgroup takes a range of image rows; per row and 32-pixel chunk every
// wave multiplies its taps of one block of 16 input channels with all output
// channels, and the accumulators run over all rows.  With RING (no dilation,
// rows up to WG_RING_W pixels) each row of the layer input is staged once and
// stays for the next two; otherwise the three rows of every panel of `pw`
// pixels are staged.  The next unit's rows are in flight meanwhile.  One
// partial per workgroup; the reduction adds them in a fixed order.
//
// Measured over the six layers of a 32-channel network at 256 x 64 x 64: 43 us
// a launch (59 with three waves per SIMD, which left a fourth round of the 1024
// workgroups; 132 when nine tap-shifted copies of each chunk were transposed by
// 2-byte LDS stores), against 25 us for the 134 MB of a 32 x 32 layer.
constexpr int WG_RING_W = 128;  // widest row of the ring (50 KB of LDS)

// Byte offset in a staged row of channel block half (16 channels), pixel p: 64
// bytes a pixel, the halves swapped in every second group of eight pixels so
// that the lanes of a transposing load, eight pixels apart, meet other banks.
__device__ __forceinline__ unsigned stage_off(int p, int half) {
  return (unsigned)(p * 64 + ((half ^ ((p >> 3) & 1)) << 5));
}

template <bool RING>
__global__ __launch_bounds__(256, RING ? 4 : 2) void k_wgrad(const WgradArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int NA = RING ? 3 : 8, NZ = RING ? 2 : 1;  // 16-byte loads per thread and unit
  constexpr int NACT = RING ? 4 : 6;  // staged act rows: a ring of four, or two sets of three
  const int tid = threadIdx.x, lane = tid & 63;
  const int wvi = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, kg = lane >> 4;
  const int R = a.n * a.h, d = a.dil;
  const int r0 = blockIdx.x * a.rows_per, r1 = min(R, r0 + a.rows_per);
  const int sp = (a.pw + 2 * d + 15) & ~15;  // pixels of a staged act row
  unsigned char* const sz = lds + NACT * sp * 64;  // two dz rows of pw pixels
  const int cvz = a.dz_p >> 3, cva = a.act_p >> 3;
  const int ncob = (a.dz_p + 15) >> 4, ncib = (a.act_p + 15) >> 4;
  // the wave's taps [tap0, tap0 + ntap) of input channel block cib
  const int cib = ncib == 2 ? wvi & 1 : 0;
  const int tap0 = ncib == 2 ? (wvi >> 1) * 5 : (wvi == 0 ? 0 : 1 + 2 * wvi);
  const int ntap = ncib == 2 ? 5 - (wvi >> 1) : (wvi == 0 ? 3 : 2);
  f4 acc[5][2];
#pragma unroll
  for (int t = 0; t < 5; ++t) acc[t][0] = acc[t][1] = f4{0.f, 0.f, 0.f, 0.f};
  float bsum[2] = {0.f, 0.f};

  const unsigned wz = (unsigned)a.w * (unsigned)a.dz_p * 2u, wa = (unsigned)a.w * (unsigned)a.act_p * 2u;
  const Rsrc RZ = rsrc(a.dz, (unsigned)R * wz), RA = rsrc(a.act, (unsigned)R * wa);
  // staging items of the thread, the same for every unit: source offset from
  // the row's panel, LDS offset, the act row (0 .. 2 with full staging)
  const int arows = RING ? 1 : 3, apx = a.pw + 2 * d;
  int apos[NA], arow[NA], zpos[NZ];
  unsigned alds[NA], zlds[NZ], acg[NA], zcg[NZ];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int e = tid + i * 256, q = e / cva, row = q / apx;
    arow[i] = row < arows ? row : -1;
    apos[i] = q - row * apx;  // pixel x0 - d + apos
    const int cg = e - q * cva;
    acg[i] = (unsigned)cg * 16u;
    alds[i] = stage_off(apos[i], cg >> 1) + (unsigned)(cg & 1) * 16u;
  }
#pragma unroll
  for (int i = 0; i < NZ; ++i) {
    const int e = tid + i * 256, q = e / cvz, cg = e - q * cvz;
    zpos[i] = q < a.pw ? q : -1;
    zcg[i] = (unsigned)cg * 16u;
    zlds[i] = stage_off(q, cg >> 1) + (unsigned)(cg & 1) * 16u;
  }
  u32x4 la[NA], lz[NZ];
  const auto load_act = [&](int row, int x0) {  // rows row, row + d, row + 2d (RING: row)
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int rr = row + arow[i] * d, x = x0 - d + apos[i];
      const bool ok = arow[i] >= 0 && rr >= 0 && rr < R && x >= 0 && x < a.w;
      la[i] = bld16(RA, ok ? (unsigned)rr * wa + (unsigned)(x * a.act_p) * 2u + acg[i] : kDrop);
    }
  };
  const auto load_dz = [&](int row, int x0) {
#pragma unroll
    for (int i = 0; i < NZ; ++i) {
      const int x = x0 + zpos[i];
      const bool ok = zpos[i] >= 0 && row < r1 && x < a.w;
      lz[i] = bld16(RZ, ok ? (unsigned)row * wz + (unsigned)(x * a.dz_p) * 2u + zcg[i] : kDrop);
    }
  };
  const auto put_act = [&](int slot) {
#pragma unroll
    for (int i = 0; i < NA; ++i)
      if (arow[i] >= 0)
        *reinterpret_cast<u32x4*>(lds + (slot + arow[i]) * sp * 64 + alds[i]) = la[i];
  };
  const auto put_dz = [&](int slot) {
#pragma unroll
    for (int i = 0; i < NZ; ++i)
      if (zpos[i] >= 0) *reinterpret_cast<u32x4*>(sz + slot * a.pw * 64 + zlds[i]) = lz[i];
  };
  const auto tr = [&](const unsigned char* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4*)p);
  };
  const auto pair = [&](s4 lo, s4 hi) {
    return __builtin_bit_cast(b8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  // lane offsets of the operands' two loads (pixels 8 kg + 0..3 and + 4..7)
  unsigned oz[2][2], oa[5][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int p = 8 * kg + 4 * h + (m >> 2);
    const unsigned c = (unsigned)(m & 3) * 8u;
    oz[0][h] = stage_off(p, 0) + c;
    oz[1][h] = stage_off(p, 1) + c;
#pragma unroll
    for (int t = 0; t < 5; ++t) oa[t][h] = stage_off(p + ((tap0 + t) % 3) * d, cib) + c;
  }

  const int panels = (a.w + a.pw - 1) / a.pw;
  int r = r0, x0 = 0, u = 0;
  if (RING) {  // rows r0-1 and r0, then r0+1 with the first dz row
    load_act(r0 - 1, 0);
    put_act((r0 + 3) & 3);
    load_act(r0, 0);
    put_act(r0 & 3);
    load_act(r0 + 1, 0);
    put_act((r0 + 1) & 3);
  } else {
    load_act(r0 - d, 0);
    put_act(0);
  }
  load_dz(r0, 0);
  put_dz(0);
  __syncthreads();
  while (r < r1) {
    int rn = r, xn = x0 + a.pw;  // the next unit
    if (xn >= panels * a.pw) { xn = 0; ++rn; }
    if (RING) load_act(rn + 1, 0);
    else load_act(rn - d, xn);
    load_dz(rn, xn);
    __builtin_amdgcn_sched_barrier(0);
    const int y = r % a.h;
    const int chunks = (min(a.pw, a.w - x0) + 31) >> 5;
    if (cib < ncib) {
      for (int c = 0; c < chunks; ++c) {
        const unsigned char* pz = sz + (u & 1) * a.pw * 64 + c * 2048;
        s4 zr[2][2];
        b8 av[2];
#pragma unroll
        for (int cob = 0; cob < 2; ++cob) {
          if (cob < ncob) {
            zr[cob][0] = tr(pz + oz[cob][0]);
            zr[cob][1] = tr(pz + oz[cob][1]);
            av[cob] = pair(zr[cob][0], zr[cob][1]);
          }
        }
#pragma unroll
        for (int t = 0; t < 5; ++t) {
          const int ky = (tap0 + t) / 3 - 1, yy = y + ky * d;
          if (t < ntap && yy >= 0 && yy < a.h) {
            const int slot = RING ? (r + ky) & 3 : (u & 1) * 3 + ky + 1;
            const unsigned char* pa = lds + slot * sp * 64 + c * 2048;
            const b8 bv = pair(tr(pa + oa[t][0]), tr(pa + oa[t][1]));
            acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[0], bv, acc[t][0], 0, 0, 0);
            if (ncob == 2)
              acc[t][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[1], bv, acc[t][1], 0, 0, 0);
          }
        }
        if (wvi == 0) {
#pragma unroll
          for (int cob = 0; cob < 2; ++cob) {
            if (cob < ncob) {
              const u32x4 w4 = __builtin_bit_cast(u32x4, av[cob]);
#pragma unroll
              for (int j = 0; j < 4; ++j)
                bsum[cob] += __uint_as_float(w4[j] << 16) + __uint_as_float(w4[j] & 0xffff0000u);
            }
          }
        }
      }
    }
    // the slots written hold no row that this unit reads: RING row r+2 (mod 4),
    // otherwise the other set
    ++u;
    if (RING) put_act((rn + 1) & 3);
    else put_act((u & 1) * 3);
    put_dz(u & 1);
    __syncthreads();
    r = rn;
    x0 = xn;
  }
  if (cib >= ncib) return;
  float* P = a.part + (long long)blockIdx.x * WG_STRIDE;
  const int ci = cib * 16 + m;
#pragma unroll
  for (int t = 0; t < 5; ++t)
#pragma unroll
    for (int cob = 0; cob < 2; ++cob)
      if (t < ntap && cob < ncob)
#pragma unroll
        for (int j = 0; j < 4; ++j)  // D[m = co][n = ci]: co = cob*16 + 4 kg + j
          P[((tap0 + t) * MAXC + cob * 16 + 4 * kg + j) * MAXC + ci] = acc[t][cob][j];
  // bias: lanes m, m+16, m+32, m+48 hold pixels of channel cob*16 + m
#pragma unroll
  for (int cob = 0; cob < 2; ++cob) {
    float b = bsum[cob];
    b += __shfl_xor(b, 16);
    b += __shfl_xor(b, 32);
    if (wvi == 0 && kg == 0 && cob < ncob) P[9 * MAXC * MAXC + cob * 16 + m] = b;
  }
}

// Deterministic two-level sum of the workgroup partials into the layer's
// gradient (W[co][ci][ky][kx] then b[co]): group g adds its share of the
// partials in order (FP64), then the groups are added in order.  A block takes
// the 32 input channels of one tap and output channel (one 128-byte line of
// every partial), or the 32 biases; thread (g, ci).
__global__ __launch_bounds__(32 * WG_LEVEL1) void k_wgrad_reduce(const float* part, int P, int cin,
                                                                 int cout, float* grad) {
  __shared__ double sh[WG_LEVEL1][32];
  const int ci = threadIdx.x & 31, g = threadIdx.x >> 5;
  const int G = min(WG_LEVEL1, P);
  const int tc = blockIdx.x;  // tap * cout + co; 9 * cout: the biases
  const bool bias = tc == 9 * cout;
  const int t = tc / cout, co = tc - t * cout;
  const int src = bias ? 9 * MAXC * MAXC + ci : (t * MAXC + co) * MAXC + ci;
  const bool on = bias ? ci < cout : ci < cin;
  double s = 0.0;
  if (g < G && on) {
    const int p0 = (int)((long long)P * g / G), p1 = (int)((long long)P * (g + 1) / G);
#pragma unroll 8
    for (int p = p0; p < p1; ++p) s += (double)part[(long long)p * WG_STRIDE + src];
  }
  sh[g][ci] = s;
  __syncthreads();
  if (g == 0 && on) {
    double v = 0.0;
    for (int i = 0; i < G; ++i) v += sh[i][ci];
    grad[bias ? cout * cin * 9 + ci : (co * cin + ci) * 9 + t] = (float)v;
  }
}

// Eight BF16 channels of a pixel as one 16-byte store; get(c): channel c.
template <typename F>
__device__ __forceinline__ void put8(bf16* dst, const F& get) {
  u32x4 v;
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = (unsigned)get(2 * k) | ((unsigned)get(2 * k + 1) << 16);
  *reinterpret_cast<u32x4*>(dst) = v;
}

// NCHW FP32 input -> NHWC BF16 (cp channels) and the FP32 residual channel 0.
// With an order (training batch from the device-resident set), image i of the
// batch is set entry order[b0 + i] and its target goes to t32.
__global__ void k_pack_input(const float* x, long long npix, int hw, int cin, int cp, bf16* act,
                             float* resid, const int* order, int b0, const float* t, float* t32) {
  for (long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x; p < npix;
       p += (long long)gridDim.x * blockDim.x) {
    const long long i = p / hw, q = p - i * hw;
    const long long nn = order ? order[b0 + i] : i;
    const float* px = x + nn * cin * hw + q;
    for (int c = 0; c < cp; c += 8)
      put8(act + p * cp + c, [&](int k) {
        return c + k < cin ? to_bf16(px[(long long)(c + k) * hw]) : (bf16)0;
      });
    resid[p] = px[0];
    if (order) t32[p] = t[nn * hw + q];
  }
}

// Loss gradient of mean((y - t)^2): dz = 2(y - t)/npix in BF16 channel 0 of
// a cp-channel NHWC array; diff = y - t for the loss.
__global__ void k_loss_grad(const float* y, const float* t, long long npix, int cp, float scale,
                            bf16* dz, float* diff) {
  for (long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x; p < npix;
       p += (long long)gridDim.x * blockDim.x) {
    const float d = y[p] - t[p];
    diff[p] = d;
    for (int c = 0; c < cp; c += 8)
      put8(dz + p * cp + c, [&](int k) { return c + k == 0 ? to_bf16(scale * d) : (bf16)0; });
  }
}

__global__ void k_adam(float* p, const float* g, float* m, float* v, int n, float lr, float b1,
                       float b2, float eps, float c1, float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * (gi * gi);
  m[i] = mi;
  v[i] = vi;
  p[i] = p[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

// FP32 params -> BF16 forward weights [32][kf] (k = tap*cin_p + ci),
// backward-data weights [32][kb] (row ci, k = tap'*cout_p + co with the flipped
// tap 8 - tap) and the padded bias, of layer blockIdx.y.
struct PackLayer {
  const float* prm;
  bf16 *wf, *wb;
  float* bias;
  int cin, cout, cin_p, cout_p, kf, kb;
};
struct PackArgs {
  PackLayer l[MAXL];
};
__global__ void k_pack_weights(const PackArgs a) {
  const PackLayer& l = a.l[blockIdx.y];
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < MAXC * l.kf) {
    const int co = e / l.kf, k = e % l.kf, tap = k / l.cin_p, ci = k % l.cin_p;
    float v = 0.0f;
    if (co < l.cout && ci < l.cin && tap < 9) v = l.prm[(co * l.cin + ci) * 9 + tap];
    l.wf[e] = to_bf16(v);
  }
  if (e < MAXC * l.kb) {
    const int ci = e / l.kb, k = e % l.kb, tp = k / l.cout_p, co = k % l.cout_p;
    float v = 0.0f;
    if (ci < l.cin && co < l.cout && tp < 9) v = l.prm[(co * l.cin + ci) * 9 + (8 - tp)];
    l.wb[e] = to_bf16(v);
  }
  if (e < MAXC) l.bias[e] = e < l.cout ? l.prm[l.cout * l.cin * 9 + e] : 0.0f;
}

// FP64 sum of squares (fixed order: block partials, then one block).
__global__ __launch_bounds__(256) void k_sumsq(const float* d, long long n, double* part) {
  __shared__ double sh[256];
  double s = 0.0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    s += (double)d[i] * (double)d[i];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

inline int pad8(int c) { return (c + 7) & ~7; }
inline int pad32(int k) { return (k + 31) & ~31; }
inline unsigned nblk(long long n, int per = 256, long long cap = 8192) {
  long long b = (n + per - 1) / per;
  if (b < 1) b = 1;
  return (unsigned)(b > cap ? cap : b);
}

}  // namespace

struct rtm_cnn {
  int L = 0;
  int c[MAXL + 1] = {0};
  int cp[MAXL + 1] = {0};
  int kf[MAXL] = {0}, kb[MAXL] = {0};
  int dil[MAXL] = {0};
  int off[MAXL + 1] = {0};  // parameter offsets per layer
  int np = 0;
  long long cap_pix = 0, cap_rows = 0;
  hipStream_t stream = nullptr;
  std::string err;
  std::vector<void*> allocs;
  float *prm = nullptr, *grad = nullptr, *am = nullptr, *av = nullptr;
  bf16* wf[MAXL] = {nullptr};
  bf16* wb[MAXL] = {nullptr};
  float* bias[MAXL] = {nullptr};
  bf16* act[MAXL] = {nullptr};  // act[l]: input of layer l, NHWC cp[l]
  bf16* dz[MAXL] = {nullptr};   // dz[l]: gradient at the output of layer l, NHWC cp[l+1]
  float *x32 = nullptr, *resid = nullptr, *y32 = nullptr, *t32 = nullptr, *diff = nullptr;
  float* part = nullptr;    // weight-gradient partials [WG_GROUPS][WG_STRIDE]
  double* sq = nullptr;
  int adam_t = 0;
  bool grad_ok = false;
  // device-resident training set
  float *ds_x = nullptr, *ds_t = nullptr;
  int* ds_order = nullptr;
  double* ds_sq = nullptr;  // loss partial sums of up to LOSS_BATCHES batches
  int ds_nb = 0;
  long long ds_cap = 0;
  int ds_n = 0;
};

namespace {

int cfail(rtm_cnn* c, int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  if (c) c->err = buf;
  return code;
}

#define CNNCHK(c, expr)                                                                  \
  do {                                                                                   \
    hipError_t e_ = (expr);                                                              \
    if (e_ != hipSuccess) return cfail((c), RTM_CNN_E_HIP, "%s: %s", #expr, hipGetErrorString(e_)); \
  } while (0)

template <typename T>
int calloc_dev(rtm_cnn* c, T** p, size_t count) {
  void* q = nullptr;
  if (count == 0) count = 1;
  hipError_t e = hipMalloc(&q, count * sizeof(T));
  if (e != hipSuccess) return cfail(c, RTM_CNN_E_NOMEM, "hipMalloc(%zu): %s", count * sizeof(T), hipGetErrorString(e));
  c->allocs.push_back(q);
  *p = static_cast<T*>(q);
  return RTM_CNN_OK;
}

// Release one allocation made by calloc_dev before the network is destroyed.
template <typename T>
void cfree_dev(rtm_cnn* c, T** p) {
  if (!*p) return;
  for (size_t i = 0; i < c->allocs.size(); ++i)
    if (c->allocs[i] == static_cast<void*>(*p)) {
      c->allocs.erase(c->allocs.begin() + i);
      break;
    }
  (void)hipFree(*p);
  *p = nullptr;
}

int check_shape(rtm_cnn* c, int n, int h, int w) {
  if (n < 1 || h < 1 || w < 1) return cfail(c, RTM_CNN_E_ARG, "shape %d x %d x %d", n, h, w);
  if ((long long)n * h * w > c->cap_pix) return cfail(c, RTM_CNN_E_ARG, "%lld pixels > capacity %lld", (long long)n * h * w, c->cap_pix);
  if ((long long)n * h > c->cap_rows) return cfail(c, RTM_CNN_E_ARG, "%lld rows > capacity %lld", (long long)n * h, c->cap_rows);
  return RTM_CNN_OK;
}

int pack_weights(rtm_cnn* c) {
  PackArgs a{};
  int most = 0;
  for (int l = 0; l < c->L; ++l) {
    a.l[l] = PackLayer{c->prm + c->off[l], c->wf[l], c->wb[l], c->bias[l], c->c[l], c->c[l + 1],
                       c->cp[l], c->cp[l + 1], c->kf[l], c->kb[l]};
    most = std::max(most, MAXC * std::max(c->kf[l], c->kb[l]));
  }
  hipLaunchKernelGGL(k_pack_weights, dim3((unsigned)((most + 255) / 256), (unsigned)c->L), dim3(256), 0,
                     c->stream, a);
  CNNCHK(c, hipGetLastError());
  return RTM_CNN_OK;
}

template <int NK, int NCOB>
void conv_go(const ConvArgs& a, unsigned blocks, hipStream_t s) {
  hipLaunchKernelGGL((k_conv<NK, NCOB>), dim3(blocks), dim3(256), 0, s, a);
}

int launch_conv(rtm_cnn* c, ConvArgs a) {
  const int nk = a.kpad / 32;
  if (a.cin_p == 32) {
    // Strips of sixteen rows (two halo rows each) where that still gives every
    // SIMD four, shorter ones below; the waves that fit at once (two per SIMD)
    // take an equal number each.
    const long long cols = (long long)a.n * a.dil * ((a.w + 15) / 16);
    const int per = (a.h + a.dil - 1) / a.dil;
    a.ch = 16;
    while (a.ch > 1 && cols * ((per + a.ch - 1) / a.ch) < 4096) a.ch /= 2;
    const long long strips = cols * ((per + a.ch - 1) / a.ch);
    const long long rounds = (strips + 2047) / 2048, waves = (strips + rounds - 1) / rounds;
    const dim3 grid((unsigned)((waves + 3) / 4));
    if (a.ncob == 2) hipLaunchKernelGGL((k_conv_rows<2>), grid, dim3(256), 0, c->stream, a);
    else hipLaunchKernelGGL((k_conv_rows<1>), grid, dim3(256), 0, c->stream, a);
    CNNCHK(c, hipGetLastError());
    return RTM_CNN_OK;
  }
  const long long tiles = (long long)a.n * a.h * ((a.w + 15) / 16);
  const unsigned blocks = (unsigned)std::min<long long>((tiles + 3) / 4, 2048);
  switch (nk * 4 + a.ncob) {
    case 3 * 4 + 1: conv_go<3, 1>(a, blocks, c->stream); break;
    case 3 * 4 + 2: conv_go<3, 2>(a, blocks, c->stream); break;
    case 5 * 4 + 1: conv_go<5, 1>(a, blocks, c->stream); break;
    case 5 * 4 + 2: conv_go<5, 2>(a, blocks, c->stream); break;
    case 7 * 4 + 1: conv_go<7, 1>(a, blocks, c->stream); break;
    case 7 * 4 + 2: conv_go<7, 2>(a, blocks, c->stream); break;
    default: return cfail(c, RTM_CNN_E_ARG, "no convolution for K %d, %d channel blocks", a.kpad, a.ncob);
  }
  CNNCHK(c, hipGetLastError());
  return RTM_CNN_OK;
}

// Forward of the batch already packed in act[0] / resid; y32 = output.
int forward_dev(rtm_cnn* c, int n, int h, int w) {
  for (int l = 0; l < c->L; ++l) {
    ConvArgs a{};
    a.in = c->act[l];
    a.wt = c->wf[l];
    a.bias = c->bias[l];
    a.n = n; a.h = h; a.w = w;
    a.cin_p = c->cp[l];
    a.kpad = c->kf[l];
    a.cout_p = c->cp[l + 1];
    a.dil = c->dil[l];
    a.ncob = (l + 1 < c->L) ? (c->cp[l + 1] + 15) / 16 : 1;
    if (l + 1 < c->L) {
      a.mode = 0;
      a.out = c->act[l + 1];
    } else {
      a.mode = 1;
      a.out32 = c->y32;
      a.resid = c->resid;
    }
    int rc = launch_conv(c, a);
    if (rc != RTM_CNN_OK) return rc;
  }
  return RTM_CNN_OK;
}

// order: a training batch, images order[b0 ..] of the set x_dev with targets t_dev.
int pack_input(rtm_cnn* c, const float* x_dev, int n, int h, int w, const int* order = nullptr,
               int b0 = 0, const float* t_dev = nullptr) {
  const long long npix = (long long)n * h * w;
  hipLaunchKernelGGL(k_pack_input, dim3(nblk(npix)), dim3(256), 0, c->stream, x_dev, npix, h * w,
                     c->c[0], c->cp[0], c->act[0], c->resid, order, b0, t_dev, c->t32);
  CNNCHK(c, hipGetLastError());
  return RTM_CNN_OK;
}

constexpr int SQ_BLOCKS = 256;  // partial sums of a batch's loss
constexpr int LOSS_BATCHES = 1024;  // losses that rtm_cnn_fit reads back at a time (2 MB)
// The loss of a batch of npix pixels from its partial sums.
double loss_of(const double* part, long long npix) {
  double s = 0.0;
  for (int i = 0; i < SQ_BLOCKS; ++i) s += part[i];
  return s / (double)npix;
}

// Gradients for the batch in act[0] / resid with targets t_dev; sq: device
// room for the partial sums of its loss, or null.
int loss_grad_dev(rtm_cnn* c, const float* t_dev, int n, int h, int w, double* sq) {
  int rc = forward_dev(c, n, h, w);
  if (rc != RTM_CNN_OK) return rc;
  const long long npix = (long long)n * h * w;
  const int L = c->L;
  hipLaunchKernelGGL(k_loss_grad, dim3(nblk(npix)), dim3(256), 0, c->stream, c->y32, t_dev, npix,
                     c->cp[L], (float)(2.0 / (double)npix), c->dz[L - 1], c->diff);
  CNNCHK(c, hipGetLastError());
  for (int l = L - 1; l >= 0; --l) {
    const int rows = n * h;
    const int rows_per = (rows + WG_GROUPS - 1) / WG_GROUPS;
    const int P = (rows + rows_per - 1) / rows_per;
    const int d = c->dil[l];
    const bool ring = d == 1 && w <= WG_RING_W;
    // panel: the whole row in the ring; else 64 pixels, 32 where the halo of the
    // dilated taps needs the room
    const int pw = ring ? (w + 31) / 32 * 32 : (d <= 8 ? 64 : 32);
    WgradArgs g{c->dz[l], c->act[l], c->part, n, h, w, c->cp[l + 1], c->cp[l], d, rows_per, pw};
    const size_t row = (size_t)((pw + 2 * d + 15) & ~15) * 64;
    if (ring)
      hipLaunchKernelGGL((k_wgrad<true>), dim3((unsigned)P), dim3(256), 4 * row + 128 * (size_t)pw,
                         c->stream, g);
    else
      hipLaunchKernelGGL((k_wgrad<false>), dim3((unsigned)P), dim3(256), 6 * row + 128 * (size_t)pw,
                         c->stream, g);
    CNNCHK(c, hipGetLastError());
    hipLaunchKernelGGL(k_wgrad_reduce, dim3((unsigned)(9 * c->c[l + 1] + 1)), dim3(32 * WG_LEVEL1), 0,
                       c->stream, c->part, P, c->c[l], c->c[l + 1], c->grad + c->off[l]);
    CNNCHK(c, hipGetLastError());
    if (l > 0) {  // dz[l-1] = conv(dz[l], W^T flipped) * (act[l] > 0)
      ConvArgs a{};
      a.in = c->dz[l];
      a.wt = c->wb[l];
      a.out = c->dz[l - 1];
      a.mask = c->act[l];
      a.n = n; a.h = h; a.w = w;
      a.cin_p = c->cp[l + 1];
      a.kpad = c->kb[l];
      a.cout_p = c->cp[l];
      a.mode = 2;
      a.dil = c->dil[l];
      a.ncob = (c->cp[l] + 15) / 16;
      rc = launch_conv(c, a);
      if (rc != RTM_CNN_OK) return rc;
    }
  }
  if (sq) {
    hipLaunchKernelGGL(k_sumsq, dim3(SQ_BLOCKS), dim3(256), 0, c->stream, c->diff, npix, sq);
    CNNCHK(c, hipGetLastError());
  }
  c->grad_ok = true;
  return RTM_CNN_OK;
}

int adam_dev(rtm_cnn* c, float lr, float b1, float b2, float eps) {
  c->adam_t += 1;
  const double c1 = 1.0 / (1.0 - pow((double)b1, c->adam_t));
  const double c2 = 1.0 / (1.0 - pow((double)b2, c->adam_t));
  hipLaunchKernelGGL(k_adam, dim3((c->np + 255) / 256), dim3(256), 0, c->stream, c->prm, c->grad,
                     c->am, c->av, c->np, lr, b1, b2, eps, (float)c1, (float)c2);
  CNNCHK(c, hipGetLastError());
  return pack_weights(c);
}

}  // namespace

extern "C" {

int rtm_cnn_create(int nlayer, const int* channels, const int* dilation, long long max_pixels,
                   long long max_rows, rtm_cnn** out) {
  if (!channels || !out) return RTM_CNN_E_ARG;
  *out = nullptr;
  if (nlayer < 1 || nlayer > MAXL) return RTM_CNN_E_ARG;
  for (int l = 0; l <= nlayer; ++l)
    if (channels[l] < 1 || channels[l] > MAXC) return RTM_CNN_E_ARG;
  if (dilation)
    for (int l = 0; l < nlayer; ++l)
      if (dilation[l] < 1 || dilation[l] > 64) return RTM_CNN_E_ARG;
  if (channels[nlayer] != 1 || max_pixels < 1 || max_rows < 1) return RTM_CNN_E_ARG;
  if (max_pixels > MAX_PIXELS || max_rows > max_pixels) return RTM_CNN_E_ARG;
  rtm_cnn* c = new (std::nothrow) rtm_cnn();
  if (!c) return RTM_CNN_E_NOMEM;
  c->L = nlayer;
  for (int l = 0; l <= nlayer; ++l) {
    c->c[l] = channels[l];
    c->cp[l] = pad8(channels[l]);
  }
  for (int l = 0; l < nlayer; ++l) {
    c->dil[l] = dilation ? dilation[l] : 1;
    c->kf[l] = pad32(9 * c->cp[l]);
    c->kb[l] = pad32(9 * c->cp[l + 1]);
    c->off[l + 1] = c->off[l] + c->c[l + 1] * c->c[l] * 9 + c->c[l + 1];
  }
  c->np = c->off[nlayer];
  c->cap_pix = max_pixels;
  c->cap_rows = max_rows;
  int rc = RTM_CNN_OK;
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) rc = RTM_CNN_E_HIP;
  if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->prm, c->np);
  if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->grad, c->np);
  if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->am, c->np);
  if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->av, c->np);
  for (int l = 0; l < nlayer && rc == RTM_CNN_OK; ++l) {
    rc = calloc_dev(c, &c->wf[l], (size_t)MAXC * c->kf[l]);
    if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->wb[l], (size_t)MAXC * c->kb[l]);
    if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->bias[l], MAXC);
    if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->act[l], (size_t)max_pixels * c->cp[l]);
    if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->dz[l], (size_t)max_pixels * c->cp[l + 1]);
  }
  if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->x32, (size_t)max_pixels * c->c[0]);
  if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->resid, (size_t)max_pixels);
  if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->y32, (size_t)max_pixels);
  if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->t32, (size_t)max_pixels);
  if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->diff, (size_t)max_pixels);
  if (rc == RTM_CNN_OK)
    rc = calloc_dev(c, &c->part, (size_t)std::min<long long>(max_rows, WG_GROUPS) * WG_STRIDE);
  if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->sq, SQ_BLOCKS);
  if (rc == RTM_CNN_OK) {
    if (hipMemsetAsync(c->am, 0, c->np * sizeof(float), c->stream) != hipSuccess ||
        hipMemsetAsync(c->av, 0, c->np * sizeof(float), c->stream) != hipSuccess ||
        hipMemsetAsync(c->prm, 0, c->np * sizeof(float), c->stream) != hipSuccess)
      rc = RTM_CNN_E_HIP;
  }
  if (rc == RTM_CNN_OK) rc = pack_weights(c);
  if (rc == RTM_CNN_OK && hipStreamSynchronize(c->stream) != hipSuccess) rc = RTM_CNN_E_HIP;
  if (rc != RTM_CNN_OK) {
    rtm_cnn_destroy(c);
    return rc;
  }
  *out = c;
  return RTM_CNN_OK;
}

int rtm_cnn_destroy(rtm_cnn* c) {
  if (!c) return RTM_CNN_OK;
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (void* p : c->allocs) (void)hipFree(p);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
  return RTM_CNN_OK;
}

const char* rtm_cnn_last_error(const rtm_cnn* c) { return c ? c->err.c_str() : "null network"; }

int rtm_cnn_num_params(const rtm_cnn* c) { return c ? c->np : 0; }

int rtm_cnn_set_params(rtm_cnn* c, const float* p) {
  if (!c || !p) return RTM_CNN_E_ARG;
  CNNCHK(c, hipMemcpyAsync(c->prm, p, c->np * sizeof(float), hipMemcpyHostToDevice, c->stream));
  CNNCHK(c, hipMemsetAsync(c->am, 0, c->np * sizeof(float), c->stream));
  CNNCHK(c, hipMemsetAsync(c->av, 0, c->np * sizeof(float), c->stream));
  c->adam_t = 0;
  int rc = pack_weights(c);
  if (rc != RTM_CNN_OK) return rc;
  CNNCHK(c, hipStreamSynchronize(c->stream));
  return RTM_CNN_OK;
}

int rtm_cnn_get_params(rtm_cnn* c, float* p) {
  if (!c || !p) return RTM_CNN_E_ARG;
  CNNCHK(c, hipMemcpyAsync(p, c->prm, c->np * sizeof(float), hipMemcpyDeviceToHost, c->stream));
  CNNCHK(c, hipStreamSynchronize(c->stream));
  return RTM_CNN_OK;
}

int rtm_cnn_forward(rtm_cnn* c, const float* x, int n, int h, int w, float* y) {
  if (!c || !x || !y) return RTM_CNN_E_ARG;
  int rc = check_shape(c, n, h, w);
  if (rc != RTM_CNN_OK) return rc;
  const size_t npix = (size_t)n * h * w;
  CNNCHK(c, hipMemcpyAsync(c->x32, x, npix * c->c[0] * sizeof(float), hipMemcpyHostToDevice, c->stream));
  rc = pack_input(c, c->x32, n, h, w);
  if (rc == RTM_CNN_OK) rc = forward_dev(c, n, h, w);
  if (rc != RTM_CNN_OK) return rc;
  CNNCHK(c, hipMemcpyAsync(y, c->y32, npix * sizeof(float), hipMemcpyDeviceToHost, c->stream));
  CNNCHK(c, hipStreamSynchronize(c->stream));
  return RTM_CNN_OK;
}

int rtm_cnn_loss_grad(rtm_cnn* c, const float* x, const float* t, int n, int h, int w, double* loss,
                      float* grad) {
  if (!c || !x || !t) return RTM_CNN_E_ARG;
  int rc = check_shape(c, n, h, w);
  if (rc != RTM_CNN_OK) return rc;
  const size_t npix = (size_t)n * h * w;
  CNNCHK(c, hipMemcpyAsync(c->x32, x, npix * c->c[0] * sizeof(float), hipMemcpyHostToDevice, c->stream));
  CNNCHK(c, hipMemcpyAsync(c->t32, t, npix * sizeof(float), hipMemcpyHostToDevice, c->stream));
  rc = pack_input(c, c->x32, n, h, w);
  if (rc == RTM_CNN_OK) rc = loss_grad_dev(c, c->t32, n, h, w, loss ? c->sq : nullptr);
  if (rc != RTM_CNN_OK) return rc;
  double part[SQ_BLOCKS];
  if (loss) CNNCHK(c, hipMemcpyAsync(part, c->sq, sizeof(part), hipMemcpyDeviceToHost, c->stream));
  if (grad) CNNCHK(c, hipMemcpyAsync(grad, c->grad, c->np * sizeof(float), hipMemcpyDeviceToHost, c->stream));
  CNNCHK(c, hipStreamSynchronize(c->stream));
  if (loss) *loss = loss_of(part, (long long)npix);
  return RTM_CNN_OK;
}

int rtm_cnn_adam_step(rtm_cnn* c, float lr, float b1, float b2, float eps) {
  if (!c) return RTM_CNN_E_ARG;
  if (!c->grad_ok) return cfail(c, RTM_CNN_E_STATE, "rtm_cnn_loss_grad first");
  int rc = adam_dev(c, lr, b1, b2, eps);
  if (rc != RTM_CNN_OK) return rc;
  CNNCHK(c, hipStreamSynchronize(c->stream));
  return RTM_CNN_OK;
}

int rtm_cnn_fit(rtm_cnn* c, const float* x, const float* t, int n, int h, int w, int epochs,
                int batch, float lr, unsigned seed, double* loss_per_epoch) {
  if (!c || !x || !t || epochs < 0 || batch < 1) return RTM_CNN_E_ARG;
  if (batch > n) batch = n;
  int rc = check_shape(c, batch, h, w);
  if (rc != RTM_CNN_OK) return rc;
  const size_t img = (size_t)h * w;
  const size_t need = (size_t)n * img;
  if ((long long)need > c->ds_cap || n > c->ds_n) {  // a larger training set replaces the old copy
    CNNCHK(c, hipStreamSynchronize(c->stream));
    cfree_dev(c, &c->ds_x);
    cfree_dev(c, &c->ds_t);
    cfree_dev(c, &c->ds_order);
    c->ds_cap = 0;
    c->ds_n = 0;
    rc = calloc_dev(c, &c->ds_x, need * c->c[0]);
    if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->ds_t, need);
    if (rc == RTM_CNN_OK) rc = calloc_dev(c, &c->ds_order, (size_t)n);
    if (rc != RTM_CNN_OK) return rc;
    c->ds_cap = (long long)need;
    c->ds_n = n;
  }
  const int batches = n / batch, keep = std::min(batches, LOSS_BATCHES);
  if (keep > c->ds_nb) {
    CNNCHK(c, hipStreamSynchronize(c->stream));
    cfree_dev(c, &c->ds_sq);
    c->ds_nb = 0;
    rc = calloc_dev(c, &c->ds_sq, (size_t)keep * SQ_BLOCKS);
    if (rc != RTM_CNN_OK) return rc;
    c->ds_nb = keep;
  }
  std::vector<double> part((size_t)keep * SQ_BLOCKS);
  CNNCHK(c, hipMemcpyAsync(c->ds_x, x, need * c->c[0] * sizeof(float), hipMemcpyHostToDevice, c->stream));
  CNNCHK(c, hipMemcpyAsync(c->ds_t, t, need * sizeof(float), hipMemcpyHostToDevice, c->stream));
  std::vector<int> order(n);
  for (int i = 0; i < n; ++i) order[i] = i;
  unsigned long long s = seed * 6364136223846793005ULL + 1442695040888963407ULL;
  auto rnd = [&s]() {  // 64-bit LCG, high bits
    s = s * 6364136223846793005ULL + 1442695040888963407ULL;
    return (unsigned)(s >> 33);
  };
  for (int ep = 0; ep < epochs; ++ep) {
    for (int i = n - 1; i > 0; --i) {  // Fisher-Yates
      const int j = (int)(rnd() % (unsigned)(i + 1));
      const int tmp = order[i]; order[i] = order[j]; order[j] = tmp;
    }
    // the previous epoch ended with a stream synchronisation (the loss read-back)
    CNNCHK(c, hipMemcpyAsync(c->ds_order, order.data(), n * sizeof(int), hipMemcpyHostToDevice, c->stream));
    double sum = 0.0;
    for (int nb = 0; nb < batches; ++nb) {
      const int slot = nb % keep;
      rc = pack_input(c, c->ds_x, batch, h, w, c->ds_order, nb * batch, c->ds_t);
      if (rc == RTM_CNN_OK)
        rc = loss_grad_dev(c, c->t32, batch, h, w, c->ds_sq + (size_t)slot * SQ_BLOCKS);
      if (rc == RTM_CNN_OK) rc = adam_dev(c, lr, 0.9f, 0.999f, 1e-8f);
      if (rc != RTM_CNN_OK) return rc;
      if (slot + 1 < keep && nb + 1 < batches) continue;
      // the losses are read once an epoch, or when the room for them is full
      CNNCHK(c, hipMemcpyAsync(part.data(), c->ds_sq, (size_t)(slot + 1) * SQ_BLOCKS * sizeof(double),
                               hipMemcpyDeviceToHost, c->stream));
      CNNCHK(c, hipStreamSynchronize(c->stream));
      for (int i = 0; i <= slot; ++i)
        sum += loss_of(part.data() + (size_t)i * SQ_BLOCKS, (long long)batch * h * w);
    }
    if (loss_per_epoch) loss_per_epoch[ep] = sum / batches;
  }
  CNNCHK(c, hipStreamSynchronize(c->stream));
  return RTM_CNN_OK;
}

}  // extern "C"
