// rtm_device.h -- device helpers shared by the stencil kernels
// (rtm_stencil.hip) and the small kernels (rtm_kernels.hip).  Internal header.
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "rtm_kernels.h"

namespace rtm {

// ---------------------------------------------------------------------------
// helpers
__device__ __forceinline__ float compr(const float4& v, int i) {
  return i == 0 ? v.x : (i == 1 ? v.y : (i == 2 ? v.z : v.w));
}

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// Barrier of the block for LDS data alone: loads from memory stay in flight.
__device__ __forceinline__ void block_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Raw buffer access.  Word 3 of a gfx9-family resource: 32-bit data format,
// no swizzle, stride 0 (range check on the byte offset against num_records).
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t Rsrc;
constexpr int kRsrcWord3 = 0x00020000;
constexpr unsigned kDrop = 0x80000000u;  // column offset that is out of range of every buffer
__device__ __forceinline__ Rsrc rsrc(const void* base, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, kRsrcWord3);
}
__device__ __forceinline__ float4 bld4(Rsrc r, unsigned vo, unsigned so) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)vo, (int)so, 0);
  return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z),
                     __uint_as_float(v.w));
}
__device__ __forceinline__ uint4 bld4u(Rsrc r, unsigned vo, unsigned so) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)vo, (int)so, 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}
// Stores take the whole offset in the VGPR operand and a zero soffset.  A
// store of more than 64 bits reads its data VGPRs late, so a VALU write to them
// right after the store needs one wait state; the compiler inserts it only for
// stores whose soffset is not a register.  (With the row offset in an SGPR
// soffset the q store of the receiver step lost its first dword in some lanes
// when two blocks shared a CU.)  vo | kDrop stays >= 2^31 after adding so < 2^30.
__device__ __forceinline__ void bst4(Rsrc r, unsigned vo, unsigned so, float a, float b, float c,
                                     float d) {
  const u32x4 v = {__float_as_uint(a), __float_as_uint(b), __float_as_uint(c), __float_as_uint(d)};
  __builtin_amdgcn_raw_buffer_store_b128(v, r, (int)(vo + so), 0, 0);
}
// Streaming variants for data touched once per time step (u(k+1), u0, the
// image and illumination sums): the non-temporal policy keeps them from
// displacing what the shots of a launch share in the caches (the model's P
// and coefficient offsets, the coefficient table, the u1 halo rows).
#ifndef RTM_STREAM_POLICY
#define RTM_STREAM_POLICY 2  // cache-policy bits of the buffer instructions: nt
#endif
__device__ __forceinline__ float4 bld4s(Rsrc r, unsigned vo, unsigned so) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)vo, (int)so, RTM_STREAM_POLICY);
  return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z),
                     __uint_as_float(v.w));
}
__device__ __forceinline__ void bst4s(Rsrc r, unsigned vo, unsigned so, float a, float b, float c,
                                      float d) {
  const u32x4 v = {__float_as_uint(a), __float_as_uint(b), __float_as_uint(c), __float_as_uint(d)};
  __builtin_amdgcn_raw_buffer_store_b128(v, r, (int)(vo + so), 0, RTM_STREAM_POLICY);
}
__device__ __forceinline__ void bst1s_(Rsrc r, unsigned vo, unsigned so, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, (int)(vo + so), 0, RTM_STREAM_POLICY);
}

__device__ __forceinline__ float bld1(Rsrc r, unsigned vo, unsigned so) {
  return __uint_as_float((unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, (int)vo, (int)so, 0));
}
__device__ __forceinline__ unsigned bld1u(Rsrc r, unsigned vo, unsigned so) {
  return (unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, (int)vo, (int)so, 0);
}
// streaming variants (u0 rows, u(k+1) and strip writes: touched once per step)
__device__ __forceinline__ float bld1s(Rsrc r, unsigned vo, unsigned so) {
  return __uint_as_float((unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, (int)vo, (int)so,
                                                                        RTM_STREAM_POLICY));
}
__device__ __forceinline__ void bst1s(Rsrc r, unsigned vo, unsigned so, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, (int)(vo + so), 0, RTM_STREAM_POLICY);
}

// Coefficient row [c_0 .. c_NFD | zeros] of a cell, CS floats.  Gathering the
// rows of a wave's cells is what its loads cost most (up to 64 cache lines an
// instruction): with c_0 as the table's float, promoted here, a row of
// half-length 3 is one 16-byte gather (two when the row held (1 + hzx2_1) c_0
// in double), of 7 two, of 11 three.
template <int NFD>
struct CoefRow {
  static constexpr int CS = ((1 + NFD) + 3) & ~3;
  static constexpr int NR = CS / 4;
  float4 r[NR];
  __device__ __forceinline__ void load(const float* ctab, unsigned byte_off) {
    const float4* p = reinterpret_cast<const float4*>(reinterpret_cast<const char*>(ctab) + byte_off);
#pragma unroll
    for (int i = 0; i < NR; ++i) r[i] = p[i];
  }
  __device__ __forceinline__ void load(Rsrc t, unsigned byte_off) {
#pragma unroll
    for (int i = 0; i < NR; ++i) r[i] = bld4(t, byte_off + 16u * i, 0);
  }
  // centre coefficient (1.0 + hzx2_1) * c_0 of kernel.cu:58 in double
  __device__ __forceinline__ double c0d(double h1) const { return h1 * (double)r[0].x; }
  // tap coefficient c_l, l >= 1
  __device__ __forceinline__ float c(int l) const { return compr(r[l >> 2], l & 3); }
};

// Final combine of the two-way update.
//  FP32 form (Add, BKAdd, BKAdd_Con: kernel.cu:73,375,413): 2*u1-u0+P.
//  FP64 form (Add_Con, BKAdd_EFF, BKAdd_EFF_Con: kernel.cu:106,275,312): 2.0*u1-u0+P.
// p = v*v*tao2*h2 (evaluated left to right in FP32).
__device__ __forceinline__ float combine_p(float u, float u0, float p, float w1, bool f64) {
  if (f64) return (float)((2.0 * (double)u - (double)u0) + (double)(p * w1));
  return __builtin_fmaf(p, w1, 2.0f * u - u0);
}
__device__ __forceinline__ bool is_receiver(int c, const Rcv& r, int* s) {
  if (c < r.s_l || c > r.s_r) return false;
  int d = c - r.s_l;
  if (d % r.ds != 0) return false;
  *s = d / r.ds;
  return true;
}

__device__ __forceinline__ int mirror_idx(int g, int n) {  // kernel.cu:65-68
  if (g < 0) g = -g;
  if (g >= n) g = 2 * n - 2 - g;
  g = g < 0 ? 0 : g;
  g = g >= n ? n - 1 : g;
  return g;
}

// ---- strip encoding -------------------------------------------------------
// Power-of-two scale of a slot from its max |value|: 2^(e-15) with
// max = f*2^e, so |value/scale| < 2^15 and FP16 cannot overflow.  The scale is
// kept >= 2^-126 so that 1/scale stays finite when the maximum is subnormal
// (slots holding only the tiny precursors of the first steps).
__device__ __forceinline__ float pow2_scale(float amax) {
  float sc = 1.0f;
  if (amax > 0.0f) {
    int e;
    frexpf(amax, &e);
    sc = ldexpf(1.0f, max(e - 15, -126));
  }
  return sc;
}

__device__ __forceinline__ unsigned short f2bf(float f) {  // round to nearest even
  unsigned u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)((u >> 16) | ((u & 0xffff) ? 0x40 : 0));
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf2f(unsigned short b) { return __uint_as_float(((unsigned)b) << 16); }

// Strip slot layout: lf[mnz][nfd], rt[mnz][nfd], up[nfd][mnx], dw[nfd][mnx]
// (Dlf/Drt/Dup/Ddw of kernel.cu:199-205); a slot holds ss_of(mnx) elements.
__device__ __forceinline__ long long strip_size(const Grid& g, int mnx) {
  return 2LL * g.nfd * (g.mnz + mnx);
}
// Strip element index -> grid cell of a shot of width nx (interior mnx), in
// 32-bit arithmetic (a slot holds fewer than 2^31 elements).
__device__ __forceinline__ void strip_cell(const Grid& g, int nx, int mnx, unsigned e, int* z,
                                           int* x) {
  const unsigned nfd = (unsigned)g.nfd, a = (unsigned)g.mnz * nfd, b = nfd * (unsigned)mnx;
  if (e < 2 * a) {
    const unsigned side = e >= a ? 1u : 0u, ee = e - side * a;
    const unsigned r = ee / nfd, d = ee - r * nfd;
    *z = g.n2 + (int)r;
    *x = side ? nx - g.n2 + (int)d : g.n2 - 1 - (int)d;
  } else {
    const unsigned bot = e >= 2 * a + b ? 1u : 0u, ee = e - 2 * a - bot * b;
    const unsigned d = ee / (unsigned)mnx, c = ee - d * (unsigned)mnx;
    *z = bot ? g.nz - g.n2 + (int)d : g.n2 - 1 - (int)d;
    *x = g.n2 + (int)c;
  }
}
// Strip element of frame cell (z, x) of a shot nx wide, or -1; without branches,
// in 32 bits (a slot holds fewer than 2^31 elements).
__device__ __forceinline__ int strip_elem(const Grid& g, int nx, int mnx, int z, int x) {
  const int a = g.mnz * g.nfd, b = g.nfd * mnx, n2 = g.n2, nfd = g.nfd;
  const bool zin = z >= n2 && z < g.nz - n2, xin = x >= n2 && x < nx - n2;
  int e = -1;
  e = (zin && x >= n2 - nfd && x < n2) ? (z - n2) * nfd + (n2 - 1 - x) : e;
  e = (zin && x >= nx - n2 && x < nx - n2 + nfd) ? a + (z - n2) * nfd + (x - (nx - n2)) : e;
  e = (xin && z >= n2 - nfd && z < n2) ? 2 * a + (n2 - 1 - z) * mnx + (x - n2) : e;
  e = (xin && z >= g.nz - n2 && z < g.nz - n2 + nfd) ? 2 * a + b + (z - (g.nz - n2)) * mnx + (x - n2) : e;
  return e;
}
__device__ __forceinline__ void strip_put(const Strips& st, int shot, int k, long long e, float val) {
  if (st.fmt == 0) {
    float* p = (float*)st.base;
    p[((long long)shot * st.nslot + (k % st.nslot)) * st.ss + e] = val;
  } else {
    st.stage[((long long)shot * 2 + (k & 1)) * st.ss + e] = val;
  }
}
__device__ __forceinline__ float strip_get(const Strips& st, int shot, int k, long long e) {
  long long slot = (long long)shot * st.nslot + (k % st.nslot);
  if (st.fmt == 0) return ((const float*)st.base)[slot * st.ss + e];
  const unsigned short* p = (const unsigned short*)st.base;
  unsigned short h = p[slot * st.ss + e];
  float sc = st.scale[slot];
  if (st.fmt == 1) return __half2float(__ushort_as_half(h)) * sc;
  return bf2f(h) * sc;
}
// Strips of slot k into the rings of field f: block b of a launch with bps
// 256-thread blocks per shot restores part of shot b / bps.
__device__ __forceinline__ void strip_restore_body(const Grid& g, float* f, const Strips& st,
                                                   const ShotGeo* geo, int k, unsigned b,
                                                   unsigned bps) {
  const int shot = (int)(b / bps);
  const unsigned blk = b - (unsigned)shot * bps;
  const ShotGeo sg = geo[shot];
  const unsigned ss = (unsigned)strip_size(g, sg.mnx);
  float* F = f + (long long)shot * g.fstride + g.x0;
  const unsigned step = bps * 256u;
  // four elements at a time, loads first: one element after the other each
  // waited for its own load (two fields of 128 shots 53 us in a frame launch)
  for (unsigned e0 = blk * 256u + threadIdx.x; e0 < ss; e0 += 4u * step) {
    float v[4];
#pragma unroll
    for (unsigned i = 0; i < 4; ++i) v[i] = strip_get(st, shot, k, (long long)min(e0 + i * step, ss - 1u));
#pragma unroll
    for (unsigned i = 0; i < 4; ++i) {
      const unsigned e = e0 + i * step;
      if (e >= ss) break;
      int z, x;
      strip_cell(g, sg.nx, sg.mnx, e, &z, &x);
      F[(long)z * g.pitch + x] = v[i];
    }
  }
}

}  // namespace rtm
