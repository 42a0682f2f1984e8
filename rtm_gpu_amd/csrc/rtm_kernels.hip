// rtm_kernels.hip -- the small kernels of the 2-D acoustic RTM step (strips,
// snapshots, begin states, image post, stacks, dot products, transposes) and
// the dispatch of the stencil kernels (rtm_stencil.hip) by half-length.
#include <algorithm>

#include <hip/hip_runtime.h>

#include "rtm_device.h"

namespace rtm {

// ---------------------------------------------------------------------------
// Finite-value watch (not in the reference): *flag stays 0xffffffff while every
// checked field is finite; the first check that meets a NaN or an infinity
// stores its step k there.
__global__ void k_flag_reset(unsigned* flag) {
  if (blockIdx.x == 0 && threadIdx.x == 0) flag[0] = 0xffffffffu;
}
__global__ __launch_bounds__(256) void k_finite_check(const float4* f, long long n4, int k,
                                                      unsigned* flag) {
  bool bad = false;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n4;
       i += (long long)gridDim.x * blockDim.x) {
    const float4 v = f[i];
    bad = bad || !(isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.w));
  }
  if (__any(bad) && (threadIdx.x & 63) == 0) atomicCAS(flag, 0xffffffffu, (unsigned)k);
}

// ---------------------------------------------------------------------------
// Small kernels.
__global__ void k_fill(float* p, long long n, float val) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  long long st = (long long)gridDim.x * blockDim.x;
  for (; i < n; i += st) p[i] = val;
}

// u(0) = 0, u(1) = f(0)/2 at the source (kernel.cu:798-806).
__global__ void k_fwd_begin(Grid g, float* f0, float* f1, const ShotGeo* geo, float spike) {
  const int shot = blockIdx.y;
  const long long n = (long long)g.nz * g.pitch;
  float* a = f0 + (long long)shot * g.fstride;
  float* b = f1 + (long long)shot * g.fstride;
  const ShotGeo sg = geo[shot];
  const long long ps = (long long)sg.r_u * g.pitch + g.x0 + sg.r_x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    a[i] = 0.0f;
    b[i] = (i == ps) ? spike : 0.0f;
  }
}

__global__ void k_strip_save(Grid g, const float* f, Strips st, const ShotGeo* geo, int k) {
  const int shot = blockIdx.y;
  const ShotGeo sg = geo[shot];
  const unsigned ss = (unsigned)strip_size(g, sg.mnx);
  const float* F = f + (long long)shot * g.fstride + g.x0;
  for (unsigned e = blockIdx.x * blockDim.x + threadIdx.x; e < ss; e += gridDim.x * blockDim.x) {
    int z, x;
    strip_cell(g, sg.nx, sg.mnx, e, &z, &x);
    strip_put(st, shot, k, (long long)e, F[(long)z * g.pitch + x]);
  }
}

// Maximum |value| of the staged fp32 strips of slot k: one atomic per block
// on the bit patterns (non-negative floats order as their bits).
__global__ __launch_bounds__(256) void k_strip_amax(Grid g, Strips st, const ShotGeo* geo, int k) {
  __shared__ unsigned sh[4];
  const int shot = blockIdx.y;
  const long long ss = strip_size(g, geo[shot].mnx);
  const float* s = st.stage + ((long long)shot * 2 + (k & 1)) * st.ss;
  unsigned mx = 0u;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < ss;
       e += (long long)gridDim.x * blockDim.x)
    mx = max(mx, __float_as_uint(fabsf(s[e])));
  for (int o = 32; o > 0; o >>= 1) mx = max(mx, (unsigned)__shfl_xor((int)mx, o));
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0)
    atomicMax(&st.amax[(long long)shot * st.nslot + (k % st.nslot)],
              max(max(sh[0], sh[1]), max(sh[2], sh[3])));
}

// Quantise the staged fp32 strips of slot k with the slot's power-of-two scale.
__global__ void k_strip_finish(Grid g, Strips st, const ShotGeo* geo, int k) {
  const int shot = blockIdx.y;
  const long long ss = strip_size(g, geo[shot].mnx);
  const long long slot = (long long)shot * st.nslot + (k % st.nslot);
  const float sc = pow2_scale(__uint_as_float(st.amax[slot]));
  if (blockIdx.x == 0 && threadIdx.x == 0) st.scale[slot] = sc;
  const float inv = 1.0f / sc;     // exact: sc is a power of two
  const float* s = st.stage + ((long long)shot * 2 + (k & 1)) * st.ss;
  unsigned short* d = (unsigned short*)st.base + slot * st.ss;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < ss;
       e += (long long)gridDim.x * blockDim.x) {
    float x = s[e] * inv;
    d[e] = (st.fmt == 1) ? __half_as_ushort(__float2half_rn(x)) : f2bf(x);
  }
}

__global__ __launch_bounds__(256) void k_strip_restore(Grid g, float* f, Strips st,
                                                       const ShotGeo* geo, int k) {
  strip_restore_body(g, f, st, geo, k, blockIdx.y * gridDim.x + blockIdx.x, gridDim.x);
}

// ---- checkpoint snapshots -------------------------------------------------
// A snapshot slot holds nz*nx (widest shot) elements; shot s uses the first
// nz*nx_s of them, row-major over its own width.

__global__ void k_snap_clear(Snaps sn, int slot, int nshot) {  // a kernel, not a memset: capturable
  const int sh = blockIdx.x * blockDim.x + threadIdx.x;
  if (sh < nshot) sn.amax[(long long)sh * sn.nsnap + slot] = 0u;
}

__global__ void k_snap_amax(Grid g, const float* f, Snaps sn, const ShotGeo* geo, int slot) {
  const int shot = blockIdx.y;
  const int nx = geo[shot].nx;
  const float* F = f + (long long)shot * g.fstride + g.x0;
  const long long n = (long long)g.nz * nx;
  float mx = 0.0f;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n;
       e += (long long)gridDim.x * blockDim.x) {
    const int z = (int)(e / nx), x = (int)(e % nx);
    mx = fmaxf(mx, fabsf(F[(long)z * g.pitch + x]));
  }
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if ((threadIdx.x & 63) == 0) atomicMax(&sn.amax[(long long)shot * sn.nsnap + slot], __float_as_uint(mx));
}

__global__ void k_snap_save(Grid g, const float* f, Snaps sn, const ShotGeo* geo, int slot) {
  const int shot = blockIdx.y;
  const int nx = geo[shot].nx;
  const float* F = f + (long long)shot * g.fstride + g.x0;
  const long long n = (long long)g.nz * nx, stride = (long long)g.nz * g.nx;
  const long long so = (long long)shot * sn.nsnap + slot;
  float inv = 1.0f;
  if (sn.fmt != 0) {
    const float sc = pow2_scale(__uint_as_float(sn.amax[so]));
    if (blockIdx.x == 0 && threadIdx.x == 0) sn.scale[so] = sc;
    inv = 1.0f / sc;  // exact: sc is a power of two
  }
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n;
       e += (long long)gridDim.x * blockDim.x) {
    const int z = (int)(e / nx), x = (int)(e % nx);
    const float v = F[(long)z * g.pitch + x];
    if (sn.fmt == 0) {
      ((float*)sn.base)[so * stride + e] = v;
    } else {
      const float y = v * inv;
      ((unsigned short*)sn.base)[so * stride + e] =
          (sn.fmt == 1) ? __half_as_ushort(__float2half_rn(y)) : f2bf(y);
    }
  }
}

__global__ void k_snap_restore(Grid g, float* f, Snaps sn, const ShotGeo* geo, int slot) {
  const int shot = blockIdx.y;
  const int nx = geo[shot].nx;
  float* F = f + (long long)shot * g.fstride + g.x0;
  const long long n = (long long)g.nz * nx, stride = (long long)g.nz * g.nx;
  const long long so = (long long)shot * sn.nsnap + slot;
  const float sc = sn.fmt != 0 ? sn.scale[so] : 1.0f;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n;
       e += (long long)gridDim.x * blockDim.x) {
    const int z = (int)(e / nx), x = (int)(e % nx);
    float v;
    if (sn.fmt == 0) {
      v = ((const float*)sn.base)[so * stride + e];
    } else {
      const unsigned short h = ((const unsigned short*)sn.base)[so * stride + e];
      v = (sn.fmt == 1 ? __half2float(__ushort_as_half(h)) : bf2f(h)) * sc;
    }
    F[(long)z * g.pitch + x] = v;
  }
}

// Receiver recording of u(k): rec[shot][k][s], s < n of the shot (stride r.n).
__global__ void k_record(Grid g, Rcv r, const ShotGeo* geo, const float* f, float* rec, int k,
                         int nt) {
  const int shot = blockIdx.y;
  const ShotGeo sg = geo[shot];
  const float* F = f + (long long)shot * g.fstride + g.x0;
  for (int s = blockIdx.x * blockDim.x + threadIdx.x; s < sg.n; s += gridDim.x * blockDim.x)
    rec[((long long)shot * nt + k) * r.n + s] = F[(long)r.s_z * g.pitch + sg.s_l + s * r.ds];
}

// Backward initial state (kernel.cu:859-885).  s0 = u(nt-1) (DBW0),
// s1 = u(nt-2) (DBW1); FW0 = 0 and FW1 = spike field are host arrays there.
__global__ void k_bwd_begin(Grid g, const float* s0, const float* s1, float* q0, float* q1,
                            float* su, float* sq, float* i1, float* i2, const ShotGeo* geo,
                            float spike, int icompen) {
  const int shot = blockIdx.y;
  const long long base = (long long)shot * g.fstride;
  const ShotGeo sg = geo[shot];
  const long long ps = (long long)sg.r_u * g.pitch + g.x0 + sg.r_x;
  const long long n = (long long)g.nz * g.pitch;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const long long p = base + i;
    const float BW0 = s0[p], BW1 = s1[p];
    const float FW1 = (i == ps) ? spike : 0.0f, FW0 = 0.0f;
    q0[p] = 0.0f;
    q1[p] = 0.0f;
    if (icompen == 1) {
      const float BW2 = BW0 + BW1;
      const float FW2 = FW0 + FW1;
      su[p] = BW2;
      sq[p] = FW2;
      i1[p] = FW2 * BW2 + FW0 * BW0;
    } else {
      su[p] = 0.0f;
      sq[p] = 0.0f;
      i1[p] = FW1 * BW1 + FW0 * BW0;
    }
    i2[p] = BW1 * BW1 + BW0 * BW0;
  }
}

// max |I2| over the interior, per shot (kernel.cu:963-970).
__global__ void k_maxabs(Grid g, const ShotGeo* geo, const float* i2, unsigned* out) {
  const int shot = blockIdx.y;
  const int mnx = geo[shot].mnx;
  const float* I = i2 + (long long)shot * g.fstride + g.x0;
  const long long n = (long long)g.mnz * mnx;
  float mx = 0.0f;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n;
       e += (long long)gridDim.x * blockDim.x) {
    int z = g.n2 + (int)(e / mnx), x = g.n2 + (int)(e % mnx);
    mx = fmaxf(mx, fabsf(I[(long)z * g.pitch + x]));
  }
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if ((threadIdx.x & 63) == 0) atomicMax(&out[shot], __float_as_uint(mx));
}

// Per-shot image post (kernel.cu:935-979).  up/down: [shot][mnz][g.mnx].
__global__ void k_post(Grid g, const ShotGeo* geo, const float* v, long long mstride,
                       const float* i1, const float* i2, const unsigned* amax, float vmax,
                       float whitecoe, float* up, float* down) {
  const int shot = blockIdx.y;
  const ShotGeo sg = geo[shot];
  const int mnx = sg.mnx, nx = sg.nx;
  const float* M = i1 + (long long)shot * g.fstride + g.x0;
  const float* I = i2 + (long long)shot * g.fstride + g.x0;
  const float* Vv = v + (long long)sg.win * mstride + g.x0;
  const long long n = (long long)g.mnz * mnx;
  const float stable = __uint_as_float(amax[shot]) * whitecoe;
  const int P = g.pitch, n2 = g.n2;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n;
       e += (long long)gridDim.x * blockDim.x) {
    const int zi = (int)(e / mnx), xi = (int)(e % mnx);
    const int i = n2 + zi, j = n2 + xi;
    int i1_ = i - 1, i2_ = i + 1, j1 = j - 1, j2 = j + 1;
    if (i1_ < n2) i1_ = 2 * n2 - i1_;
    if (j1 < n2) j1 = 2 * n2 - j1;
    if (i2_ >= g.nz - n2) i2_ = 2 * (g.nz - n2 - 1) - i2_;
    if (j2 >= nx - n2) j2 = 2 * (nx - n2 - 1) - j2;
    const float sum = M[(long)i * P + j2] + M[(long)i * P + j1] + M[(long)i2_ * P + j] +
                      M[(long)i1_ * P + j] - 4.0f * M[(long)i * P + j];
    const float vv = Vv[(long)i * P + j];
    const double t = -1.0 * (double)sum * (double)vv * (double)vv / (double)(vmax * vmax);
    const long long o = ((long long)shot * g.mnz + zi) * g.mnx + xi;
    if (up) up[o] = (float)t;
    if (down) down[o] = I[(long)i * P + j] + stable;
  }
}

// Running stack in shot order (kernel.cu:1026-1039) onto an image of gw
// columns: shot s covers columns x_img .. x_img+mnx-1.
__global__ void k_stack_add(Grid g, const ShotGeo* geo, int gw, const float* up, const float* down,
                            float* s1, float* s2, int nshot) {
  const long long nI = (long long)g.mnz * gw;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < nI;
       e += (long long)gridDim.x * blockDim.x) {
    const int z = (int)(e / gw), X = (int)(e % gw);
    float a = s1[e], b = s2[e];
    for (int s = 0; s < nshot; ++s) {
      const int x = X - geo[s].x_img;
      if (x < 0 || x >= geo[s].mnx) continue;
      const long long o = ((long long)s * g.mnz + z) * g.mnx + x;
      a += up[o];
      b += down[o];
    }
    s1[e] = a;
    s2[e] = b;
  }
}

__global__ void k_refl_scatter(Grid g, const ShotGeo* geo, int gw, const float* img, float* dst,
                               long long rstride) {
  const int shot = blockIdx.y;
  const ShotGeo sg = geo[shot];
  float* D = dst + (long long)shot * rstride;
  const long long n = (long long)g.nz * g.pitch;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const int z = (int)(i / g.pitch), x = (int)(i % g.pitch) - g.x0;
    float v = 0.0f;
    const int X = x - g.n2 + sg.x_img;
    if (z >= g.n2 && z < g.nz - g.n2 && x >= g.n2 && x < sg.nx - g.n2 && X >= 0 && X < gw)
      v = img[(long long)(z - g.n2) * gw + X];
    D[i] = v;
  }
}

__global__ void k_grad_stack(Grid g, const ShotGeo* geo, int gw, const float* G, const float* pm,
                             long long mstride, int nshot, float* grad) {
  const long long n = (long long)g.mnz * gw;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n;
       e += (long long)gridDim.x * blockDim.x) {
    const int z = (int)(e / gw), X = (int)(e % gw);
    float acc = 0.0f;
    for (int s = 0; s < nshot; ++s) {
      const int x = X - geo[s].x_img;
      if (x < 0 || x >= geo[s].mnx) continue;
      const long long pc = (long long)(z + g.n2) * g.pitch + g.x0 + g.n2 + x;
      acc = acc + G[(long long)s * g.fstride + pc] / pm[(long long)geo[s].win * mstride + pc];
    }
    grad[e] = acc;
  }
}

// FP64 dot product of two float arrays in two passes with a fixed reduction
// order (the result does not depend on scheduling): each of the DOT_BLOCKS
// blocks sums a grid-stride slice in double and reduces it in LDS; one block
// then adds the partial sums in a fixed tree.
constexpr int DOT_BLOCKS = 1024;
__device__ __forceinline__ double block_sum(double v, double* sh) {
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  return sh[0];
}
// Vector v = blockIdx.y of a batch starts at v*stride in a and b; its
// partial sums fill row v of part (gridDim.x = DOT_BLOCKS entries), so every
// vector is reduced in the same order as a single-vector launch.
__global__ __launch_bounds__(256) void k_dot64_part(const float* a, const float* b, long long n,
                                                    long long stride, double* part) {
  __shared__ double sh[256];
  a += (long long)blockIdx.y * stride;
  b += (long long)blockIdx.y * stride;
  double acc = 0.0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    acc += (double)a[i] * (double)b[i];
  const double t = block_sum(acc, sh);
  if (threadIdx.x == 0) part[(long long)blockIdx.y * gridDim.x + blockIdx.x] = t;
}
// One block per vector: out[v] = the fixed-tree sum of row v of part.
__global__ __launch_bounds__(256) void k_dot64_final(const double* part, int np, double* out) {
  __shared__ double sh[256];
  part += (long long)blockIdx.x * np;
  double acc = 0.0;
  for (int i = threadIdx.x; i < np; i += blockDim.x) acc += part[i];
  const double t = block_sum(acc, sh);
  if (threadIdx.x == 0) out[blockIdx.x] = t;
}

// y = y + a*x (product, then sum)
__global__ void k_axpy(float* y, const float* x, float a, long long n) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    y[i] = y[i] + a * x[i];
}

// out[c][r] = in[r][c] for an rows x cols matrix, through 32 x 32 LDS tiles so
// that both the reads and the writes are coalesced.
__global__ __launch_bounds__(256) void k_transpose(const float* in, float* out, int rows, int cols) {
  __shared__ float tile[32][33];
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8 threads
  for (int j = ty; j < 32; j += 8) {
    const int r = r0 + j, c = c0 + tx;
    if (r < rows && c < cols) tile[j][tx] = in[(long long)r * cols + c];
  }
  __syncthreads();
  for (int j = ty; j < 32; j += 8) {
    const int c = c0 + j, r = r0 + tx;
    if (r < rows && c < cols) out[(long long)c * rows + r] = tile[tx][j];
  }
}

__global__ void k_stack_finish(int nI, const float* s1, const float* s2, int nrec, int inorm,
                               float* img, float* ill) {  // kernel.cu:1042-1059
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < nI; e += gridDim.x * blockDim.x) {
    float a = s1[e] / nrec;
    float b = s2[e] / nrec;
    // a cell that no shot of a ragged batch covers (both sums 0) stays 0
    // instead of 0/0; every other cell is divided as in the reference
    if (inorm == 1 && !(s1[e] == 0.0f && s2[e] == 0.0f)) a = a / b;
    img[e] = a;
    ill[e] = b;
  }
}

// ---------------------------------------------------------------------------
// launchers
#define RTM_NFD_CASES(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12)

int interior_queue_rows(int epi, int nfd) {
  const bool pd1 = epi == EPI_RCV || epi == EPI_BORN || epi == EPI_BORN64 || epi == EPI_ADJ ||
                   epi == EPI_ADJT;
  return 2 * nfd + 1 + (pd1 ? 1 : 2);  // EpiTraits<EPI>::PD
}

hipError_t launch_interior(int epi, int nfd, IntArgs a, int nshot, hipStream_t s) {
  // rows per wave: the requested segment rounded to a multiple of the queue length
  const int ql = interior_queue_rows(epi, nfd);
  const int mult = a.zs > ql ? (a.zs + ql / 2) / ql : 1;
  a.zs = mult * ql;
  const int nseg = (a.g.mnz + a.zs - 1) / a.zs;
  a.nshot = nshot;
  // four shots per block on shared rows, or four row segments of one shot
  // per block when the launch has fewer than four shots (k_interior)
  dim3 grid(nshot >= 4 ? a.nxt * nseg * ((nshot + 3) / 4) : a.nxt * ((nseg + 3) / 4) * nshot);
#define CASE(N) case N: return StencilOps<N>::interior(epi, grid, a, s);
  switch (nfd) {
    RTM_NFD_CASES(CASE)
    default: return hipErrorInvalidValue;
  }
#undef CASE
}

// Interior rows start on a 128-byte line.  Tiles of 224 columns write whole
// lines; others write the lines at their sides in two parts, from two blocks,
// and each part is a masked write to memory.  Where the four buffers of a field
// exceed the 256 MB last-level cache that costs more than the tiles it saves:
// two forward steps of 128 shots of 351 x 1701 302 us (224 columns), 306 (240),
// 336 (248), with the images of four 1143, 1209, 1307; 32 shots forward 87, 90,
// 97; but 16 shots 57, 58, 51.
int two_cols(const Grid& g, int nfd, int nshot) {
  const long long bytes = 4ll * nshot * g.fstride * (long long)sizeof(float);
  return bytes > (256ll << 20) ? 224 : 256 - 2 * ((nfd + 3) & ~3);
}

int two_rows(int nfd, int rows) {
  const int ql = 2 * nfd + 3;
  return std::max(1, (rows + 2 * nfd + ql / 2) / ql) * ql - 2 * nfd;
}

hipError_t launch_two(int kind, int nfd, TwoArgs a, int nshot, hipStream_t s) {
  a.zs = two_rows(nfd, a.zs);
  a.cols = two_cols(a.g, nfd, nshot);
  a.nxt = (a.g.mnx + a.cols - 1) / a.cols;
  a.nshot = nshot;
  const int nseg = (a.g.mnz + a.zs - 1) / a.zs;
  const dim3 grid(a.nxt * nseg * ((nshot + TWO_SHOTS - 1) / TWO_SHOTS));
  switch (nfd) {
    case 1: return TwoOps<1>::two(kind, grid, a, s);
    case 2: return TwoOps<2>::two(kind, grid, a, s);
    case 3: return TwoOps<3>::two(kind, grid, a, s);
    case 4: return TwoOps<4>::two(kind, grid, a, s);
    case 5: return TwoOps<5>::two(kind, grid, a, s);
    default: return hipErrorInvalidValue;
  }
}

// The velocity of a frame cell's lateral term: its own on the top edge; Dv[(N2-x)*NX+y],
// the mirrored top-band cell, on the bottom edge (kernel.cu:132); Dv[(N2-y)*NX+x], a
// top-band cell, on the sides (kernel.cu:128, 136), where z may pass a row's end.
// Read by every step from here: a wave of side cells reading the velocities
// themselves touches a cache line per lane.
__global__ void k_frame_lat(const Grid g, int nx, const float* v, float taoh2, bool keep_corners,
                            float* fs) {
  const long long n = (long long)g.nz * nx;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const int z = (int)(i / nx), x = (int)(i % nx);
    const int ar = min(min(z, x), min(g.nz - 1 - z, nx - 1 - x));
    const bool top = z == ar, bot = !top && z == g.nz - 1 - ar;
    if (keep_corners && (z - ar <= 1 || g.nz - 1 - ar - z <= 1) && (x - ar <= 1 || nx - 1 - ar - x <= 1))
      continue;
    const int zq = top ? z : (bot ? ar : min(ar + z / nx, g.nz - 1));
    const int xq = (top || bot) ? x : z % nx;
    const float vq = v[(long long)zq * g.pitch + g.x0 + xq];
    fs[(long long)z * g.pitch + g.x0 + x] = (taoh2 * vq) * vq;
  }
}

// A thread per cell of the padded layout.
__global__ void k_coef_planes(const Grid g, const Model m, long long wo, int nfd, float* cp) {
  const long long fs = g.fstride, n = (long long)g.nz * g.pitch;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const float* row = m.ctab + m.ko[wo + i] / 4u;
    for (int l = 0; l <= nfd; ++l) cp[l * fs + i] = row[l];
    cp[(nfd + 1) * fs + i] = m.pm[wo + i];
    const float tv = m.taoh * m.v[wo + i];
    cp[(nfd + 2) * fs + i] = tv;
    cp[(nfd + 3) * fs + i] = 1.0f / (tv + 1.0f);
  }
}

int frame_segment_rows(int nfd) {
  const int nb = nfd > 2 ? nfd : 2;
  return 2 * (nb + nfd + 1 + 2) - 2;  // two register-queue cycles per side run
}
// Float4 windows of the top and bottom bands: first column n2, 248 apart,
// writing [cs+4, min(cs+252, frame4_end)).  None when the band's edge cells do
// not reach one window or n2 leaves no room for the column halo.
int frame4_windows(const Grid& g, int nx) {
  const int wend = frame4_end(g.n2, nx);
  if (g.n2 < 12 || nx < 2 * g.n2 || wend <= g.n2 + 4) return 0;
  return (wend - (g.n2 + 4) + 247) / 248;
}

void frame_records(const Grid& g, int nx, int shot, int seg_tb, int seg, int kind, int4* out,
                   int* count) {
  int n = 0;
  auto put = [&](int z0, int cx0, int band, int rows, int ncol) {
    if (out) out[n] = make_int4(z0, cx0, band | (rows << 4) | (ncol << 20), shot);
    ++n;
  };
  const int nw = kind == FRAME_ALL ? 0 : frame4_windows(g, nx);
  // top band, bottom band, in runs of seg_tb rows (the float4 records: one
  // run of the whole band, each wave writing 248 columns)
  const int run = kind == FRAME_VEC ? g.n2 : seg_tb;
  for (int b = 0; b < 2; ++b) {
    const int zb = b == 0 ? 0 : g.nz - g.n2, ze = b == 0 ? g.n2 : g.nz;
    for (int z0 = zb; z0 < ze; z0 += run) {
      const int rows = std::min(run, ze - z0);
      if (nw == 0) {
        if (kind != FRAME_VEC)
          for (int cx0 = -1; cx0 + 1 < nx; cx0 += 62) put(z0, cx0, b, rows, 0);
      } else if (kind == FRAME_VEC) {
        for (int w = 0; w < nw; ++w) put(z0, g.n2 + 248 * w, b, rows, 0);
      } else {  // the columns left to the scalar kernel
        for (int c = 0; c < g.n2 + 4; c += 62) put(z0, c - 1, b, rows, std::min(62, g.n2 + 4 - c));
        for (int c = frame4_end(g.n2, nx); c < nx; c += 62) put(z0, c - 1, b, rows, std::min(62, nx - c));
      }
    }
  }
  if (kind == FRAME_VEC) {
    *count = n;
    return;
  }
  // side bands: both in one wave per row run (band 4) when each fits in half
  // a wave with its inner neighbour and the halves do not overlap
  const bool pack = g.n2 <= 30 && nx >= 64;
  for (int z0 = g.n2; z0 < g.nz - g.n2; z0 += seg) {
    const int rows = std::min(seg, g.nz - g.n2 - z0);
    if (pack) {
      put(z0, 0, 4, rows, 0);
      continue;
    }
    for (int cx0 = -1; cx0 + 1 < g.n2; cx0 += 62) put(z0, cx0, 2, rows, 0);
    for (int cx0 = nx - g.n2 - 1; cx0 + 1 < nx; cx0 += 62) put(z0, cx0, 3, rows, 0);
  }
  *count = n;
}

bool frame4_supported(int nfd) { return nfd >= 1 && nfd <= 6; }

hipError_t launch_frame4(int mode, int nfd, FrameArgs a, int nshot, int nrec, hipStream_t s) {
  a.nshot = nshot;
  a.nrec = nrec;
  if (nrec == 0) return hipSuccess;
  dim3 grid((nrec + 3) / 4);  // one wave per record
#define CASE(N) case N: return StencilOps<N>::frame4(mode, grid, a, s);
  switch (nfd) {
    CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6)
    default: return hipErrorInvalidValue;
  }
#undef CASE
}

hipError_t launch_frame_quad(int mode, int nfd, FrameArgs a, int nshot, int nrec, hipStream_t s) {
  a.nshot = nshot;
  a.nrec = nrec;
  if (mode != FR_RCV) a.rbps = 0;
  a.qrows = std::min(a.qrows, QUAD_MAX_ROWS);
  a.nquad = 2 * a.qwin * ((a.g.n2 + a.qrows - 1) / a.qrows) * ((nshot + TWO_SHOTS - 1) / TWO_SHOTS);
  const dim3 grid(a.nquad + (nrec + 3) / 4 + (a.rbps > 0 ? a.rbps * nshot * a.nrf : 0));
  switch (nfd) {
    case 1: return StencilOps<1>::frame_quad(mode, grid, a, s);
    case 2: return StencilOps<2>::frame_quad(mode, grid, a, s);
    case 3: return StencilOps<3>::frame_quad(mode, grid, a, s);
    case 4: return StencilOps<4>::frame_quad(mode, grid, a, s);
    case 5: return StencilOps<5>::frame_quad(mode, grid, a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_frame(int mode, int nfd, FrameArgs a, int nshot, int nrec, hipStream_t s) {
  a.nshot = nshot;
  a.nrec = nrec;
  if (mode != FR_RCV && mode != FR_ADJ) a.rbps = 0;
  // one wave per (region run, shot) record, then the restore blocks
  dim3 grid((nrec + 3) / 4 + (a.rbps > 0 ? a.rbps * nshot * a.nrf : 0));
#define CASE(N) case N: return StencilOps<N>::frame(mode, grid, a, s);
  switch (nfd) {
    RTM_NFD_CASES(CASE)
    default: return hipErrorInvalidValue;
  }
#undef CASE
}

// The interior grid of launch_interior (rows per wave rounded to the queue
// length) and one wave per frame record, in one k_step launch; only the
// forward and the receiver step are fused (the other kinds keep two
// launches).
bool step_fusable(int epi, int mode) {
  return (epi == EPI_FWD && mode == FR_FWD) || ((epi == EPI_RCV || epi == EPI_RCV0) && mode == FR_RCV);
}

hipError_t launch_step(int epi, int mode, int nfd, IntArgs ia, FrameArgs fa, int nshot, int nrec,
                       hipStream_t s) {
  if (!step_fusable(epi, mode)) return hipErrorInvalidValue;
  const int ql = interior_queue_rows(epi, nfd);
  const int mult = ia.zs > ql ? (ia.zs + ql / 2) / ql : 1;
  ia.zs = mult * ql;
  const int nseg = (ia.g.mnz + ia.zs - 1) / ia.zs;
  ia.nshot = nshot;
  const unsigned nint = (unsigned)(nshot >= 4 ? ia.nxt * nseg * ((nshot + 3) / 4)
                                              : ia.nxt * ((nseg + 3) / 4) * nshot);
  fa.nshot = nshot;
  fa.nrec = nrec;
  const unsigned nfr = (unsigned)((nrec + 3) / 4);
  if (nfr == 0 || nint == 0) return hipErrorInvalidValue;
  const unsigned nfu = (nfr + 7u) / 8u, niu = (nint + 7u) / 8u;
  dim3 grid((nfu + niu) * 8u);
#define CASE(N) case N: return StencilOps<N>::step(epi, grid, ia, fa, nint, nfr, s);
  switch (nfd) {
    RTM_NFD_CASES(CASE)
    default: return hipErrorInvalidValue;
  }
#undef CASE
}

hipError_t launch_tile(int pass, int nfd, const TileArgs& a, int nshot, long long cells,
                       hipStream_t s) {
  // Two cells per thread halve a tile's scalar work and share its column reads,
  // one gives twice the blocks and fewer registers.  Measured (two against
  // one): Born + adjoint at half-length 4, 22 M cells 143 / 157 ms, 1.4 M cells
  // 34.9 / 32.2; migration at half-length 2, 32 M cells 159 / 171, at 3 and
  // 23 M cells 40.5 / 40.0; at half-length 10 always slower (18.4 / 15.8).
  const long long from = (pass == TILE_BORN || pass == TILE_ADJ) ? 2500000 : 24000000;
  const int cpt = nfd <= TILE_CPT2_MAX_NFD && cells >= from ? 2 : 1;
  const int ntz = (a.g.nz + TILE_ROWS * cpt - 1) / (TILE_ROWS * cpt);
  const dim3 grid((unsigned)nshot, (unsigned)((a.g.nx + 63) / 64), (unsigned)ntz);
#define CASE(N) case N: return TileOps<N>::tile(pass, cpt, grid, a, s);
  switch (nfd) {
    RTM_NFD_CASES(CASE)
    default: return hipErrorInvalidValue;
  }
#undef CASE
}

static inline unsigned blocks_for(long long n, int per = 256, unsigned cap = 4096) {
  long long b = (n + per - 1) / per;
  if (b < 1) b = 1;
  return (unsigned)(b > cap ? cap : b);
}

// Neighbour-tap planes: for cell (z, c) of the padded layout (c the storage
// column) and l = 1..nfd, the tap-l coefficient of the rows of (z-l, c),
// (z+l, c), (z, c-l), (z, c+l) -- 0 off the grid.  Tap l
// sits at float l of a row.
__global__ void k_tap_planes(Grid g, const unsigned* ko, const float* ctab, int nfd, float* tp) {
  const long long n = (long long)g.nz * g.pitch;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const int z = (int)(i / g.pitch), c = (int)(i - (long long)z * g.pitch);
    for (int l = 1; l <= nfd; ++l) {
      const int zz[4] = {z - l, z + l, z, z};
      const int cc[4] = {c, c, c - l, c + l};
      for (int d = 0; d < 4; ++d) {
        float val = 0.0f;
        if (zz[d] >= 0 && zz[d] < g.nz && cc[d] >= 0 && cc[d] < g.pitch)
          val = ctab[ko[(long long)zz[d] * g.pitch + cc[d]] / 4u + l];
        tp[(long long)(4 * (l - 1) + d) * g.fstride + i] = val;
      }
    }
  }
}
hipError_t launch_tap_planes(const Grid& g, const unsigned* ko, const float* ctab, int nfd,
                             float* tp, hipStream_t s) {
  hipLaunchKernelGGL(k_tap_planes, dim3(blocks_for((long long)g.nz * g.pitch, 256, 2048)),
                     dim3(256), 0, s, g, ko, ctab, nfd, tp);
  return hipGetLastError();
}
hipError_t launch_frame_lat(const Grid& g, int nx, const float* v, float taoh2, bool keep_corners,
                            float* fs, hipStream_t s) {
  hipLaunchKernelGGL(k_frame_lat, dim3(blocks_for((long long)g.nz * nx, 256, 2048)), dim3(256), 0, s, g,
                     nx, v, taoh2, keep_corners, fs);
  return hipGetLastError();
}
hipError_t launch_coef_planes(const Grid& g, const Model& m, int win, int nfd, float* cp, hipStream_t s) {
  hipLaunchKernelGGL(k_coef_planes, dim3(blocks_for(g.fstride, 256, 2048)), dim3(256), 0, s, g, m,
                     (long long)win * m.mstride, nfd, cp);
  return hipGetLastError();
}
hipError_t launch_flag_reset(unsigned* flag, hipStream_t s) {
  hipLaunchKernelGGL(k_flag_reset, dim3(1), dim3(64), 0, s, flag);
  return hipGetLastError();
}
hipError_t launch_finite_check(const float* f, long long n, int k, unsigned* flag, hipStream_t s) {
  const long long n4 = n / 4;
  hipLaunchKernelGGL(k_finite_check, dim3(blocks_for(n4, 256, 2048)), dim3(256), 0, s,
                     reinterpret_cast<const float4*>(f), n4, k, flag);
  return hipGetLastError();
}
hipError_t launch_fill(float* p, long long n, float val, hipStream_t s) {
  hipLaunchKernelGGL(k_fill, dim3(blocks_for(n, 256, 8192)), dim3(256), 0, s, p, n, val);
  return hipGetLastError();
}
hipError_t launch_fwd_begin(const Grid& g, float* f0, float* f1, const ShotGeo* geo, float spike,
                            int nshot, hipStream_t s) {
  hipLaunchKernelGGL(k_fwd_begin, dim3(blocks_for((long long)g.nz * g.pitch, 256, 1024), nshot),
                     dim3(256), 0, s, g, f0, f1, geo, spike);
  return hipGetLastError();
}
static inline long long strip_size_host(const Grid& g) { return 2LL * g.nfd * (g.mnz + g.mnx); }
int strip_restore_blocks(const Grid& g) { return (int)blocks_for(strip_size_host(g), 1024); }
hipError_t launch_strip_save(const Grid& g, const float* f, Strips st, const ShotGeo* geo, int k,
                             int nshot, hipStream_t s) {
  hipLaunchKernelGGL(k_strip_save, dim3(blocks_for(strip_size_host(g)), nshot), dim3(256), 0, s, g,
                     f, st, geo, k);
  return hipGetLastError();
}
hipError_t launch_strip_finish(const Grid& g, Strips st, const ShotGeo* geo, int k, int nshot,
                               hipStream_t s) {
  hipLaunchKernelGGL(k_strip_amax, dim3(blocks_for(strip_size_host(g), 256, 64), nshot), dim3(256),
                     0, s, g, st, geo, k);
  hipLaunchKernelGGL(k_strip_finish, dim3(blocks_for(strip_size_host(g)), nshot), dim3(256), 0, s,
                     g, st, geo, k);
  return hipGetLastError();
}
hipError_t launch_strip_restore(const Grid& g, float* f, Strips st, const ShotGeo* geo, int k,
                                int nshot, hipStream_t s) {
  hipLaunchKernelGGL(k_strip_restore, dim3(blocks_for(strip_size_host(g)), nshot), dim3(256), 0, s,
                     g, f, st, geo, k);
  return hipGetLastError();
}
hipError_t launch_snap_save(const Grid& g, const float* f, Snaps sn, const ShotGeo* geo, int slot,
                            int nshot, hipStream_t s) {
  const long long n = (long long)g.nz * g.nx;
  if (sn.fmt != 0) {
    hipLaunchKernelGGL(k_snap_clear, dim3(blocks_for(nshot)), dim3(256), 0, s, sn, slot, nshot);
    hipLaunchKernelGGL(k_snap_amax, dim3(blocks_for(n, 256, 512), nshot), dim3(256), 0, s, g, f, sn,
                       geo, slot);
  }
  hipLaunchKernelGGL(k_snap_save, dim3(blocks_for(n, 256, 1024), nshot), dim3(256), 0, s, g, f, sn,
                     geo, slot);
  return hipGetLastError();
}
hipError_t launch_snap_restore(const Grid& g, float* f, Snaps sn, const ShotGeo* geo, int slot,
                               int nshot, hipStream_t s) {
  const long long n = (long long)g.nz * g.nx;
  hipLaunchKernelGGL(k_snap_restore, dim3(blocks_for(n, 256, 1024), nshot), dim3(256), 0, s, g, f,
                     sn, geo, slot);
  return hipGetLastError();
}
hipError_t launch_record(const Grid& g, const Rcv& r, const ShotGeo* geo, const float* f,
                         float* rec, int k, int nt, int nshot, hipStream_t s) {
  hipLaunchKernelGGL(k_record, dim3(blocks_for(r.n), nshot), dim3(256), 0, s, g, r, geo, f, rec, k,
                     nt);
  return hipGetLastError();
}
hipError_t launch_bwd_begin(const Grid& g, const float* s0, const float* s1, float* q0, float* q1,
                            float* su, float* sq, float* i1, float* i2, const ShotGeo* geo,
                            float spike, int icompen, int nshot, hipStream_t s) {
  hipLaunchKernelGGL(k_bwd_begin, dim3(blocks_for((long long)g.nz * g.pitch, 256, 1024), nshot),
                     dim3(256), 0, s, g, s0, s1, q0, q1, su, sq, i1, i2, geo, spike, icompen);
  return hipGetLastError();
}
hipError_t launch_maxabs(const Grid& g, const ShotGeo* geo, const float* i2, unsigned* out,
                         int nshot, hipStream_t s) {
  hipLaunchKernelGGL(k_maxabs, dim3(blocks_for((long long)g.mnz * g.mnx, 256, 256), nshot),
                     dim3(256), 0, s, g, geo, i2, out);
  return hipGetLastError();
}
hipError_t launch_post(const Grid& g, const ShotGeo* geo, const float* v, long long mstride,
                       const float* i1, const float* i2, const unsigned* amax, float vmax,
                       float whitecoe, float* up, float* down, int nshot, hipStream_t s) {
  hipLaunchKernelGGL(k_post, dim3(blocks_for((long long)g.mnz * g.mnx, 256, 1024), nshot),
                     dim3(256), 0, s, g, geo, v, mstride, i1, i2, amax, vmax, whitecoe, up, down);
  return hipGetLastError();
}
hipError_t launch_stack_add(const Grid& g, const ShotGeo* geo, int gw, const float* up,
                            const float* down, float* s1, float* s2, int nshot, hipStream_t s) {
  hipLaunchKernelGGL(k_stack_add, dim3(blocks_for((long long)g.mnz * gw)), dim3(256), 0, s, g, geo,
                     gw, up, down, s1, s2, nshot);
  return hipGetLastError();
}
hipError_t launch_refl_scatter(const Grid& g, const ShotGeo* geo, int gw, const float* img,
                               float* dst, long long rstride, int nshot, hipStream_t s) {
  const int ny = rstride == 0 ? 1 : nshot;
  hipLaunchKernelGGL(k_refl_scatter, dim3(blocks_for((long long)g.nz * g.pitch), ny), dim3(256), 0,
                     s, g, geo, gw, img, dst, rstride);
  return hipGetLastError();
}

hipError_t launch_grad_stack(const Grid& g, const ShotGeo* geo, int gw, const float* G,
                             const float* pm, long long mstride, int nshot, float* grad,
                             hipStream_t s) {
  hipLaunchKernelGGL(k_grad_stack, dim3(blocks_for((long long)g.mnz * gw)), dim3(256), 0, s, g, geo,
                     gw, G, pm, mstride, nshot, grad);
  return hipGetLastError();
}

int dot64_part_size() { return DOT_BLOCKS; }

hipError_t launch_dot64(const float* a, const float* b, long long n, long long stride, int nvec,
                        double* part, double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_dot64_part, dim3(DOT_BLOCKS, nvec), dim3(256), 0, s, a, b, n, stride,
                     part);
  hipLaunchKernelGGL(k_dot64_final, dim3(nvec), dim3(256), 0, s, part, DOT_BLOCKS, out);
  return hipGetLastError();
}

hipError_t launch_axpy(float* y, const float* x, float a, long long n, hipStream_t s) {
  hipLaunchKernelGGL(k_axpy, dim3(blocks_for(n)), dim3(256), 0, s, y, x, a, n);
  return hipGetLastError();
}

hipError_t launch_transpose(const float* in, float* out, int rows, int cols, hipStream_t s) {
  hipLaunchKernelGGL(k_transpose, dim3((cols + 31) / 32, (rows + 31) / 32), dim3(256), 0, s, in, out,
                     rows, cols);
  return hipGetLastError();
}

hipError_t launch_stack_finish(int nI, const float* s1, const float* s2, int nrec, int inorm,
                               float* img, float* illum, hipStream_t s) {
  hipLaunchKernelGGL(k_stack_finish, dim3(blocks_for(nI)), dim3(256), 0, s, nI, s1, s2, nrec, inorm,
                     img, illum);
  return hipGetLastError();
}

}  // namespace rtm
