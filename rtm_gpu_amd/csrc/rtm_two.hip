// rtm_two.hip -- two time steps of the interior in one launch, for large
// batches; compiled once per stencil half-length (-DRTM_NFD=1..5).
//
// A step of one field moves 12 bytes per cell, two steps in one pass 16: u(t+1)
// and u(t+2) from u(t) and u(t-1), u(t+1) staying in registers.  The frame
// cells of u(t+1) that step t+2 reads (NFD deep around the interior) are in the
// buffer of u(t+1) already: the forward and receiver passes run the frame of
// t+1 first, the reconstruction restores its strips first.
//
// A wave marches 256 columns of one shot, computes u(t+1) on all of them and
// u(t+2) on the a.cols <= 256 - 2H in the middle, NFD rows behind: row z of u(t+1) comes
// from a register queue of u(t) rows and goes to a second queue, row z - NFD of
// u(t+2) comes from that one, with the oldest row of the first queue as its
// older operand.  A segment of zs rows takes zs + 2 NFD iterations.
//
// The four waves of a block march four shots over the same cells of one model
// window, row by row together: the window's coefficients are loaded as planes
// (one float per cell and coefficient, coalesced), each plane by one wave, two
// rows ahead, and shared through a ring of LDS rows, where the second step finds
// them again NFD rows later.  With a gather of every cell's coefficient row per
// wave and step, the L1 is what such a kernel waits for: two steps took 401 us
// at half-length 3 (128 reverse-VSP shots), one step per launch 2 x 212.
// Measured on 128 shots of 351 x 1701, us for two steps (two launches of
// k_interior): forward 298 (424) at half-length 3, 354 (532) at 5; the receiver
// field, four steps with their images, 1434 (1790).  Counters at half-length 4:
// 1.59 GB for two forward steps (1.22 are the fields, the rest halo rows and
// columns) and 6.10 GB with the images of four, 5.2-5.3 TB/s, the rate of a
// streaming kernel (5.3).  Imaging operands loaded a row ahead (253 registers)
// changed nothing.  At half-length 6 the 256 registers of two waves per SIMD
// spill (469 against 510 us; 137 against 106 on 24 shots): not built.
//
// Every cell takes the operations of k_interior in their order: same bits.
#include <hip/hip_runtime.h>

#include "rtm_device.h"

namespace rtm {

template <int NFD, int KIND>
__global__ __launch_bounds__(256, 2) void k_two(const TwoArgs a) {
  constexpr bool RCV = KIND == TWO_RCV0 || KIND == TWO_RCV, IMG = KIND == TWO_RCV;
  constexpr bool F64 = KIND == TWO_FWD64 || KIND == TWO_SRC;  // "2.0*" combine
  constexpr int H = (NFD + 3) & ~3;
  constexpr int PD = 2;  // rows of look-ahead, of the fields and of the planes
  constexpr int QL = 2 * NFD + 1 + PD;
  constexpr int W4 = 64 + 2 * (H / 4);
  constexpr int NWIN = 1 + 2 * (H / 4);
  constexpr int NP = NFD + 2;  // planes: c_0 .. c_NFD, P
  constexpr int RS = NFD + 2;  // LDS rows of planes: z - NFD .. z + 1
  __shared__ float4 cf[RS][NP][64];
  __shared__ float4 ex[4][2][W4];

  const Grid& g = a.g;
  const Model& m = a.m;
  const int WC = a.cols, M = (256 - WC) / 2;  // M >= H, a multiple of 4
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // blocks shot group fastest, as k_interior's
  const unsigned nsg = ((unsigned)a.nshot + 3u) >> 2;
  const int sw = (int)(blockIdx.x % nsg) * TWO_SHOTS + wv;
  const int tile = (int)(blockIdx.x / nsg);
  const bool live = sw < a.nshot;  // a wave past the batch only loads planes
  const int shot = live ? sw : a.nshot - 1;
  const int zseg = tile / a.nxt, xt = tile % a.nxt;
  const ShotGeo sg = a.geo[shot];
  const int n2 = g.n2, zhi = g.nz - n2, zlast = g.nz - 1;
  const int zs = n2 + zseg * a.zs, ze = min(zs + a.zs, zhi);  // rows written
  const int cend = sg.nx - n2;
  const int cb = n2 + xt * WC;  // first column written
  if (zs >= zhi || cb >= cend) return;     // the same for the block's shots
  const int cw = min(cb + WC, cend);  // first column not written
  const int c0 = cb - M + lane * 4;
  const int clast = sg.nx - ((sg.nx - n2) & 3);
  const unsigned vcol = (unsigned)(g.x0 + min(c0, clast)) * 4u;
  bool colok[4], wr[4], full = live, any_out = false;
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) {
    colok[jj] = c0 + jj >= n2 && c0 + jj < cend;
    wr[jj] = live && c0 + jj >= cb && c0 + jj < cw;
    full = full && wr[jj];
    any_out = any_out || !colok[jj];
  }
  const bool edge_tile = cend < cb + WC;  // the wave holds the interior's right edge
  const unsigned vst = (unsigned)(g.x0 + c0) * 4u, vst4 = full ? vst : kDrop;
  const unsigned vout = any_out ? vcol : kDrop;  // lanes with cells of u(t+1) off the interior
  unsigned vhal = kDrop;
  int hpos = H / 4 + lane;
  if (lane < H / 4) { vhal = (unsigned)max(g.x0 + cb - M - H + 4 * lane, 0) * 4u; hpos = lane; }
  else if (lane < 2 * (H / 4)) {
    vhal = (unsigned)(g.x0 + min(cb - M + 256 + 4 * (lane - H / 4), clast)) * 4u;
    hpos = 64 + lane;
  }

  const long long so = (long long)shot * g.fstride;
  const unsigned fb = (unsigned)g.fstride * 4u;
  const Rsrc R1 = rsrc(a.u1 + so, fb), R0 = rsrc(a.u0 + so, fb);
  const Rsrc RA = rsrc(a.ua + so, fb), RB = rsrc(a.ub + so, fb);
  // the wave's planes: wv, and wv + 4 where there is one
  const float* cp = a.cp + (long long)sg.win * a.cpstride;
  const bool second = wv + 4 < NP;
  const Rsrc RPA = rsrc(cp + (long long)min(wv, NP - 1) * g.fstride, fb);
  const Rsrc RPB = rsrc(cp + (long long)min(wv + 4, NP - 1) * g.fstride, second ? fb : 0u);
  const unsigned P4 = (unsigned)g.pitch * 4u;
  const float hzx2_1 = m.hzx2_1;
  const double h1 = m.h1;
  auto rowb = [=](int z) -> unsigned { return (unsigned)min(max(z, 0), zlast) * P4; };

  // source cell; receivers on row s_z: samples of the two steps
  const int srow = RCV ? a.r.s_z : sg.r_u;
  bool srcc[4];
  float da[4] = {0.f, 0.f, 0.f, 0.f}, db[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) srcc[jj] = c0 + jj == sg.r_x;
  if (RCV && srow >= zs - NFD && srow < ze + NFD) {
    Rcv rr = a.r;
    rr.s_l = sg.s_l;
    rr.s_r = sg.s_r;
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      int s;
      if (is_receiver(c0 + jj, rr, &s)) {  // step k takes sample k+1 (kernel.cu:349-354, 905-909)
        da[jj] = a.data[((long long)shot * a.nt + a.k + 1) * a.r.n + s];
        db[jj] = a.data[((long long)shot * a.nt + a.k) * a.r.n + s];
      }
    }
  }
  Rsrc RI1, RI2, RSU, RSQ, RU[4];
  unsigned vi = kDrop, vc = kDrop, vis = kDrop, vcs = kDrop, vu[2] = {kDrop, kDrop};
  if (IMG) {
    RI1 = rsrc(a.i1 + so, fb); RI2 = rsrc(a.i2 + so, fb);
    RSU = rsrc(a.su + so, fb); RSQ = rsrc(a.sq + so, fb);
#pragma unroll
    for (int i = 0; i < 4; ++i) RU[i] = rsrc(a.us[i] + so, fb);
    const bool any = wr[0] || wr[1] || wr[2] || wr[3];
    vi = any ? vcol : kDrop;
    vis = any ? vst : kDrop;
    if (a.icompen) { vc = vi; vcs = vis; }
    if (a.nimg >= 4) vu[0] = vi;
    if (a.nimg >= 3) vu[1] = vi;
  }

  // Values of a row: centre qc, column rows col(l), window win, coefficients and
  // P from LDS row cr, older field ov; source or data samples on row srow.
  const auto row4 = [&](const float4 (*cr)[64], const float4& qc, auto col, const float4* win,
                        const float4& ov, bool on_row, float wav, const float* dv,
                        float* out) __attribute__((always_inline)) {
    const float4 k0 = cr[0][lane], pv = cr[NFD + 1][lane];
    float w1[4];
#pragma unroll
    for (int jj = 0; jj < 4; ++jj)
      w1[jj] = (float)((h1 * (double)compr(k0, jj)) * (double)compr(qc, jj));
#pragma unroll
    for (int l = 1; l <= NFD; ++l) {
      const float4 kl = cr[l][lane];
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        float s = compr(col(-l), jj) + compr(col(l), jj);
        s = __builtin_fmaf(s, hzx2_1, compr(win[(H + jj - l) >> 2], (H + jj - l) & 3));
        s = s + compr(win[(H + jj + l) >> 2], (H + jj + l) & 3);
        w1[jj] = __builtin_fmaf(compr(kl, jj), s, w1[jj]);
      }
    }
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const float o = combine_p(compr(qc, jj), compr(ov, jj), compr(pv, jj), w1[jj], F64);
      if (RCV) out[jj] = (on_row && dv[jj] != 0.0f) ? dv[jj] : o;  // data replacement
      else out[jj] = (on_row && srcc[jj]) ? o + wav : o;           // source (kernel.cu:74-77, 277-280)
    }
  };
  const auto store4 = [&](Rsrc r, unsigned drop, unsigned row,
                          const float* o) __attribute__((always_inline)) {
    bst4s(r, vst4 | drop, row, o[0], o[1], o[2], o[3]);
    if (edge_tile) {
#pragma unroll
      for (int jj = 0; jj < 3; ++jj)
        bst1s_(r, ((wr[jj] && !full) ? vst + 4u * jj : kDrop) | drop, row, o[jj]);
    }
  };

  const int zb = zs - NFD;  // row of u(t+1) of the first iteration
  auto vring = [=](int z) -> unsigned { return z < n2 || z >= zhi ? vcol : vout; };
  float4 q[QL], r[QL];      // rows of u(t), of u(t+1)
#pragma unroll
  for (int s = 0; s < QL; ++s) r[s] = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 pa[PD + 1], pb[PD + 1];  // planes of rows z+1 .. z+1+PD
  pa[0] = bld4(RPA, vcol, rowb(zb));
  pb[0] = bld4(RPB, vcol, rowb(zb));
#pragma unroll
  for (int s = 0; s < 2 * NFD + PD; ++s) q[s] = bld4(R1, vcol, rowb(zb - NFD + s));
  float4 hvb[PD + 1], u0b[PD + 1], rgb[2];
#pragma unroll
  for (int d = 0; d < PD; ++d) {
    u0b[d] = bld4s(R0, vcol, rowb(zb + d));
    hvb[d] = bld4(R1, vhal, rowb(zb + d));
  }
  rgb[0] = bld4(RA, vring(zb), rowb(zb));
  // LDS rows: row zb in slot 0; the slots read before they are filled (rows
  // above the segment) only feed rows that are not written
  if (wv < NP) cf[0][wv][lane] = pa[0];
  if (second) cf[0][wv + 4][lane] = pb[0];
#pragma unroll
  for (int d = 0; d < PD; ++d) {
    pa[d] = bld4(RPA, vcol, rowb(zb + 1 + d));
    pb[d] = bld4(RPB, vcol, rowb(zb + 1 + d));
  }
  block_lds_sync();

  int s1 = 0, s2 = RS - NFD;  // LDS slots of rows zz and zz - NFD
  for (int z = zb; z < ze + NFD; z += QL) {
#pragma unroll
    for (int j = 0; j < QL; ++j) {
      const int zz = z + j, z2 = zz - NFD;
      // imaging operands of row z2, ahead of the look-ahead so that their wait
      // leaves it in flight
      float4 iu[4] = {}, ii1 = {}, ii2 = {}, isu = {}, isq = {}, iq = {};
      if (IMG) {
        const unsigned rz = rowb(z2);
        iu[0] = bld4s(RU[0], vu[0], rz);
        iu[1] = bld4s(RU[1], vu[1], rz);
        iu[2] = bld4(RU[2], vi, rz);
        iu[3] = bld4(RU[3], vi, rz);
        ii1 = bld4s(RI1, vi, rz);
        ii2 = bld4s(RI2, vi, rz);
        isu = bld4s(RSU, vc, rz);
        isq = bld4s(RSQ, vc, rz);
        iq = bld4s(R0, vu[0], rz);
      }
      // operands of later rows
      q[(j + 2 * NFD + PD) % QL] = bld4(R1, vcol, rowb(zz + NFD + PD));
      u0b[PD] = bld4s(R0, vcol, rowb(zz + PD));
      hvb[PD] = bld4(R1, vhal, rowb(zz + PD));
      rgb[1] = bld4(RA, vring(zz + 1), rowb(zz + 1));
      pa[PD] = bld4(RPA, vcol, rowb(zz + 1 + PD));
      pb[PD] = bld4(RPB, vcol, rowb(zz + 1 + PD));
      __builtin_amdgcn_sched_barrier(0);
      // planes of row zz + 1
      const int sn = s1 + 1 == RS ? 0 : s1 + 1;
      if (wv < NP) cf[sn][wv][lane] = pa[0];
      if (second) cf[sn][wv + 4][lane] = pb[0];
      // row zz of u(t+1)
      const float4 qc = q[(j + NFD) % QL];
      ex[wv][0][hpos] = hvb[0];
      ex[wv][0][H / 4 + lane] = qc;
      wave_lds_sync();
      float4 win[NWIN];
#pragma unroll
      for (int t = 0; t < NWIN; ++t) win[t] = ex[wv][0][lane + t];
      float oa[4];
      row4(cf[s1], qc, [&](int l) { return q[(j + NFD + l) % QL]; }, win, u0b[0], zz == srow, a.wa, da, oa);
      store4(RA, zz >= zs && zz < ze ? 0u : kDrop, rowb(zz), oa);
      const bool in1 = zz >= n2 && zz < zhi;
      r[j] = make_float4(in1 && colok[0] ? oa[0] : rgb[0].x, in1 && colok[1] ? oa[1] : rgb[0].y,
                         in1 && colok[2] ? oa[2] : rgb[0].z, in1 && colok[3] ? oa[3] : rgb[0].w);
      // row z2 of u(t+2)
      const float4 rc = r[(j - NFD + QL) % QL];
      ex[wv][1][H / 4 + lane] = rc;
      wave_lds_sync();
#pragma unroll
      for (int t = 0; t < NWIN; ++t) win[t] = ex[wv][1][lane + t];
      float ob[4];
      row4(cf[s2], rc, [&](int l) { return r[(j - NFD + l + QL) % QL]; }, win, q[j], z2 == srow, a.wb, db, ob);
      const unsigned drop = z2 >= zs && z2 < ze ? 0u : kDrop;
      store4(RB, drop, rowb(z2), ob);
      if (IMG) {  // imaging (kernel.cu:489-517) of steps k+nimg-2 .. k-1, in that order
        float r1o[4], r2o[4], rsu[4], rsq[4];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          float x1 = compr(ii1, jj), x2 = compr(ii2, jj), su = compr(isu, jj), sq = compr(isq, jj);
          auto image = [&](float u, float qv, bool on) {  // cells off the interior keep their values
            const float a1 = a.icompen ? su + u : u, b1 = a.icompen ? sq + qv : qv;
            x1 = on ? __builtin_fmaf(b1, a1, x1) : x1;
            x2 = on ? __builtin_fmaf(u, u, x2) : x2;
            su = on ? a1 : su;
            sq = on ? b1 : sq;
          };
          image(compr(iu[0], jj), compr(iq, jj), wr[jj] && a.nimg >= 4);
          image(compr(iu[1], jj), compr(q[j], jj), wr[jj] && a.nimg >= 3);
          image(compr(iu[2], jj), compr(rc, jj), wr[jj]);
          image(compr(iu[3], jj), ob[jj], wr[jj]);
          r1o[jj] = x1; r2o[jj] = x2; rsu[jj] = su; rsq[jj] = sq;
        }
        const unsigned rz = rowb(z2);
        bst4s(RI1, vis | drop, rz, r1o[0], r1o[1], r1o[2], r1o[3]);
        bst4s(RI2, vis | drop, rz, r2o[0], r2o[1], r2o[2], r2o[3]);
        bst4s(RSU, vcs | drop, rz, rsu[0], rsu[1], rsu[2], rsu[3]);
        bst4s(RSQ, vcs | drop, rz, rsq[0], rsq[1], rsq[2], rsq[3]);
      }
#pragma unroll
      for (int d = 0; d < PD; ++d) {
        u0b[d] = u0b[d + 1]; hvb[d] = hvb[d + 1]; pa[d] = pa[d + 1]; pb[d] = pb[d + 1];
      }
      rgb[0] = rgb[1];
      s1 = sn;
      s2 = s2 + 1 == RS ? 0 : s2 + 1;
      block_lds_sync();
    }
  }
}

template <>
hipError_t TwoOps<RTM_NFD>::two(int kind, dim3 grid, const TwoArgs& a, hipStream_t s) {
  constexpr int N = RTM_NFD;
  const dim3 block(256);
  if (kind == TWO_FWD) hipLaunchKernelGGL((k_two<N, TWO_FWD>), grid, block, 0, s, a);
  else if (kind == TWO_FWD64) hipLaunchKernelGGL((k_two<N, TWO_FWD64>), grid, block, 0, s, a);
  else if (kind == TWO_SRC) hipLaunchKernelGGL((k_two<N, TWO_SRC>), grid, block, 0, s, a);
  else if (kind == TWO_RCV0) hipLaunchKernelGGL((k_two<N, TWO_RCV0>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((k_two<N, TWO_RCV>), grid, block, 0, s, a);
  return hipGetLastError();
}

}  // namespace rtm
