// rtm_stencil.hip -- hand-written gfx950 kernels of the 2-D acoustic RTM step,
// compiled once per stencil half-length (-DRTM_NFD=1..12).
//
// Reference kernels (caixh90/RTM_GPU kernel.cu) and where their work lives here:
//   Add/Add_Con (46-114)            -> k_interior<EPI_FWD> + k_frame<FR_FWD> (two-way part)
//   Hybrid1/Hybrid2 (116-183)       -> k_frame<FR_FWD> (one-way + blend, from pre-blend values)
//   Equal/Hybrid3 (18-45, 184-208)  -> k_strip_save, and k_frame<FR_FWD> for k >= 2
//   Deliver/Deliver_EFF (210-221, 323-337) -> none: the host rotates buffer pointers
//   BKEqual (222-245)               -> k_strip_restore (into the buffer that becomes u(k+1))
//   BKAdd_EFF(_Con) (246-320)       -> k_interior<EPI_SRC>
//   BKAdd(_Con) (339-418)           -> k_interior<EPI_RCV> + k_frame<FR_RCV>
//   BKHybrid1/2 (421-487)           -> k_frame<FR_RCV>
//   Rel_Compen/Rel_NonCompen (489-517) -> k_interior<EPI_RCV> epilogue (interior only)
//
// Arithmetic follows the reference formulas operation by operation (build
// flags: -ffp-contract=off, IEEE division, denormals kept), with explicit
// fused multiply-adds only at the per-tap stencil sum, the tap accumulation,
// the FP32 final combine and the imaging accumulations.
#include <hip/hip_runtime.h>

#include "rtm_device.h"

namespace rtm {

// ---------------------------------------------------------------------------
// Interior update: cells [n2, nz-n2) x [n2, nx-n2).  One wave owns 256
// columns (4 per lane, float4 rows) and marches down a segment of rows.
// Vertical taps come from a register queue of rows; horizontal taps from a
// per-wave LDS row with a halo of H columns each side.  No mirror is needed:
// every tap stays inside the grid because NFD <= n2.
//
// Memory goes through buffer instructions: the per-shot base and size live in
// a scalar resource, the row offset in a scalar register, the column offset
// in a per-lane register that stays fixed along the march.  A lane that must
// not store gets a column offset at or above 2^31, past every buffer's size,
// and the hardware drops the access; the row body therefore has no branch.
//
// Software pipeline per row: (a) the coefficient rows of the row are gathered
// (their byte offsets were fetched PD rows earlier); (b) every stencil operand
// of row z+PD is fetched (u1 row z+NFD+PD, the halo row, u0, the p and offset
// rows); (c) the
// LDS exchange and the stencil read only data fetched in earlier iterations
// or in (a).  The memory counter is in-order, so (a) goes first: the wait on
// the gathers then leaves the prefetches in flight.  Scheduling barriers keep
// that order.  A segment is a multiple of the queue length QL, so the row
// loop is fully unrolled without a remainder; rows past the interior at the
// end of the last segment are computed from clamped rows and not stored.
//
// Imaging.  The sums and images are 32 of the 60 bytes that a backward step
// moved per cell when every step updated them.  The three rotating buffers of
// each field still hold steps k+2, k+1 and k when the receiver step k runs, and
// that step has q(k+2) and q(k+1) in registers as its own operands, so every
// third receiver step (EPI_RCV, nimg = 3) applies the terms of three steps in
// their order, bit for bit the same, and the two before it are plain updates
// (EPI_RCV0): (36 + 24 + 56) / 3 = 38.7 bytes per cell and backward step.
template <int EPI>
struct EpiTraits {
  static constexpr bool f64 =
      EPI == EPI_FWD64 || EPI == EPI_SRC || EPI == EPI_BORN64;  // "2.0*"
  static constexpr bool rcv = EPI == EPI_RCV || EPI == EPI_RCV0;  // receiver step
  static constexpr bool img = EPI == EPI_RCV;  // ... with the imaging of up to three steps
  static constexpr bool born = EPI == EPI_BORN || EPI == EPI_BORN64;
  static constexpr bool adj = EPI == EPI_ADJ || EPI == EPI_ADJT;
  static constexpr bool adjt = EPI == EPI_ADJT;  // transposed stencil (per-cell rows)
  static constexpr bool src = !rcv && !born && !adj;  // injects the source wavelet
  static constexpr int PD = (img || born || adj) ? 1 : 2;  // prefetch distance of the stencil operands
};

// Interior body for block bid (k_interior: bid = blockIdx.x; k_step gives
// the interior blocks of a launch shared with the frame their own numbering).
template <int NFD, int EPI>
__device__ __forceinline__ void interior_body(const IntArgs& a, const unsigned bid) {
  using T = EpiTraits<EPI>;
  constexpr int H = (NFD + 3) & ~3;
  constexpr int PD = T::PD;
  constexpr int QL = 2 * NFD + 1 + PD;
  constexpr int W4 = 64 + 2 * (H / 4);
  constexpr int NWIN = 1 + 2 * (H / 4);
  __shared__ float4 lds[4][W4];

  const Grid& g = a.g;
  const Model& m = a.m;
  const int lane = threadIdx.x & 63;
  // wave index: uniform in the wave, so row offsets derived from it stay scalar
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // The four waves of block b march the same rows and columns (tile
  // b / nsg) for four shots (group b % nsg; launches of at least four
  // shots), so their reads of the shared
  // model rows (p, coefficient offsets, coefficient rows) coincide in time and
  // hit the CU's L1.  Workgroups reach the eight XCDs round-robin by b, so
  // the blocks one XCD holds at a time are more shots of the same few tiles,
  // whose model reads hit that XCD's L2.
  // With fewer than four shots the waves of a block take four consecutive
  // row segments of one shot instead (block b: shot b % B, tile b / B).
  int shot, zseg;
  int tile;
  if (a.nshot >= 4) {
    const unsigned nsg = ((unsigned)a.nshot + 3u) >> 2;
    shot = (int)(bid % nsg) * 4 + wv;
    tile = (int)(bid / nsg);
    if (shot >= a.nshot) return;
    zseg = tile / a.nxt;
  } else {
    shot = (int)(bid % (unsigned)a.nshot);
    tile = (int)(bid / (unsigned)a.nshot);
    zseg = (tile / a.nxt) * 4 + wv;
  }
  const int xt = tile % a.nxt;
  const ShotGeo sg = a.geo[shot];
  const int zhi = g.nz - g.n2;
  const int zs = g.n2 + zseg * a.zs;  // a.zs is a multiple of QL
  const int cend = sg.nx - g.n2;                // first column past the shot's interior
  const int cb = g.n2 + xt * 256;
  if (zs >= zhi || cb >= cend) return;          // tiles past a narrower shot's width
  const int ze = zs + a.zs;
  const int c0 = cb + lane * 4;
  const int clast = sg.nx - ((sg.nx - g.n2) & 3);  // largest c == n2 (mod 4) with c <= nx
  const int cl = min(c0, clast);
  const unsigned vcol = (unsigned)(g.x0 + cl) * 4u;
  const unsigned vst = c0 < cend ? (unsigned)(g.x0 + c0) * 4u : kDrop;
  bool colok[4];
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) colok[jj] = c0 + jj < cend;
  // The last four columns of an interior row may reach 1..3 frame columns
  // (interior widths that are not multiples of 4).  Those belong to the frame
  // kernel, which may run in the same launch (k_step), so the lane holding
  // them stores its valid columns one by one; only the wave whose tile holds
  // the interior's right edge (uniform) issues those stores.
  const bool edge_tile = cend < cb + 256;
  const bool part = !colok[3];
  const unsigned vst4 = part ? kDrop : vst;

  // Halo columns: the first 2H/4 lanes fetch them; the others fetch nothing
  // (a dropped load returns 0) and write that to their own slot, which the
  // centre row overwrites right after.
  unsigned vhal = kDrop;
  int hpos = H / 4 + lane;
  if (lane < H / 4) { vhal = (unsigned)(g.x0 + min(cb - H + 4 * lane, clast)) * 4u; hpos = lane; }
  else if (lane < 2 * (H / 4)) { vhal = (unsigned)(g.x0 + min(cb + 256 + 4 * (lane - H / 4), clast)) * 4u; hpos = 64 + lane; }

  const long long so = (long long)shot * g.fstride;
  const unsigned fb = (unsigned)g.fstride * 4u;
  const Rsrc R1 = rsrc(a.u1 + so, fb), R0 = rsrc(a.u0 + so, fb), R2 = rsrc(a.u2 + so, fb);
  const long long mo = (long long)sg.win * m.mstride;
  const Rsrc RP = rsrc(m.pm + mo, fb), RK = rsrc(m.ko + mo, fb);
  const Rsrc RC = rsrc(m.ctab, (unsigned)(m.nrow * m.cs) * 4u);
  const unsigned P4 = (unsigned)g.pitch * 4u;
  auto rowb = [&](int z) -> unsigned { return (unsigned)min(z, g.nz - 1) * P4; };
  Rsrc RTP;
  if (T::adjt) RTP = rsrc(m.tp + (long long)sg.win * m.tpstride, (unsigned)(4 * NFD) * fb);

  const int2 sp = make_int2(sg.r_u, sg.r_x);
  Rcv rr = a.r;  // this shot's receivers; a.r.n stays the stride of the data layout
  rr.s_l = sg.s_l;
  rr.s_r = sg.s_r;
  bool srcc[4];
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) srcc[jj] = c0 + jj == sp.y;

  // receiver step: data replacement of row s_z (kernel.cu:349-354), read once;
  // adjoint: the residual of step k added (times P) at the receivers
  float dval[4] = {0.f, 0.f, 0.f, 0.f};
  bool rflag[4] = {false, false, false, false};
  if ((T::rcv || T::adj) && a.r.s_z >= zs && a.r.s_z < min(ze, zhi)) {
    const int kd = T::rcv ? a.k + 1 : a.k;
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      int s;
      if (colok[jj] && is_receiver(c0 + jj, rr, &s)) {
        dval[jj] = a.data[((long long)shot * a.nt + kd) * a.r.n + s];
        rflag[jj] = true;
      }
    }
  }
  Rsrc RU, RU1, RU2, RI1, RI2, RSU, RSQ;
  unsigned vcs = kDrop, vss = kDrop, vu1 = kDrop, vu2 = kDrop;
  if (T::img) {
    RU = rsrc(a.uk + so, fb); RU1 = rsrc(a.ua + so, fb); RU2 = rsrc(a.ub + so, fb);
    RI1 = rsrc(a.i1 + so, fb); RI2 = rsrc(a.i2 + so, fb);
    RSU = rsrc(a.su + so, fb); RSQ = rsrc(a.sq + so, fb);
    if (a.icompen) { vcs = vcol; vss = vst; }
    if (a.nimg >= 2) vu1 = vcol;
    if (a.nimg >= 3) vu2 = vcol;
  }
  // Born / adjoint operands of the centre row: the background fields and the
  // reflectivity (Born) or the gradient accumulator (adjoint, when imaging)
  Rsrc RA, RB, RCC, RX;
  unsigned vxl = kDrop, vxs = kDrop;
  if (T::born || T::adj) {
    RA = rsrc(a.ua + so, fb); RB = rsrc(a.ub + so, fb); RCC = rsrc(a.uc + so, fb);
    RX = T::born ? rsrc(m.refl + (long long)shot * m.rstride, fb) : rsrc(a.i1 + so, fb);
    if (T::born || a.image) { vxl = vcol; vxs = vst; }
  }

  float4 q[QL];
#pragma unroll
  for (int s = 0; s < 2 * NFD + PD; ++s) q[s] = bld4(R1, vcol, rowb(zs - NFD + s));
  float4 hvb[PD + 1], u0b[PD + 1], pb[PD + 1];
  uint4 kb[PD + 1];
#pragma unroll
  for (int d = 0; d < PD; ++d) {
    kb[d] = bld4u(RK, vcol, rowb(zs + d));
    pb[d] = bld4(RP, vcol, rowb(zs + d));
    u0b[d] = bld4s(R0, vcol, rowb(zs + d));
    hvb[d] = bld4(R1, vhal, rowb(zs + d));
  }
  float4 ukb = {}, uk1b = {}, uk2b = {}, i1b = {}, i2b = {}, sub = {}, sqb = {};
  float4 xab[2], xbb[2], xcb[2], xxb[2];
  if (T::born || T::adj) {
    xab[0] = bld4(RA, vxl, rowb(zs));
    xbb[0] = bld4(RB, vxl, rowb(zs));
    xcb[0] = bld4(RCC, vxl, rowb(zs));
    xxb[0] = bld4(RX, vxl, rowb(zs));
  }

  for (int z = zs; z < ze; z += QL) {
#pragma unroll
    for (int j = 0; j < QL; ++j) {
      const int zz = z + j;
      // (a) coefficient rows of this row (transposed stencil: the cells' own
      // c0' and the neighbour-tap planes of the row)
      CoefRow<T::adjt ? 1 : NFD> cr[4];
      float4 tpv[T::adjt ? 4 * NFD : 1];
      if (T::adjt) {
        cr[0].r[0] = bld4(RC, kb[0].x, 0);
        cr[1].r[0] = bld4(RC, kb[0].y, 0);
        cr[2].r[0] = bld4(RC, kb[0].z, 0);
        cr[3].r[0] = bld4(RC, kb[0].w, 0);
#pragma unroll
        for (int t = 0; t < 4 * NFD; ++t) tpv[t] = bld4(RTP, vcol, rowb(zz) + (unsigned)t * fb);
      } else {
        cr[0].load(RC, kb[0].x);
        cr[1].load(RC, kb[0].y);
        cr[2].load(RC, kb[0].z);
        cr[3].load(RC, kb[0].w);
      }
      __builtin_amdgcn_sched_barrier(0);
      // Imaging receiver step: this row's imaging operands, issued ahead of
      // the prefetches so that their wait leaves the prefetches in flight (a
      // row of look-ahead for them would cost VGPRs the kernel needs).
      if (T::img) {
        const unsigned rzz = rowb(zz);
        ukb = bld4(RU, vcol, rzz);
        uk1b = bld4(RU1, vu1, rzz);
        uk2b = bld4s(RU2, vu2, rzz);
        i1b = bld4s(RI1, vcol, rzz);
        i2b = bld4s(RI2, vcol, rzz);
        sub = bld4s(RSU, vcs, rzz);
        sqb = bld4s(RSQ, vcs, rzz);
      }
      // (b) operands of later rows
      q[(j + 2 * NFD + PD) % QL] = bld4(R1, vcol, rowb(zz + NFD + PD));
      kb[PD] = bld4u(RK, vcol, rowb(zz + PD));
      pb[PD] = bld4(RP, vcol, rowb(zz + PD));
      u0b[PD] = bld4s(R0, vcol, rowb(zz + PD));
      hvb[PD] = bld4(R1, vhal, rowb(zz + PD));
      if (T::born || T::adj) {
        xab[1] = bld4(RA, vxl, rowb(zz + 1));
        xbb[1] = bld4(RB, vxl, rowb(zz + 1));
        xcb[1] = bld4(RCC, vxl, rowb(zz + 1));
        xxb[1] = bld4(RX, vxl, rowb(zz + 1));
      }
      __builtin_amdgcn_sched_barrier(0);
      // (c) horizontal neighbours through LDS
      const float4 qc = q[(j + NFD) % QL];
      lds[wv][hpos] = hvb[0];
      lds[wv][H / 4 + lane] = qc;
      wave_lds_sync();
      float4 win[NWIN];
#pragma unroll
      for (int t = 0; t < NWIN; ++t) win[t] = lds[wv][lane + t];
      wave_lds_sync();

      const float4 pv = pb[0], u0v = u0b[0];
      float out[4];
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const float u = compr(qc, jj);
        float w1 = (float)(cr[jj].c0d(m.h1) * (double)u);
        if (T::adjt) {  // each tap with the neighbour's coefficient: (L^T mu)
#pragma unroll
          for (int l = 1; l <= NFD; ++l) {
            const float cu = compr(tpv[4 * (l - 1)], jj), cd = compr(tpv[4 * (l - 1) + 1], jj);
            const float cl = compr(tpv[4 * (l - 1) + 2], jj), cr2 = compr(tpv[4 * (l - 1) + 3], jj);
            const float vs = __builtin_fmaf(cu, compr(q[(j + NFD - l) % QL], jj),
                                            cd * compr(q[(j + NFD + l) % QL], jj));
            float s = __builtin_fmaf(vs, m.hzx2_1,
                                     cl * compr(win[(H + jj - l) >> 2], (H + jj - l) & 3));
            s = __builtin_fmaf(cr2, compr(win[(H + jj + l) >> 2], (H + jj + l) & 3), s);
            w1 = w1 + s;
          }
        } else {
#pragma unroll
          for (int l = 1; l <= NFD; ++l) {
            float s = compr(q[(j + NFD - l) % QL], jj) + compr(q[(j + NFD + l) % QL], jj);
            s = __builtin_fmaf(s, m.hzx2_1, compr(win[(H + jj - l) >> 2], (H + jj - l) & 3));
            s = s + compr(win[(H + jj + l) >> 2], (H + jj + l) & 3);
            w1 = __builtin_fmaf(cr[jj].c(l), s, w1);
          }
        }
        float o = combine_p(u, compr(u0v, jj), compr(pv, jj), w1, T::f64);
        if (T::src)       // source (kernel.cu:74-77, 277-280)
          o = (zz == sp.x && srcc[jj]) ? o + a.wav : o;
        else if (T::rcv)  // data replacement
          o = (zz == a.r.s_z && dval[jj] != 0.0f) ? dval[jj] : o;
        else if (T::adj)  // residual injection, P * r(k)
          o = (zz == a.r.s_z && rflag[jj]) ? o + compr(pv, jj) * dval[jj] : o;
        if (T::born) {    // scattering source m * D2u(k)
          const float d2u = (compr(xab[0], jj) - 2.0f * compr(xbb[0], jj)) + compr(xcb[0], jj);
          o = __builtin_fmaf(compr(xxb[0], jj), d2u, o);
        }
        out[jj] = o;
      }
      const unsigned rowdrop = zz < zhi ? 0u : kDrop;
      const unsigned rz = rowb(zz);
      bst4s(R2, vst4 | rowdrop, rz, out[0], out[1], out[2], out[3]);
      if (edge_tile) {
#pragma unroll
        for (int jj = 0; jj < 3; ++jj)
          bst1s_(R2, ((part && colok[jj]) ? vst + 4u * jj : kDrop) | rowdrop, rz, out[jj]);
      }
      if (T::img) {  // imaging (kernel.cu:489-517) of steps k+nimg-1 .. k, in that order
        float r1o[4], r2o[4], rsu[4], rsq[4];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          float x1 = compr(i1b, jj), x2 = compr(i2b, jj), su = compr(sub, jj), sq = compr(sqb, jj);
          auto image = [&](float u, float q, bool on) {  // frame columns keep their values
            const float a1 = a.icompen ? su + u : u, b1 = a.icompen ? sq + q : q;
            x1 = on ? __builtin_fmaf(b1, a1, x1) : x1;
            x2 = on ? __builtin_fmaf(u, u, x2) : x2;
            su = on ? a1 : su;
            sq = on ? b1 : sq;
          };
          image(compr(uk2b, jj), compr(u0v, jj), colok[jj] && a.nimg >= 3);
          image(compr(uk1b, jj), compr(qc, jj), colok[jj] && a.nimg >= 2);
          image(compr(ukb, jj), out[jj], colok[jj]);
          r1o[jj] = x1; r2o[jj] = x2; rsu[jj] = su; rsq[jj] = sq;
        }
        bst4s(RI1, vst | rowdrop, rz, r1o[0], r1o[1], r1o[2], r1o[3]);
        bst4s(RI2, vst | rowdrop, rz, r2o[0], r2o[1], r2o[2], r2o[3]);
        bst4s(RSU, vss | rowdrop, rz, rsu[0], rsu[1], rsu[2], rsu[3]);
        bst4s(RSQ, vss | rowdrop, rz, rsq[0], rsq[1], rsq[2], rsq[3]);
      }
      if (T::adj) {  // G += D2u(k+1) * mu(k+2); mu(k+2) is this update's u0
        float go[4];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const float d2u = (compr(xab[0], jj) - 2.0f * compr(xbb[0], jj)) + compr(xcb[0], jj);
          const float gi = compr(xxb[0], jj);
          go[jj] = colok[jj] ? __builtin_fmaf(d2u, compr(u0v, jj), gi) : gi;
        }
        bst4(RX, vxs | rowdrop, rz, go[0], go[1], go[2], go[3]);
      }
      if (T::born || T::adj) {
        xab[0] = xab[1]; xbb[0] = xbb[1]; xcb[0] = xcb[1]; xxb[0] = xxb[1];
      }
#pragma unroll
      for (int d = 0; d < PD; ++d) {
        kb[d] = kb[d + 1]; pb[d] = pb[d + 1]; u0b[d] = u0b[d + 1]; hvb[d] = hvb[d + 1];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Frame update (hybrid ABC) as a row march.  The frame is cut into four
// regions: top rows [0, n2) and bottom rows [nz-n2, nz) over all columns,
// left columns [0, n2) and right columns [nx-n2, nx) over the rows between.
// A wave owns 64 consecutive columns of a region (lanes 1..62 write; lanes 0
// and 63 only supply lateral neighbours) and a run of its rows.  Marching
// down, iteration t computes on all 64 columns the pre-blend two-way value T
// of row t -- the value the reference's Hybrid1 reads from the un-blended
// DFW2: Add / BKAdd on the frame with the source, the data replacement, the
// Born source or the adjoint residual -- and then the one-way value and the
// blend of row t-1 (Hybrid1/Hybrid2, kernel.cu:116-183), which read T of rows
// t-2, t-1 and t: the inner neighbour and its laterals sit one row or one
// column away.  Vertical taps come from a register queue of u1 rows,
// horizontal taps from a per-wave LDS row; the reference's outer mirror
// (kernel.cu:65-68) is applied to the row and column indices of the loads.
//
// The row body has no branch (selects; accesses that must not happen get an
// out-of-range buffer offset), so the memory-counter waits stay exact: the
// coefficient row of row t+1 is gathered during row t (its offset arrived a
// row earlier), row operands arrive PD rows ahead and the one-way operands two
// rows ahead, and each row waits only on loads issued a row or more before.
// No block-level barrier: the four waves of a block are independent.
//
// SIDE (forward and receiver): a record of the side bands, whose written cells
// are all side cells of Hybrid1/Hybrid2 (kernel.cu:126-137), the corner rows'
// innermost ones aside.  Their inner neighbour is one column away in a
// direction that is the lane's own, so two cross-lane reads a row replace ten,
// and the ring and blend weight of a lane are its own.  The side bands are bound
// by instruction issue and by the L1: 128 shots of 351 x 1701 took 44 us a step
// (half-length 3), 36 with this body and the lateral factors of Model::fs (a
// side cell's velocity lies in another row for every lane).
template <int NFD, int MODE, bool SIDE>
__device__ __forceinline__ void frame_body(const FrameArgs& a, const int4 rec) {
  constexpr int PD = 2;                   // rows of prefetch
  constexpr int NB = NFD > 2 ? NFD : 2;   // queue rows kept behind the T row
  // The row loop is unrolled by U, a multiple of 12 that holds the u1 rows
  // t-NB .. t+NFD+PD; every other per-row buffer is circular with a length
  // dividing 12 (2, 3 or 6), so no buffer is ever copied, only renamed.
  constexpr int U = (NB + NFD + 1 + PD + 11) / 12 * 12;
  // LDS row: halo | 64 columns | halo | dump slot; a packed side record
  // (band 4) uses halo | 32 columns | halo | halo | 32 columns | halo | dump
  constexpr int WN = 64 + 4 * NFD + 1;
  __shared__ float win[4][WN];
  const Grid& g = a.g;
  const Model& m = a.m;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int z0 = rec.x, cx0 = rec.y, band = rec.z & 15, nrows = (rec.z >> 4) & 0xffff, shot = rec.w;
  const int ncol = (rec.z >> 20) & 0xff;  // top/bottom: written lanes 1..ncol (0: 1..62)
  const ShotGeo sg = a.geo[shot];
  const int NX = sg.nx, NZ = g.nz, N2 = g.n2;
  // Band 4 packs both side bands of a row run into one wave (n2 <= 30):
  // lanes 0..31 hold columns -1..30 (the left band and its inner
  // neighbour), lanes 32..63 columns nx-31..nx; lanes 1..30 and 33..62
  // write.  The +-1 lane shuffles of the one-way update stay inside a half.
  const bool packed = (SIDE || MODE == FR_BORN || MODE == FR_ADJ) && band == 4;
  const bool rhalf = packed && lane >= 32;
  const int x = packed ? (rhalf ? NX - 63 + lane : lane - 1) : cx0 + lane;
  const int xm = mirror_idx(x, NX);
  int ccl = 0, ccr = NX;  // output columns of the region
  if (band == 2) ccr = N2;
  else if (band == 3) ccl = NX - N2;
  else if (packed) { ccl = rhalf ? NX - N2 : 0; ccr = rhalf ? NX : N2; }
  const int hl_ = packed ? (lane & 31) : lane;  // lane within its (half) run
  const bool outcol = hl_ >= 1 && hl_ <= (packed ? 30 : (ncol ? ncol : 62)) && x >= ccl && x < ccr;
  // LDS slot of the lane's column (packed: the right half after the left
  // half's right halo and its own left halo)
  const int slot = packed && rhalf ? 3 * NFD + lane : NFD + lane;
  // A top or bottom run whose written columns all lie in [n2+1, nx-n2-2]
  // holds only cells of the top (bottom) edges: no corner cell, no side cell
  // (the ring of (z, x) is z, resp. nz-1-z).  Those waves take a shorter
  // one-way update; the choice is uniform per wave.
  const bool pure_tb = band < 2 && cx0 + 1 >= N2 + 1 && cx0 + 62 <= NX - N2 - 2;

  const long long so = (long long)shot * g.fstride;
  const unsigned fb = (unsigned)g.fstride * 4u;
  const Rsrc R1 = rsrc(a.u1 + so, fb), R0 = rsrc(a.u0 + so, fb), R2 = rsrc(a.u2 + so, fb);
  const long long mo = (long long)sg.win * m.mstride;
  const Rsrc RP = rsrc(m.pm + mo, fb), RK = rsrc(m.ko + mo, fb);
  const Rsrc RV = rsrc(m.v + mo, fb), RR = rsrc(m.r1 + mo, fb), RQ = rsrc(m.fs + sg.fw * g.fstride, fb);
  const Rsrc RC = rsrc(m.ctab, (unsigned)(m.nrow * m.cs) * 4u);
  const Rsrc RW = rsrc(m.w, (unsigned)(N2 + 1) * 4u);
  const unsigned P4 = (unsigned)g.pitch * 4u;
  auto rowm = [=](int z) __attribute__((always_inline)) -> unsigned { return (unsigned)mirror_idx(z, NZ) * P4; };
  auto colb = [&](int c) __attribute__((always_inline)) -> unsigned { return (unsigned)(g.x0 + c) * 4u; };
  const unsigned vcol = colb(xm), vst = outcol ? vcol : kDrop;

  // halo columns of the LDS row: lanes 0..NFD-1 the left ones, NFD..2NFD-1
  // the right ones (packed: the left half's two halos, then lanes
  // 2NFD..4NFD-1 the right half's); the other lanes fetch nothing and write
  // the dump slot
  unsigned vhal = kDrop;
  int hpos = WN - 1;
  if (!packed) {
    if (lane < NFD) { vhal = colb(mirror_idx(cx0 - NFD + lane, NX)); hpos = lane; }
    else if (lane < 2 * NFD) { vhal = colb(mirror_idx(cx0 + 64 + lane - NFD, NX)); hpos = 64 + lane; }
  } else {
    if (lane < NFD) { vhal = colb(mirror_idx(-1 - NFD + lane, NX)); hpos = lane; }
    else if (lane < 2 * NFD) { vhal = colb(mirror_idx(31 + lane - NFD, NX)); hpos = 32 + lane; }
    else if (lane < 3 * NFD) { vhal = colb(mirror_idx(NX - 31 - 3 * NFD + lane, NX)); hpos = 32 + lane; }
    else if (lane < 4 * NFD) { vhal = colb(mirror_idx(NX + 1 - 3 * NFD + lane, NX)); hpos = 64 + lane; }
  }

  // receivers on row s_z (kernel.cu:349): this step's data sample of the lane's
  // trace (receiver field: sample k+1; adjoint: sample k), dropped elsewhere
  Rcv rr = a.r;
  rr.s_l = sg.s_l;
  rr.s_r = sg.s_r;
  int rs = 0;
  const bool isrcv = (MODE == FR_RCV || MODE == FR_ADJ) && is_receiver(x, rr, &rs);
  float ev = 0.f;
  if (MODE == FR_RCV || MODE == FR_ADJ) {
    const int kd = MODE == FR_RCV ? a.k + 1 : a.k;
    const Rsrc RD = rsrc(a.data + ((long long)shot * a.nt + kd) * a.r.n, (unsigned)a.r.n * 4u);
    ev = bld1(RD, isrcv ? (unsigned)rs * 4u : kDrop, 0u);
  }
  // strip slot of this step (FP32) or its FP32 staging (FP16 / BF16)
  Rsrc RS;
  if (MODE == FR_FWD) {
    const long long ss = a.st.ss;
    const float* sb = a.st.fmt == 0
        ? (const float*)a.st.base + ((long long)shot * a.st.nslot + a.k % a.st.nslot) * ss
        : a.st.stage + ((long long)shot * 2 + (a.k & 1)) * ss;
    RS = rsrc(sb, a.save_strips ? (unsigned)ss * 4u : 0u);
  }
  // strip element of (z, x) (strip_elem): the lane's part, and the row's in the loop
  unsigned vstrip = kDrop;
  if (MODE == FR_FWD) {
    if (SIDE) {
      if (x >= N2 - g.nfd && x < N2) vstrip = (unsigned)(N2 - 1 - x) * 4u;
      else if (x >= NX - N2 && x < NX - N2 + g.nfd) vstrip = (unsigned)(g.mnz * g.nfd + x - (NX - N2)) * 4u;
    } else if (x >= N2 && x < NX - N2) {
      vstrip = (unsigned)(2 * g.mnz * g.nfd + x - N2) * 4u;
    }
    if (!outcol) vstrip = kDrop;
  }
  const int sd = g.nfd, smnx = sg.mnx;
  auto strip_put_row = [=](int z, unsigned drop, float val) __attribute__((always_inline)) {
    const bool up = z >= N2 - sd && z < N2, dn = z >= NZ - N2 && z < NZ - N2 + sd;
    const int e = SIDE ? (z - N2) * sd : (up ? (N2 - 1 - z) * smnx : (sd + z - (NZ - N2)) * smnx);
    const bool on = SIDE ? z >= N2 && z < NZ - N2 : up || dn;
    bst1s(RS, (vstrip + (on ? (unsigned)e * 4u : 0u)) | drop | (on ? 0u : kDrop), 0u, val);
  };
  // adjoint with per-cell rows: the interior cells of the march (the rows and
  // columns next to the frame, whose pre-blend values the one-way update
  // reads) take the transposed stencil of the interior kernel
  const bool adjt = MODE == FR_ADJ && a.adjt != 0;
  Rsrc RTP;
  if (MODE == FR_ADJ) RTP = rsrc(m.tp + (long long)sg.win * m.tpstride, adjt ? (unsigned)(4 * NFD) * fb : 0u);
  Rsrc RBX, RBA, RBB, RBC;
  if (MODE == FR_BORN) {
    RBX = rsrc(m.refl + (long long)shot * m.rstride, fb);
    RBA = rsrc(a.ua + so, fb); RBB = rsrc(a.ub + so, fb); RBC = rsrc(a.uc + so, fb);
  }
  constexpr int NE = MODE == FR_BORN ? 4 : 1;  // extra operands of a T row

  // one-way operands of row zr (velocity, r1, lateral factor, blend weight; SIDE:
  // the weight is the lane's, r1 that of the corner rows)
  auto abc_ops = [&](int zr, float& vp, float& r1v, float& sqv, float& wv_) __attribute__((always_inline)) {
    vp = bld1(RV, vcol, rowm(zr));
    sqv = bld1(RQ, vcol, rowm(zr));
    if (!SIDE) {
      const int ar = min(min(zr, x), min(NZ - 1 - zr, NX - 1 - x));
      r1v = bld1(RR, vcol, rowm(zr));
      wv_ = bld1(RW, (unsigned)min(max(N2 - ar, 0), N2) * 4u, 0u);
    }
  };
  // extra operands of T row zr: the Born source terms
  auto t_ops = [&](int zr, float* e) __attribute__((always_inline)) {
    if (MODE == FR_BORN) {
      const unsigned rz = rowm(zr);
      e[0] = bld1(RBX, vcol, rz); e[1] = bld1(RBA, vcol, rz);
      e[2] = bld1(RBB, vcol, rz); e[3] = bld1(RBC, vcol, rz);
    } else {
      e[0] = 0.f;
    }
  };
  float r1top = 0.f, r1bot = 0.f, wside = 0.f;
  const bool inr = x < N2;  // SIDE: inner neighbour to the right
  const bool clane = x == N2 - 1 || x == NX - N2;
  const int inl = (inr ? lane + 1 : lane - 1) * 4;
  if (SIDE) {
    r1top = bld1(RR, vcol, rowm(N2));
    r1bot = bld1(RR, vcol, rowm(NZ - N2 - 1));
    wside = bld1(RW, (unsigned)min(max(N2 - min(x, NX - 1 - x), 0), N2) * 4u, 0u);
  }
  float TS[3] = {0.f, 0.f, 0.f};  // SIDE: T rows it-2 .. it at the inner neighbour
  float US[2] = {0.f, 0.f};       // SIDE: u1 rows it-1, it there

  // Circular buffers, indexed by the iteration number it (T row t0 + it):
  //   q[U]     u1 rows (row t0 - NB + i in slot i % U)
  //   kob[6]   coefficient offsets of T rows it-1 .. it+KD (KD = 4 rows ahead:
  //            the coefficient row of it+1 is gathered from them one row early)
  //   pmb, halb [3]: P and halo of T rows it .. it+PD
  //   u0b[6]   u0 rows it-2 .. it+PD; cr[2] coefficient rows of it, it+1
  //   abc [3]  one-way operands of rows it-1 .. it+1; ext[2] T-row extras
  //   T[3]     T rows it-2 .. it
  const int t0 = z0 - 1;          // T row of the first iteration
  const int niter = nrows + 2;    // T rows z0-1 .. z0+nrows
  float q[U];
#pragma unroll
  for (int s = 0; s < NB + NFD + PD; ++s) q[s] = bld1(R1, vcol, rowm(t0 - NB + s));
  constexpr int KD = 4;
  unsigned kob[6];
#pragma unroll
  for (int d = 0; d < KD; ++d) kob[d] = bld1u(RK, vcol, rowm(t0 + d));
  float pmb[3], halb[3], u0b[6];
#pragma unroll
  for (int d = 0; d < PD; ++d) {
    pmb[d] = bld1(RP, vcol, rowm(t0 + d));
    halb[d] = bld1(R1, vhal, rowm(t0 + d));
    u0b[2 + d] = bld1s(R0, vcol, rowm(t0 + d));   // slot (it + 2) % 6 holds row t0 + it
  }
  u0b[0] = bld1s(R0, vcol, rowm(t0 - 2));
  u0b[1] = bld1s(R0, vcol, rowm(t0 - 1));
  CoefRow<NFD> cr[2];
  cr[0].load(RC, kob[0]);
  float ext[2][NE];
  t_ops(t0, ext[0]);
  float T[3] = {0.f, 0.f, 0.f};
  float vpb[3] = {0.f, 0.f, 0.f}, r1b[3] = {0.f, 0.f, 0.f}, vqb[3] = {0.f, 0.f, 0.f},
        wb[3] = {0.f, 0.f, 0.f};   // slot (it + 1) % 3 holds row t0 + it

  for (int base = 0; base < niter; base += U) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int it = base + j;   // base is a multiple of U, so it % L == j % L for L | 12
      if (it >= niter) break;
      const int tt = t0 + it;
      // (1) coefficient row of T row tt+1 (its offset arrived a row ago)
      cr[(j + 1) % 2].load(RC, kob[(j + 1) % 6]);
      // (2) operands of later rows
      kob[(j + KD) % 6] = bld1u(RK, vcol, rowm(tt + KD));
      q[(j + NB + NFD + PD) % U] = bld1(R1, vcol, rowm(tt + NFD + PD));
      pmb[(j + PD) % 3] = bld1(RP, vcol, rowm(tt + PD));
      halb[(j + PD) % 3] = bld1(R1, vhal, rowm(tt + PD));
      u0b[(j + 2 + PD) % 6] = bld1s(R0, vcol, rowm(tt + PD));
      abc_ops(tt + 1, vpb[(j + 2) % 3], r1b[(j + 2) % 3], vqb[(j + 2) % 3], wb[(j + 2) % 3]);
      t_ops(tt + 1, ext[(j + 1) % 2]);
      __builtin_amdgcn_sched_barrier(0);
      // (3) horizontal neighbours of row tt through LDS
      const float u = q[(j + NB) % U];
      win[wv][slot] = u;
      win[wv][hpos] = halb[j % 3];
      wave_lds_sync();
      float hl[NFD], hr[NFD];
#pragma unroll
      for (int l = 1; l <= NFD; ++l) {
        hl[l - 1] = win[wv][slot - l];
        hr[l - 1] = win[wv][slot + l];
      }
      wave_lds_sync();
      // (4) pre-blend two-way value T of (tt, x) (Add / BKAdd, kernel.cu:46-80, 339-380)
      const CoefRow<NFD>& crc = cr[j % 2];
      float w1 = (float)(crc.c0d(m.h1) * (double)u);
#pragma unroll
      for (int l = 1; l <= NFD; ++l) {
        float s = q[(j + NB - l + U) % U] + q[(j + NB + l) % U];
        s = __builtin_fmaf(s, m.hzx2_1, hl[l - 1]);
        s = s + hr[l - 1];
        w1 = __builtin_fmaf(crc.c(l), s, w1);
      }
      if (MODE == FR_ADJ) {  // (L^T mu) on interior cells, each tap with the neighbour's row
        const bool inner = tt >= N2 && tt < NZ - N2 && x >= N2 && x < NX - N2;
        float w1t = (float)(crc.c0d(m.h1) * (double)u);
#pragma unroll
        for (int l = 1; l <= NFD; ++l) {
          const unsigned rz = rowm(tt);
          const float cu = bld1(RTP, vcol, rz + (unsigned)(4 * (l - 1)) * fb);
          const float cd = bld1(RTP, vcol, rz + (unsigned)(4 * (l - 1) + 1) * fb);
          const float cl = bld1(RTP, vcol, rz + (unsigned)(4 * (l - 1) + 2) * fb);
          const float cr2 = bld1(RTP, vcol, rz + (unsigned)(4 * (l - 1) + 3) * fb);
          const float vs = __builtin_fmaf(cu, q[(j + NB - l + U) % U], cd * q[(j + NB + l) % U]);
          float sv = __builtin_fmaf(vs, m.hzx2_1, cl * hl[l - 1]);
          sv = __builtin_fmaf(cr2, hr[l - 1], sv);
          w1t = w1t + sv;
        }
        w1 = (adjt && inner) ? w1t : w1;
      }
      const float u0 = u0b[(j + 2) % 6], pmv = pmb[j % 3];
      const float* ex = ext[j % 2];
      float Tn;
      if (MODE == FR_FWD) {
        Tn = combine_p(u, u0, pmv, w1, a.f64comb != 0);
        Tn = (tt == sg.r_u && x == sg.r_x) ? Tn + a.wav : Tn;
      } else if (MODE == FR_BORN) {  // scattered field: m * D2u on the interior, no source
        Tn = combine_p(u, u0, pmv, w1, a.f64comb != 0);
        const float d2u = (ex[1] - 2.0f * ex[2]) + ex[3];
        const bool inner = tt >= N2 && tt < NZ - N2 && x >= N2 && x < NX - N2;
        Tn = inner ? __builtin_fmaf(ex[0], d2u, Tn) : Tn;
      } else if (MODE == FR_ADJ) {   // adjoint field: P * r(k) added at the receivers
        Tn = combine_p(u, u0, pmv, w1, false);
        Tn = (isrcv && tt == a.r.s_z) ? Tn + pmv * ev : Tn;
      } else {                       // receiver field: data replace where non-zero
        Tn = combine_p(u, u0, pmv, w1, false);
        Tn = (tt == a.r.s_z && ev != 0.0f) ? ev : Tn;  // 0 without a receiver
      }
      T[j % 3] = Tn;
      // (5) one-way value and blend of row z = tt - 1 (written from the third row on)
      if (SIDE) {  // left edge (inner column x+1) or right edge (x-1) (kernel.cu:126-129,134-137)
        const int z = tt - 1;
        TS[j % 3] = __int_as_float(__builtin_amdgcn_ds_bpermute(inl, __float_as_int(Tn)));
        const float Ti = TS[(j + 2) % 3], Tip = TS[j % 3], Tim = TS[(j + 1) % 3];
        const float U0z = u0b[(j + 1) % 6], U0p = u0b[(j + 2) % 6], U0m = u0b[j % 6];
        const float U0i = __int_as_float(__builtin_amdgcn_ds_bpermute(inl, __float_as_int(U0z)));
        const float U1z = q[(j + NB - 1) % U], U1i = US[(j + 1) % 2];
        US[j % 2] = inr ? hr[0] : hl[0];
        const int ab = j % 3;
        const float tv = m.taoh * vpb[ab];
        const float t1 = tv * ((Ti - U0i) + U0z);
        const float t2 = ((((-2.0f * U1z) + U0z) + Ti) - 2.0f * U1i) + U0i;
        const float lap = ((((Tip - 2.0f * Ti) + Tim) + U0p) - 2.0f * U0z) + U0m;
        const float t3 = vqb[ab] * lap;
        // the corner cells of the first and last row (kernel.cu:138-155)
        const bool corner = clane && (z == N2 || z == NZ - N2 - 1);
        const float r1v = z == N2 ? r1top : r1bot;
        const float num_c = U1z + r1v * (Ti + (z == N2 ? T[j % 3] : T[(j + 1) % 3]));
        const float den = corner ? 2.0f * r1v + 1.0f : tv + 1.0f;
        const float O = (1.0f / den) * (corner ? num_c : (t1 - t2) + t3);
        const float val = (1.0f - wside) * T[(j + 2) % 3] + wside * O;
        const unsigned rd = it >= 2 && z < z0 + nrows ? 0u : kDrop;
        bst1s(R2, vst | rd, rowm(z), val);
        if (MODE == FR_FWD) strip_put_row(z, rd, val);  // Hybrid3 (kernel.cu:184-208)
      } else if (pure_tb) {  // top edge (inner row z+1) or bottom edge (inner row z-1) (kernel.cu:122-125,130-133)
        const int z = tt - 1;
        const bool tp = band == 0;
        const float T0 = T[(j + 2) % 3];
        const float Tin = tp ? T[j % 3] : T[(j + 1) % 3];
        const float U1z = q[(j + NB - 1) % U];
        const float U1i = tp ? q[(j + NB) % U] : q[(j + NB - 2) % U];
        const float U0z = u0b[(j + 1) % 6];
        const float U0i = tp ? u0b[(j + 2) % 6] : u0b[j % 6];
        const float Til = __shfl_up(Tin, 1), Tir = __shfl_down(Tin, 1);
        const float U0l = __shfl_up(U0z, 1), U0r = __shfl_down(U0z, 1);
        const int ab = j % 3;
        const float vp = vpb[ab], wgt = wb[ab];
        const float tv = m.taoh * vp;
        const float t1 = tv * ((Tin - U0i) + U0z);
        const float t2 = ((((-2.0f * U1z) + U0z) + Tin) - 2.0f * U1i) + U0i;
        const float lap = ((((Tir - 2.0f * Tin) + Til) + U0r) - 2.0f * U0z) + U0l;
        const float t3 = vqb[ab] * lap;
        const float O = (1.0f / (tv + 1.0f)) * ((t1 - t2) + t3);
        const float val = (1.0f - wgt) * T0 + wgt * O;
        const unsigned rd = it >= 2 && z < z0 + nrows ? 0u : kDrop;
        bst1s(R2, vst | rd, rowm(z), val);
        if (MODE == FR_FWD) strip_put_row(z, rd, val);  // Hybrid3 (kernel.cu:184-208)
      } else {
        const int z = tt - 1;
        const float Tm = T[(j + 1) % 3], T0 = T[(j + 2) % 3], Tp = T[j % 3];
        const float U1m = q[(j + NB - 2) % U], U1z = q[(j + NB - 1) % U], U1p = q[(j + NB) % U];
        const float U0m = u0b[j % 6], U0z = u0b[(j + 1) % 6], U0p = u0b[(j + 2) % 6];
        const float T0l = __shfl_up(T0, 1), T0r = __shfl_down(T0, 1);
        const float Tml = __shfl_up(Tm, 1), Tmr = __shfl_down(Tm, 1);
        const float Tpl = __shfl_up(Tp, 1), Tpr = __shfl_down(Tp, 1);
        const float U0l = __shfl_up(U0z, 1), U0r = __shfl_down(U0z, 1);
        const float U1l = __shfl_up(U1z, 1), U1r = __shfl_down(U1z, 1);
        const int ar = min(min(z, x), min(NZ - 1 - z, NX - 1 - x));  // ring
        const int br = NZ - 1 - ar, crr = NX - 1 - ar;
        const bool zc = (z - ar <= 1) || (br - z <= 1);
        const bool xc = (x - ar <= 1) || (crr - x <= 1);
        const bool corner = zc && xc;
        const bool top = z == ar, bot = !top && z == br, side = !top && !bot;
        const bool inr = x == ar;  // side cell with its inner neighbour to the right
        const int ab = j % 3;      // one-way operands of row z
        const float vp = vpb[ab], r1v = r1b[ab], wgt = wb[ab];
        // corner cells (kernel.cu:138-155)
        const float Tx = (x - ar <= 1) ? T0r : T0l;
        const float Tz = (z - ar <= 1) ? Tp : Tm;
        const float num_c = U1z + r1v * (Tx + Tz);
        const float den_c = 2.0f * r1v + 1.0f;
        // one-way update of the edges (kernel.cu:122-137)
        const float Ti = top ? Tp : (bot ? Tm : (inr ? T0r : T0l));
        const float Tip = top ? Tpr : (bot ? Tmr : (inr ? Tpr : Tpl));
        const float Tim = top ? Tpl : (bot ? Tml : (inr ? Tmr : Tml));
        const float U0i = top ? U0p : (bot ? U0m : (inr ? U0r : U0l));
        const float U0pp = side ? U0p : U0r, U0pm = side ? U0m : U0l;
        const float U1i = top ? U1p : (bot ? U1m : (inr ? U1r : U1l));
        const float tv = m.taoh * vp;
        const float t1 = tv * ((Ti - U0i) + U0z);
        const float t2 = ((((-2.0f * U1z) + U0z) + Ti) - 2.0f * U1i) + U0i;
        const float lap = ((((Tip - 2.0f * Ti) + Tim) + U0pp) - 2.0f * U0z) + U0pm;
        const float t3 = vqb[ab] * lap;
        const float num_s = (t1 - t2) + t3;
        const float den_s = tv + 1.0f;
        const float O = (1.0f / (corner ? den_c : den_s)) * (corner ? num_c : num_s);
        const float val = (1.0f - wgt) * T0 + wgt * O;
        const unsigned rd = it >= 2 && z < z0 + nrows ? 0u : kDrop;
        bst1s(R2, vst | rd, rowm(z), val);
        if (MODE == FR_FWD) strip_put_row(z, rd, val);  // Hybrid3 (kernel.cu:184-208)
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Top and bottom bands away from the corners, four columns per lane.  A record
// (z0, cs, band | rows << 4, shot) covers the 256 columns cs .. cs+255 (cs ==
// n2 mod 4, so each lane's float4 is aligned like the interior kernel's) and
// writes the columns cs+4 .. cs+251 left of frame4_end.  Every written cell is a
// top-edge (bottom-edge) cell of Hybrid1/Hybrid2 (kernel.cu:122-125, 130-133):
// its one-way update reads the inner row and the lateral neighbours x-1, x+1
// of the same row, so lanes 0 and 63 only supply neighbours, and a lane writes
// all of its float4 or nothing.  The row march, the look-ahead of the operands and the
// arithmetic are those of frame_body's top/bottom path, operation for
// operation, so both give the same bits; per cell this one spends a quarter of
// the row addressing, masks and buffer instructions.  FR_FWD and FR_RCV only.
template <int NFD, int MODE, bool BOT>
__device__ __forceinline__ void frame_tb4_body(const FrameArgs& a, const int4 rec) {
  static_assert(MODE == FR_FWD || MODE == FR_RCV, "forward and receiver frames only");
  constexpr int PD = 2;                   // rows of prefetch
  constexpr int NB = NFD > 2 ? NFD : 2;   // queue rows kept behind the T row
  constexpr int U = (NB + NFD + 1 + PD + 11) / 12 * 12;
  constexpr int H = (NFD + 3) & ~3;
  constexpr int W4 = 64 + 2 * (H / 4);
  constexpr int NWIN = 1 + 2 * (H / 4);
  __shared__ float4 lds[4][W4];
  const Grid& g = a.g;
  const Model& m = a.m;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int z0 = rec.x, cs = rec.y, nrows = (rec.z >> 4) & 0xffff, shot = rec.w;
  const ShotGeo sg = a.geo[shot];
  const int NX = sg.nx, NZ = g.nz, N2 = g.n2;
  const int wend = frame4_end(N2, NX);
  const int c0 = cs + 4 * lane;
  const int clast = NX - ((NX - N2) & 3);  // largest c == n2 (mod 4) with c <= nx
  const unsigned vcol = (unsigned)(g.x0 + min(c0, clast)) * 4u;
  const bool out = lane >= 1 && lane <= 62 && c0 < wend;
  const unsigned vst = out ? (unsigned)(g.x0 + c0) * 4u : kDrop;
  // halo float4s of the LDS row: lanes 0 .. H/4-1 left, H/4 .. 2H/4-1 right
  // (columns past the shot's width only feed unwritten columns)
  unsigned vhal = kDrop;
  int hpos = H / 4 + lane;
  if (lane < H / 4) { vhal = (unsigned)(g.x0 + cs - H + 4 * lane) * 4u; hpos = lane; }
  else if (lane < 2 * (H / 4)) {
    vhal = (unsigned)(g.x0 + min(cs + 256 + 4 * (lane - H / 4), clast)) * 4u;
    hpos = 64 + lane;
  }

  const long long so = (long long)shot * g.fstride;
  const unsigned fb = (unsigned)g.fstride * 4u;
  const Rsrc R1 = rsrc(a.u1 + so, fb), R0 = rsrc(a.u0 + so, fb), R2 = rsrc(a.u2 + so, fb);
  const long long mo = (long long)sg.win * m.mstride;
  const Rsrc RP = rsrc(m.pm + mo, fb), RK = rsrc(m.ko + mo, fb), RV = rsrc(m.v + mo, fb);
  const Rsrc RQ = rsrc(m.fs + sg.fw * g.fstride, fb);
  const Rsrc RC = rsrc(m.ctab, (unsigned)(m.nrow * m.cs) * 4u);
  const Rsrc RW = rsrc(m.w, (unsigned)(N2 + 1) * 4u);
  const unsigned P4 = (unsigned)g.pitch * 4u;
  auto rowm = [&](int z) -> unsigned { return (unsigned)mirror_idx(z, NZ) * P4; };
  // ring of row zr: zr (top edge), nz-1-zr (bottom edge)
  auto ring = [&](int zr) -> int { return BOT ? NZ - 1 - zr : zr; };

  // receiver field: this step's data sample (k+1) of each receiver column,
  // replacing the field on row s_z where non-zero (kernel.cu:349-354)
  // (a column without a receiver reads 0: its dropped load returns 0)
  float ev[4] = {0.f, 0.f, 0.f, 0.f};
  if (MODE == FR_RCV) {
    Rcv rr = a.r;
    rr.s_l = sg.s_l;
    rr.s_r = sg.s_r;
    const Rsrc RD = rsrc(a.data + ((long long)shot * a.nt + a.k + 1) * a.r.n, (unsigned)a.r.n * 4u);
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      int rs = 0;
      const bool isr = is_receiver(c0 + jj, rr, &rs);
      ev[jj] = bld1(RD, isr ? (unsigned)rs * 4u : kDrop, 0u);
    }
  }
  // strip slot of this step (FP32) or its FP32 staging (FP16 / BF16): the
  // rows n2-nfd .. n2-1 (top) and nz-n2 .. nz-n2+nfd-1 (bottom), Hybrid3
  // (kernel.cu:184-208), element 2a + (n2-1-z)*mnx + x-n2, resp.
  // 2a + b + (z-(nz-n2))*mnx + x-n2, as strip_elem
  Rsrc RS;
  if (MODE == FR_FWD) {
    const long long ss = a.st.ss;
    const float* sb = a.st.fmt == 0
        ? (const float*)a.st.base + ((long long)shot * a.st.nslot + a.k % a.st.nslot) * ss
        : a.st.stage + ((long long)shot * 2 + (a.k & 1)) * ss;
    RS = rsrc(sb, a.save_strips ? (unsigned)ss * 4u : 0u);
  }
  const int sa = g.mnz * g.nfd, sbb = g.nfd * sg.mnx;

  const int t0 = z0 - 1;          // T row of the first iteration
  const int niter = nrows + 2;    // T rows z0-1 .. z0+nrows
  float4 q[U];
#pragma unroll
  for (int s = 0; s < NB + NFD + PD; ++s) q[s] = bld4(R1, vcol, rowm(t0 - NB + s));
  uint4 kb[3];
  float4 pmb[3], halb[3], u0b[6];
#pragma unroll
  for (int d = 0; d < PD; ++d) {
    kb[d] = bld4u(RK, vcol, rowm(t0 + d));
    pmb[d] = bld4(RP, vcol, rowm(t0 + d));
    halb[d] = bld4(R1, vhal, rowm(t0 + d));
    u0b[2 + d] = bld4s(R0, vcol, rowm(t0 + d));   // slot (it + 2) % 6 holds row t0 + it
  }
  u0b[0] = bld4s(R0, vcol, rowm(t0 - 2));
  u0b[1] = bld4s(R0, vcol, rowm(t0 - 1));
  CoefRow<NFD> cr[2][4];  // coefficient rows of T rows it, it+1 (slot it % 2)
  cr[0][0].load(RC, kb[0].x);
  cr[0][1].load(RC, kb[0].y);
  cr[0][2].load(RC, kb[0].z);
  cr[0][3].load(RC, kb[0].w);
  const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 T[3] = {z4, z4, z4};
  float4 vpb[3] = {z4, z4, z4}, sqb[3] = {z4, z4, z4};  // slot (it + 1) % 3 holds row t0 + it
  float wb[3] = {0.f, 0.f, 0.f};

  for (int base = 0; base < niter; base += U) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int it = base + j;   // base is a multiple of U, so it % L == j % L for L | 12
      if (it >= niter) break;
      const int tt = t0 + it;
      // (1) coefficient rows of T row tt+1 (their offsets arrived a row ago)
      {
        const uint4 kn = kb[(j + 1) % 3];
        cr[(j + 1) % 2][0].load(RC, kn.x);
        cr[(j + 1) % 2][1].load(RC, kn.y);
        cr[(j + 1) % 2][2].load(RC, kn.z);
        cr[(j + 1) % 2][3].load(RC, kn.w);
      }
      // (2) operands of later rows
      q[(j + NB + NFD + PD) % U] = bld4(R1, vcol, rowm(tt + NFD + PD));
      kb[(j + PD) % 3] = bld4u(RK, vcol, rowm(tt + PD));
      pmb[(j + PD) % 3] = bld4(RP, vcol, rowm(tt + PD));
      halb[(j + PD) % 3] = bld4(R1, vhal, rowm(tt + PD));
      u0b[(j + 2 + PD) % 6] = bld4s(R0, vcol, rowm(tt + PD));
      // one-way operands of row tt+1: velocity, on the bottom edge the lateral
      // factor (on the top edge the velocity's own), the blend weight of its ring
      vpb[(j + 2) % 3] = bld4(RV, vcol, rowm(tt + 1));
      if (BOT) sqb[(j + 2) % 3] = bld4(RQ, vcol, rowm(tt + 1));
      wb[(j + 2) % 3] = bld1(RW, (unsigned)min(max(N2 - ring(tt + 1), 0), N2) * 4u, 0u);
      __builtin_amdgcn_sched_barrier(0);
      // (3) horizontal neighbours of row tt through LDS
      const float4 qc = q[(j + NB) % U];
      lds[wv][hpos] = halb[j % 3];
      lds[wv][H / 4 + lane] = qc;
      wave_lds_sync();
      float4 win[NWIN];
#pragma unroll
      for (int t = 0; t < NWIN; ++t) win[t] = lds[wv][lane + t];
      wave_lds_sync();
      // (4) pre-blend two-way values T of row tt (Add / BKAdd, kernel.cu:46-80, 339-380)
      const float4 u0v = u0b[(j + 2) % 6], pv = pmb[j % 3];
      float tn[4];
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const CoefRow<NFD>& crc = cr[j % 2][jj];
        const float u = compr(qc, jj);
        float w1 = (float)(crc.c0d(m.h1) * (double)u);
#pragma unroll
        for (int l = 1; l <= NFD; ++l) {
          float s = compr(q[(j + NB - l + U) % U], jj) + compr(q[(j + NB + l) % U], jj);
          s = __builtin_fmaf(s, m.hzx2_1, compr(win[(H + jj - l) >> 2], (H + jj - l) & 3));
          s = s + compr(win[(H + jj + l) >> 2], (H + jj + l) & 3);
          w1 = __builtin_fmaf(crc.c(l), s, w1);
        }
        float Tn;
        if (MODE == FR_FWD) {
          Tn = combine_p(u, compr(u0v, jj), compr(pv, jj), w1, a.f64comb != 0);
          Tn = (tt == sg.r_u && c0 + jj == sg.r_x) ? Tn + a.wav : Tn;
        } else {
          Tn = combine_p(u, compr(u0v, jj), compr(pv, jj), w1, false);
          Tn = (tt == a.r.s_z && ev[jj] != 0.0f) ? ev[jj] : Tn;
        }
        tn[jj] = Tn;
      }
      T[j % 3] = make_float4(tn[0], tn[1], tn[2], tn[3]);
      // (5) one-way value and blend of row z = tt - 1 (written from the third row on)
      const int z = tt - 1;
      const float4 T0v = T[(j + 2) % 3];
      const float4 Tinv = BOT ? T[(j + 1) % 3] : T[j % 3];
      const float4 U1zv = q[(j + NB - 1) % U];
      const float4 U1iv = BOT ? q[(j + NB - 2) % U] : q[(j + NB) % U];
      const float4 U0zv = u0b[(j + 1) % 6];
      const float4 U0iv = BOT ? u0b[j % 6] : u0b[(j + 2) % 6];
      // lateral neighbours across lanes: x-1 of component 0, x+1 of component 3
      const float Tl = __shfl_up(Tinv.w, 1), Tr = __shfl_down(Tinv.x, 1);
      const float Ul = __shfl_up(U0zv.w, 1), Ur = __shfl_down(U0zv.x, 1);
      const int ab = j % 3;
      const float4 vpv = vpb[ab];
      const float4 sqv = sqb[ab];
      const float wgt = wb[ab];
      float val[4];
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const float T0 = compr(T0v, jj), Tin = compr(Tinv, jj);
        const float U1z = compr(U1zv, jj), U1i = compr(U1iv, jj);
        const float U0z = compr(U0zv, jj), U0i = compr(U0iv, jj);
        const float Til = jj == 0 ? Tl : compr(Tinv, jj - 1);
        const float Tir = jj == 3 ? Tr : compr(Tinv, jj + 1);
        const float U0l = jj == 0 ? Ul : compr(U0zv, jj - 1);
        const float U0r = jj == 3 ? Ur : compr(U0zv, jj + 1);
        const float vp = compr(vpv, jj);
        const float tv = m.taoh * vp;
        const float t1 = tv * ((Tin - U0i) + U0z);
        const float t2 = ((((-2.0f * U1z) + U0z) + Tin) - 2.0f * U1i) + U0i;
        const float lap = ((((Tir - 2.0f * Tin) + Til) + U0r) - 2.0f * U0z) + U0l;
        const float t3 = (BOT ? compr(sqv, jj) : (m.taoh2 * vp) * vp) * lap;
        const float O = (1.0f / (tv + 1.0f)) * ((t1 - t2) + t3);
        val[jj] = (1.0f - wgt) * T0 + wgt * O;
      }
      const bool rowout = it >= 2 && z < z0 + nrows;
      const unsigned rz = rowm(z);
      bst4s(R2, vst | (rowout ? 0u : kDrop), rz, val[0], val[1], val[2], val[3]);
      if (MODE == FR_FWD) {  // Hybrid3 (kernel.cu:184-208)
        const bool srow = BOT ? (z >= NZ - N2 && z < NZ - N2 + g.nfd) : (z >= N2 - g.nfd && z < N2);
        if (rowout && srow) {
          const int sbase = BOT ? 2 * sa + sbb + (z - (NZ - N2)) * sg.mnx - N2
                                : 2 * sa + (N2 - 1 - z) * sg.mnx - N2;
          bst4s(RS, out ? (unsigned)(sbase + c0) * 4u : kDrop, 0u, val[0], val[1], val[2], val[3]);
        }
      }
    }
  }
}

template <int NFD, int EPI>
__global__ __launch_bounds__(256) void k_interior(const IntArgs a) {
  interior_body<NFD, EPI>(a, blockIdx.x);
}

// One wave per float4 top/bottom record (frame_tb4_body).
template <int NFD, int MODE>
__global__ __launch_bounds__(256) void k_frame4(const FrameArgs a) {
  const int ri = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (ri >= a.nrec) return;
  const int4 rec = a.recs[ri];
  if ((rec.z & 15) == 0) frame_tb4_body<NFD, MODE, false>(a, rec);
  else frame_tb4_body<NFD, MODE, true>(a, rec);
}

// Receiver and adjoint frame launches may carry the strip restore of the
// reconstructed field (FrameArgs::rf): its blocks follow the record blocks and
// fill the wave slots the frame's few long waves leave free.
template <int NFD, int MODE>
__device__ __forceinline__ void frame_records_body(const FrameArgs& a, const unsigned bid) {
  if ((MODE == FR_RCV || MODE == FR_ADJ) && a.rbps > 0) {
    const unsigned nfb = ((unsigned)a.nrec + 3u) >> 2;
    if (bid >= nfb) {
      const unsigned b = bid - nfb, per = (unsigned)(a.rbps * a.nshot);
      const bool second = b >= per;  // of two fields
      strip_restore_body(a.g, second ? a.rf[1] : a.rf[0], a.st, a.geo, second ? a.rk[1] : a.rk[0],
                         second ? b - per : b, (unsigned)a.rbps);
      return;
    }
  }
  const int ri = (int)bid * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (ri >= a.nrec) return;
  const int4 rec = a.recs[ri];
  if ((MODE == FR_FWD || MODE == FR_RCV) && (rec.z & 15) >= 2) frame_body<NFD, MODE, true>(a, rec);
  else frame_body<NFD, MODE, false>(a, rec);
}

template <int NFD, int MODE>
__global__ __launch_bounds__(256) void k_frame(const FrameArgs a) {
  frame_records_body<NFD, MODE>(a, blockIdx.x);
}

#if RTM_NFD <= 5  // TWO_MAX_NFD
// The same cells for batches whose blocks of four shots share a model window
// (k_two's): the four waves of a block march the band of four shots row by row
// together, and the window's coefficient planes, P and the three one-way
// operands (TwoArgs::cp, Model::fs) go through LDS, each plane loaded by one
// wave.  Seven
// buffer instructions a row instead of eleven and no division; 155 registers
// instead of 217 at half-length 3, three waves per SIMD.
template <int NFD, int MODE, bool BOT>
__device__ __forceinline__ void frame_quad_body(const FrameArgs& a, const int z0, const int nrows,
                                                const int cs, const int s4,
                                                float4 (*cf)[NFD + 5][64], float4 (*lds)[64 + 2 * ((NFD + 3) / 4)],
                                                float4* dat) {
  static_assert(MODE == FR_FWD || MODE == FR_RCV, "forward and receiver frames only");
  constexpr int PD = 2;                   // rows of prefetch
  constexpr int NB = NFD > 2 ? NFD : 2;   // queue rows kept behind the T row
  constexpr int U = (NB + NFD + 1 + PD + 11) / 12 * 12;
  constexpr int H = (NFD + 3) & ~3;
  constexpr int NWIN = 1 + 2 * (H / 4);
  constexpr int NPL = NFD + 5, NL = (NPL + 3) / 4;
  const Grid& g = a.g;
  const Model& m = a.m;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool live = s4 + wv < a.nshot;  // a wave past the batch only loads planes
  const int shot = live ? s4 + wv : a.nshot - 1;
  const ShotGeo sg = a.geo[shot];
  const int NX = sg.nx, NZ = g.nz, N2 = g.n2;
  const int wend = frame4_end(N2, NX);
  if (cs + 4 >= wend) return;  // the same for the block's shots
  const int c0 = cs + 4 * lane;
  const int clast = NX - ((NX - N2) & 3);  // largest c == n2 (mod 4) with c <= nx
  const unsigned vcol = (unsigned)(g.x0 + min(c0, clast)) * 4u;
  const bool out = live && lane >= 1 && lane <= 62 && c0 < wend;
  const unsigned vst = out ? (unsigned)(g.x0 + c0) * 4u : kDrop;
  unsigned vhal = kDrop;
  int hpos = H / 4 + lane;
  if (lane < H / 4) { vhal = (unsigned)(g.x0 + cs - H + 4 * lane) * 4u; hpos = lane; }
  else if (lane < 2 * (H / 4)) {
    vhal = (unsigned)(g.x0 + min(cs + 256 + 4 * (lane - H / 4), clast)) * 4u;
    hpos = 64 + lane;
  }

  const long long so = (long long)shot * g.fstride;
  const unsigned fb = (unsigned)g.fstride * 4u;
  const Rsrc R1 = rsrc(a.u1 + so, fb), R0 = rsrc(a.u0 + so, fb), R2 = rsrc(a.u2 + so, fb);
  const Rsrc RW = rsrc(m.w, (unsigned)(N2 + 1) * 4u);
  // the wave's planes: wv, wv + 4, ..; the one-way operands lag a row
  const float* cp = a.cp + (long long)sg.win * a.cpstride;
  Rsrc RPL[NL];
  int lag[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int pl = wv + 4 * i;
    const float* p = pl < NPL - 1 ? cp + pl * g.fstride : m.fs + sg.fw * g.fstride;
    RPL[i] = rsrc(p, pl < NPL ? fb : 0u);
    lag[i] = pl >= NFD + 2 ? 1 : 0;
  }
  const unsigned P4 = (unsigned)g.pitch * 4u;
  auto rowm = [=](int z) -> unsigned { return (unsigned)mirror_idx(z, NZ) * P4; };

  if (MODE == FR_RCV) {  // this step's data samples, as in frame_tb4_body
    float ev[4];
    Rcv rr = a.r;
    rr.s_l = sg.s_l;
    rr.s_r = sg.s_r;
    const Rsrc RD = rsrc(a.data + ((long long)shot * a.nt + a.k + 1) * a.r.n, (unsigned)a.r.n * 4u);
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      int rs = 0;
      const bool isr = is_receiver(c0 + jj, rr, &rs);
      ev[jj] = bld1(RD, isr ? (unsigned)rs * 4u : kDrop, 0u);
    }
    dat[threadIdx.x] = make_float4(ev[0], ev[1], ev[2], ev[3]);
  }
  Rsrc RS;  // strip rows, as in frame_tb4_body
  if (MODE == FR_FWD) {
    const long long ss = a.st.ss;
    const float* sb = a.st.fmt == 0
        ? (const float*)a.st.base + ((long long)shot * a.st.nslot + a.k % a.st.nslot) * ss
        : a.st.stage + ((long long)shot * 2 + (a.k & 1)) * ss;
    RS = rsrc(sb, a.save_strips ? (unsigned)ss * 4u : 0u);
  }
  const int sa = g.mnz * g.nfd, sbb = g.nfd * sg.mnx;
  const float hzx2_1 = m.hzx2_1;
  const double h1 = m.h1;
  const int srow = MODE == FR_FWD ? sg.r_u : a.r.s_z;
  const bool f64comb = MODE == FR_FWD && a.f64comb != 0;

  const int t0 = z0 - 1;          // T row of the first iteration
  const int niter = nrows + 2;    // T rows z0-1 .. z0+nrows
  float4 q[U];
  float4 pl[NL];                  // planes of iteration it + 1
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const float4 p0 = bld4(RPL[i], vcol, rowm(t0 - lag[i]));
    pl[i] = bld4(RPL[i], vcol, rowm(t0 + 1 - lag[i]));
    if (wv + 4 * i < NPL) cf[0][wv + 4 * i][lane] = p0;
  }
#pragma unroll
  for (int s = 0; s < NB + NFD + PD; ++s) q[s] = bld4(R1, vcol, rowm(t0 - NB + s));
  float4 halb[3], u0b[6];
#pragma unroll
  for (int d = 0; d < PD; ++d) {
    halb[d] = bld4(R1, vhal, rowm(t0 + d));
    u0b[2 + d] = bld4s(R0, vcol, rowm(t0 + d));   // slot (it + 2) % 6 holds row t0 + it
  }
  u0b[0] = bld4s(R0, vcol, rowm(t0 - 2));
  u0b[1] = bld4s(R0, vcol, rowm(t0 - 1));
  const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 T[3] = {z4, z4, z4};
  // blend weight of row t0 + lane (QUAD_MAX_ROWS keeps a run's rows in the lanes)
  const int ringl = BOT ? NZ - 1 - (t0 + lane) : t0 + lane;
  const int wlane = __float_as_int(bld1(RW, (unsigned)min(max(N2 - ringl, 0), N2) * 4u, 0u));
  block_lds_sync();

  for (int base = 0; base < niter; base += U) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int it = base + j;   // base is a multiple of U, so it % L == j % L for L | 12
      if (it >= niter) break;    // the same for the whole block
      const int tt = t0 + it;
      // planes of the next row to LDS, of the row after it from memory
#pragma unroll
      for (int i = 0; i < NL; ++i)
        if (wv + 4 * i < NPL) cf[(j + 1) & 1][wv + 4 * i][lane] = pl[i];
#pragma unroll
      for (int i = 0; i < NL; ++i) pl[i] = bld4(RPL[i], vcol, rowm(tt + 2 - lag[i]));
      q[(j + NB + NFD + PD) % U] = bld4(R1, vcol, rowm(tt + NFD + PD));
      halb[(j + PD) % 3] = bld4(R1, vhal, rowm(tt + PD));
      u0b[(j + 2 + PD) % 6] = bld4s(R0, vcol, rowm(tt + PD));
      __builtin_amdgcn_sched_barrier(0);
      // horizontal neighbours of row tt through LDS
      const float4 qc = q[(j + NB) % U];
      lds[wv][hpos] = halb[j % 3];
      lds[wv][H / 4 + lane] = qc;
      wave_lds_sync();
      float4 win[NWIN];
#pragma unroll
      for (int t = 0; t < NWIN; ++t) win[t] = lds[wv][lane + t];
      wave_lds_sync();
      // pre-blend two-way values T of row tt (Add / BKAdd, kernel.cu:46-80, 339-380)
      const float4 (*cr)[64] = cf[j & 1];
      const float4 u0v = u0b[(j + 2) % 6], k0 = cr[0][lane], pv = cr[NFD + 1][lane];
      float w1[4], tn[4];
#pragma unroll
      for (int jj = 0; jj < 4; ++jj)
        w1[jj] = (float)((h1 * (double)compr(k0, jj)) * (double)compr(qc, jj));
#pragma unroll
      for (int l = 1; l <= NFD; ++l) {
        const float4 kl = cr[l][lane];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          float s = compr(q[(j + NB - l + U) % U], jj) + compr(q[(j + NB + l) % U], jj);
          s = __builtin_fmaf(s, hzx2_1, compr(win[(H + jj - l) >> 2], (H + jj - l) & 3));
          s = s + compr(win[(H + jj + l) >> 2], (H + jj + l) & 3);
          w1[jj] = __builtin_fmaf(compr(kl, jj), s, w1[jj]);
        }
      }
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        float Tn = combine_p(compr(qc, jj), compr(u0v, jj), compr(pv, jj), w1[jj], f64comb);
        if (MODE == FR_FWD) Tn = (tt == srow && c0 + jj == sg.r_x) ? Tn + a.wav : Tn;
        tn[jj] = Tn;
      }
      if (MODE == FR_RCV && tt == srow) {
        const float4 ev = dat[threadIdx.x];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) tn[jj] = compr(ev, jj) != 0.0f ? compr(ev, jj) : tn[jj];
      }
      T[j % 3] = make_float4(tn[0], tn[1], tn[2], tn[3]);
      __builtin_amdgcn_sched_barrier(0);
      // one-way value and blend of row z = tt - 1 (written from the third row on)
      const int z = tt - 1;
      const float4 T0v = T[(j + 2) % 3];
      const float4 Tinv = BOT ? T[(j + 1) % 3] : T[j % 3];
      const float4 U1zv = q[(j + NB - 1) % U];
      const float4 U1iv = BOT ? q[(j + NB - 2) % U] : q[(j + NB) % U];
      const float4 U0zv = u0b[(j + 1) % 6];
      const float4 U0iv = BOT ? u0b[j % 6] : u0b[(j + 2) % 6];
      const float Tl = __shfl_up(Tinv.w, 1), Tr = __shfl_down(Tinv.x, 1);
      const float Ul = __shfl_up(U0zv.w, 1), Ur = __shfl_down(U0zv.x, 1);
      const float wgt = __int_as_float(__builtin_amdgcn_readlane(wlane, max(it - 1, 0)));
      const float4 tvv = cr[NFD + 2][lane], div = cr[NFD + 3][lane], sqv = cr[NFD + 4][lane];
      float val[4];
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const float T0 = compr(T0v, jj), Tin = compr(Tinv, jj);
        const float U1z = compr(U1zv, jj), U1i = compr(U1iv, jj);
        const float U0z = compr(U0zv, jj), U0i = compr(U0iv, jj);
        const float Til = jj == 0 ? Tl : compr(Tinv, jj - 1);
        const float Tir = jj == 3 ? Tr : compr(Tinv, jj + 1);
        const float U0l = jj == 0 ? Ul : compr(U0zv, jj - 1);
        const float U0r = jj == 3 ? Ur : compr(U0zv, jj + 1);
        const float t1 = compr(tvv, jj) * ((Tin - U0i) + U0z);
        const float t2 = ((((-2.0f * U1z) + U0z) + Tin) - 2.0f * U1i) + U0i;
        const float lap = ((((Tir - 2.0f * Tin) + Til) + U0r) - 2.0f * U0z) + U0l;
        const float t3 = compr(sqv, jj) * lap;
        const float O = compr(div, jj) * ((t1 - t2) + t3);
        val[jj] = (1.0f - wgt) * T0 + wgt * O;
      }
      const bool rowout = it >= 2 && z < z0 + nrows;
      const unsigned rz = rowm(z);
      bst4s(R2, vst | (rowout ? 0u : kDrop), rz, val[0], val[1], val[2], val[3]);
      if (MODE == FR_FWD) {  // Hybrid3 (kernel.cu:184-208)
        const bool strow = BOT ? (z >= NZ - N2 && z < NZ - N2 + g.nfd) : (z >= N2 - g.nfd && z < N2);
        if (rowout && strow) {
          const int sbase = BOT ? 2 * sa + sbb + (z - (NZ - N2)) * sg.mnx - N2
                                : 2 * sa + (N2 - 1 - z) * sg.mnx - N2;
          bst4s(RS, out ? (unsigned)(sbase + c0) * 4u : kDrop, 0u, val[0], val[1], val[2], val[3]);
        }
      }
      block_lds_sync();
    }
  }
}

// The whole frame of a forward or receiver step of such a batch in one launch:
// the blocks of frame_quad_body, shot group fastest, then those of k_frame.
// Against one launch of k_frame on every cell or, for large batches, one each of
// k_frame and k_frame4 (whichever the autotuner had chosen), half-length 3, us a
// step: 128 shots of 351 x 1701 forward 112 -> 77, receiver field (half of the
// launches with the restore of two strip sets) 106 -> 86; 32 shots 50 -> 28; 16
// shots 24 -> 21.  Counters of 128 shots: 0.34 GB a step, 140 MB of it results
// and their operands, at 4 TB/s: halo rows of the runs, and side bands that take
// a part of every line they touch.
template <int NFD, int MODE>
__global__ __launch_bounds__(256, NFD <= 3 ? 3 : 2) void k_frame_quad(const FrameArgs a) {
  __shared__ float4 cf[2][NFD + 5][64];
  __shared__ float4 lds[4][64 + 2 * ((NFD + 3) / 4)];
  __shared__ float4 dat[MODE == FR_RCV ? 256 : 1];
  unsigned b = blockIdx.x;
  if (b < (unsigned)a.nquad) {
    const unsigned nsg = ((unsigned)a.nshot + 3u) >> 2;
    const int s4 = (int)(b % nsg) * 4;
    const unsigned t = b / nsg;
    const int w = (int)(t % (unsigned)a.qwin), r = (int)(t / (unsigned)a.qwin);
    const int zr = (r >> 1) * a.qrows, rows = min(a.qrows, a.g.n2 - zr), cs = a.g.n2 + 248 * w;
    if (r & 1) frame_quad_body<NFD, MODE, true>(a, a.g.nz - a.g.n2 + zr, rows, cs, s4, cf, lds, dat);
    else frame_quad_body<NFD, MODE, false>(a, zr, rows, cs, s4, cf, lds, dat);
    return;
  }
  frame_records_body<NFD, MODE>(a, b - (unsigned)a.nquad);
}
#endif

// One time step's interior and frame work in one launch.  The two write
// disjoint cells of u(k+1) and only read u(k), u(k-1) and the model, so they
// may run concurrently; the interior kernel waits on memory most of the time
// and the frame kernel on instruction issue, so frame blocks placed among the
// interior blocks fill the interior's idle issue slots.  Blocks go in units
// of 8 (one per XCD): every R-th unit is a frame unit while frame units last,
// so an interior block keeps its own index modulo 8 (its XCD, which its L2
// sharing of model rows relies on); indices past a part's block count exit.
template <int NFD, int EPI, int MODE>
__global__ __launch_bounds__(256) void k_step(const IntArgs ia, const FrameArgs fa, unsigned nint,
                                              unsigned nfr) {
  const unsigned nfu = (nfr + 7u) >> 3, niu = (nint + 7u) >> 3;
  const unsigned R = (nfu + niu) / nfu;
  const unsigned u = blockIdx.x >> 3, s8 = blockIdx.x & 7u;
  const unsigned before = min(nfu, (u + R - 1u) / R);  // frame units ahead of unit u
  if (u % R == 0u && u / R < nfu) {
    const unsigned b = (u / R) * 8u + s8;
    if (b < nfr) frame_records_body<NFD, MODE>(fa, b);
  } else {
    const unsigned b = (u - before) * 8u + s8;
    if (b < nint) interior_body<NFD, EPI>(ia, b);
  }
}

// ---------------------------------------------------------------------------
// launches of this half-length
template <>
hipError_t StencilOps<RTM_NFD>::interior(int epi, dim3 grid, const IntArgs& a, hipStream_t s) {
  constexpr int N = RTM_NFD;
  const dim3 block(256);
  if (epi == EPI_FWD) hipLaunchKernelGGL((k_interior<N, EPI_FWD>), grid, block, 0, s, a);
  else if (epi == EPI_FWD64) hipLaunchKernelGGL((k_interior<N, EPI_FWD64>), grid, block, 0, s, a);
  else if (epi == EPI_SRC) hipLaunchKernelGGL((k_interior<N, EPI_SRC>), grid, block, 0, s, a);
  else if (epi == EPI_BORN) hipLaunchKernelGGL((k_interior<N, EPI_BORN>), grid, block, 0, s, a);
  else if (epi == EPI_BORN64) hipLaunchKernelGGL((k_interior<N, EPI_BORN64>), grid, block, 0, s, a);
  else if (epi == EPI_ADJ) hipLaunchKernelGGL((k_interior<N, EPI_ADJ>), grid, block, 0, s, a);
  else if (epi == EPI_ADJT) hipLaunchKernelGGL((k_interior<N, EPI_ADJT>), grid, block, 0, s, a);
  else if (epi == EPI_RCV0) hipLaunchKernelGGL((k_interior<N, EPI_RCV0>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((k_interior<N, EPI_RCV>), grid, block, 0, s, a);
  return hipGetLastError();
}

template <>
hipError_t StencilOps<RTM_NFD>::frame(int mode, dim3 grid, const FrameArgs& a, hipStream_t s) {
  constexpr int N = RTM_NFD;
  const dim3 block(256);
  if (mode == FR_FWD) hipLaunchKernelGGL((k_frame<N, FR_FWD>), grid, block, 0, s, a);
  else if (mode == FR_BORN) hipLaunchKernelGGL((k_frame<N, FR_BORN>), grid, block, 0, s, a);
  else if (mode == FR_ADJ) hipLaunchKernelGGL((k_frame<N, FR_ADJ>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((k_frame<N, FR_RCV>), grid, block, 0, s, a);
  return hipGetLastError();
}

template <>
hipError_t StencilOps<RTM_NFD>::frame4(int mode, dim3 grid, const FrameArgs& a, hipStream_t s) {
#if RTM_NFD <= 6
  constexpr int N = RTM_NFD;
  const dim3 block(256);
  if (mode == FR_FWD) hipLaunchKernelGGL((k_frame4<N, FR_FWD>), grid, block, 0, s, a);
  else if (mode == FR_RCV) hipLaunchKernelGGL((k_frame4<N, FR_RCV>), grid, block, 0, s, a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
#else
  return hipErrorInvalidValue;
#endif
}

template <>
hipError_t StencilOps<RTM_NFD>::frame_quad(int mode, dim3 grid, const FrameArgs& a, hipStream_t s) {
#if RTM_NFD <= 5
  constexpr int N = RTM_NFD;
  const dim3 block(256);
  if (mode == FR_FWD) hipLaunchKernelGGL((k_frame_quad<N, FR_FWD>), grid, block, 0, s, a);
  else if (mode == FR_RCV) hipLaunchKernelGGL((k_frame_quad<N, FR_RCV>), grid, block, 0, s, a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
#else
  return hipErrorInvalidValue;
#endif
}

template <>
hipError_t StencilOps<RTM_NFD>::step(int epi, dim3 grid, const IntArgs& ia, const FrameArgs& fa,
                                     unsigned nint, unsigned nfr, hipStream_t s) {
  constexpr int N = RTM_NFD;
  const dim3 block(256);
  if (epi == EPI_FWD)
    hipLaunchKernelGGL((k_step<N, EPI_FWD, FR_FWD>), grid, block, 0, s, ia, fa, nint, nfr);
  else if (epi == EPI_RCV0)
    hipLaunchKernelGGL((k_step<N, EPI_RCV0, FR_RCV>), grid, block, 0, s, ia, fa, nint, nfr);
  else
    hipLaunchKernelGGL((k_step<N, EPI_RCV, FR_RCV>), grid, block, 0, s, ia, fa, nint, nfr);
  return hipGetLastError();
}

}  // namespace rtm
