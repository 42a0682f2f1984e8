// rtm_tile.hip -- a whole time step in one launch, one cell per thread: the
// kernels of small batches, compiled once per stencil half-length
// (-DRTM_NFD=1..12).
//
// The marching kernels (rtm_stencil.hip) give a wave a long run of rows, which
// is what bandwidth wants, and need a batch that fills the GPU with such runs:
// on a 240 x 440 grid a step pair took five launches of 8 to 19 us each, nearly
// all of it the latency of a row times 20 to 30 rows.  Here a block takes a
// tile of 64 x 8 CPT cells of one shot, all its loads are in flight at once, and
// a step is two dependent memory accesses deep (coefficient offset, then
// coefficient row).  Interior and frame share the launch: the frame's one-way
// update reads the pre-blend values T of neighbouring cells of u(k+1), which a
// tile that touches the frame recomputes on a ring of one cell around itself.
//
//   TILE_FWD   Add + Hybrid1/2/3 (kernel.cu:46-208), strips, receiver records
//   TILE_MIG   BKAdd_EFF on the interior and BKEqual on the strip rings of
//              u(k) (222-320); BKAdd, data replacement and BKHybrid1/2 of the
//              receiver field (339-487); Rel_* of up to three steps (489-517)
//   TILE_BORN  TILE_FWD and the scattered field with its records
//   TILE_ADJ   the reconstruction of u(k), the adjoint field and its gradient
//
// Every value is computed by the operations of the marching kernels in their
// order, so both give the same bits.  The fields written in a step (u2, q2)
// are read by no thread of the same launch.
#include <hip/hip_runtime.h>

#include "rtm_device.h"

namespace rtm {

// Loads at a byte offset from a base the whole block shares (a scalar base and
// a 32-bit vector offset).  An access that must not happen reads offset 0
// instead and is not used: the block's scalar instructions are what a launch
// of many tiles is short of, and a buffer resource per array costs twice those
// of a base.
__device__ __forceinline__ float ldg(const float* base, unsigned byte_off) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + byte_off);
}
__device__ __forceinline__ void stg(float* base, unsigned byte_off, float v) {
  *reinterpret_cast<float*>(reinterpret_cast<char*>(base) + byte_off) = v;
}

template <int NFD, int PASS, int CPT>
__global__ __launch_bounds__(512) void k_tile(const TileArgs a) {
  constexpr bool FWD = PASS == TILE_FWD || PASS == TILE_BORN;  // u on the whole grid
  constexpr bool MIG = PASS == TILE_MIG, BORN = PASS == TILE_BORN, ADJ = PASS == TILE_ADJ;
  constexpr bool TWO = PASS != TILE_FWD;                       // q on the whole grid
  constexpr int NT = 512, TH = 8 * CPT;
  constexpr int R = tile_halo(NFD), LW = 64 + 2 * R, LH = TH + 2 * R, NL = (LH * LW + NT - 1) / NT;
  constexpr int RW = 66, RH = TH + 2, NR = (RH * RW + NT - 1) / NT;  // cells with a T value
  __shared__ float su1[LH * LW], sq1[TWO ? LH * LW : 1];
  __shared__ float tu[FWD ? RH * RW : 1], tu0[FWD ? RH * RW : 1];
  __shared__ float tq[TWO ? RH * RW : 1], tq0[TWO ? RH * RW : 1];

  const Grid& g = a.g;
  const Model& m = a.m;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int shot = (int)blockIdx.x;  // fastest: an XCD holds shots of the same tile
  const ShotGeo sg = a.geo[shot];
  const int NX = sg.nx, NZ = g.nz, N2 = g.n2;
  const int x0 = (int)blockIdx.y * 64, z0 = (int)blockIdx.z * TH;
  if (x0 >= NX) return;  // a narrower shot of a ragged batch
  const int zw = z0 + wv * CPT, x = x0 + lane;  // the thread's cells: rows zw .. zw+CPT-1
  const auto is_inner = [&](int zz, int xx) {
    return zz >= N2 && zz < NZ - N2 && xx >= N2 && xx < NX - N2;
  };
  // uniform: tiles with frame cells, tiles with interior cells
  const bool edge = tile_edge(z0, x0, TH, NFD, N2, NZ, NX);
  const bool has_inner = z0 + TH > N2 && z0 < NZ - N2 && x0 + 64 > N2 && x0 < NX - N2;

  const long long so = (long long)shot * g.fstride, mo = (long long)sg.win * m.mstride;
  const float *u1 = a.u1 + so, *pu = a.u0 + so, *q1 = a.q1 + so, *pq = a.q0 + so;
  const float *mp = m.pm + mo, *mk = reinterpret_cast<const float*>(m.ko) + mo;
  const unsigned P4 = (unsigned)g.pitch * 4u;
  const auto at = [&](int zz, int xx) { return (unsigned)zz * P4 + (unsigned)(g.x0 + xx) * 4u; };
  unsigned own[CPT];  // cells past the grid read its last row and column
  bool cell[CPT], inner[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    cell[j] = zw + j < NZ && x < NX;
    own[j] = at(min(zw + j, NZ - 1), min(x, NX - 1));
    inner[j] = is_inner(zw + j, x);
  }

  // ---- loads: coefficient offsets first, the coefficient rows wait on them
  const bool need_u = FWD || has_inner;  // the reconstruction has no frame cells
  unsigned ko[CPT] = {}, kr[NR];
  unsigned ro[NR];  // T cells of a tile with frame cells: the tile and a ring of one cell
  int rz[NR], rx[NR];
  if (edge) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int e = tid + i * NT, r = e / RW;
      rz[i] = z0 - 1 + r;
      rx[i] = x0 - 1 + e - r * RW;
      ro[i] = at(min(max(rz[i], 0), NZ - 1), min(max(rx[i], 0), NX - 1));
      kr[i] = __float_as_uint(ldg(mk, ro[i]));
    }
  }
  if (!edge || MIG || ADJ) {
#pragma unroll
    for (int j = 0; j < CPT; ++j) ko[j] = __float_as_uint(ldg(mk, own[j]));
  }
  float lu[NL], lq[TWO ? NL : 1];
  if (edge) {  // the outer mirror (kernel.cu:65-68)
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = tid + i * NT, r = e / LW;
      const unsigned o = at(mirror_idx(z0 - R + r, NZ), mirror_idx(x0 - R + e - r * LW, NX));
      lu[i] = need_u ? ldg(u1, o) : 0.f;
      if (TWO) lq[i] = ldg(q1, o);
    }
  } else {  // every access inside the grid
    const int r = tid / LW;
    int c = tid - r * LW;
    unsigned o = at(z0 - R + r, x0 - R + c);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const unsigned oo = tid + i * NT < LH * LW ? o : 0u;
      lu[i] = ldg(u1, oo);
      if (TWO) lq[i] = ldg(q1, oo);
      c += NT % LW;
      o += (unsigned)(NT / LW) * P4 + (unsigned)(NT % LW) * 4u;
      if (c >= LW) { c -= LW; o += P4 - (unsigned)LW * 4u; }
    }
  }
  float pm[CPT], u0[CPT] = {}, q0[CPT] = {};
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    pm[j] = ldg(mp, own[j]);
    if (need_u) u0[j] = ldg(pu, own[j]);
    if (TWO) q0[j] = ldg(pq, own[j]);
  }
  float prm[NR], pu0[NR], pq0[NR];
  if (edge) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      prm[i] = ldg(mp, ro[i]);
      if (FWD) pu0[i] = ldg(pu, ro[i]);
      if (TWO) pq0[i] = ldg(pq, ro[i]);
    }
  }
  // imaging: sums and images of the own cells; the adjoint's gradient
  float si1[CPT] = {}, si2[CPT] = {}, ssu[CPT] = {}, ssq[CPT] = {};
  float *i1 = a.i1 + so, *i2 = a.i2 + so, *su = a.su + so, *sq = a.sq + so;
  if ((MIG && a.nimg > 0) || ADJ) {
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      si1[j] = ldg(i1, own[j]);
      if (MIG) {
        si2[j] = ldg(i2, own[j]);
        if (a.icompen) {
          ssu[j] = ldg(su, own[j]);
          ssq[j] = ldg(sq, own[j]);
        }
      }
    }
  }

  // receivers on row s_z: data of step k+1 replaces the receiver field
  // (kernel.cu:349-354), residuals of step k add to the adjoint field
  Rcv rr = a.r;
  rr.s_l = sg.s_l;
  rr.s_r = sg.s_r;
  const float* data = a.data + ((long long)shot * a.nt + (MIG ? a.k + 1 : a.k)) * rr.n;
  const auto data_at = [&](int zz, int xx, float* d) {
    int s = 0;
    if (zz != rr.s_z || !is_receiver(xx, rr, &s)) return false;
    *d = ldg(data, (unsigned)s * 4u);
    return true;
  };
  // what else the values of a cell need: its data sample or residual, or (Born)
  // its reflectivity; of the own cells, or of a frame tile's T cells
  constexpr int NX2 = NR > CPT ? NR : CPT;
  float ext[NX2] = {};
  bool isr[NX2] = {};
  if (MIG || ADJ || BORN) {
#pragma unroll
    for (int i = 0; i < NX2; ++i) {
      const float* refl = m.refl + (long long)shot * m.rstride;
      if (edge && i < NR) {
        if (BORN) ext[i] = ldg(refl, ro[i]);
        else isr[i] = data_at(rz[i], rx[i], &ext[i]);
      } else if (!edge && i < CPT) {
        if (BORN) ext[i] = ldg(refl, own[i]);
        else isr[i] = data_at(zw + i, x, &ext[i]);
      }
    }
  }
  // one-way operands of the frame cells (kernel.cu:116-183) and their strips
  float vp[CPT] = {}, fsv[CPT] = {}, r1v[CPT] = {}, wgt[CPT] = {}, ring[CPT] = {};
  int se[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    se[j] = -1;
    if (!edge || !cell[j] || inner[j]) continue;
    const int z = zw + j, ar = min(min(z, x), min(NZ - 1 - z, NX - 1 - x));
    vp[j] = ldg(m.v + mo, own[j]);
    fsv[j] = ldg(m.fs + sg.fw * g.fstride, own[j]);
    r1v[j] = ldg(m.r1 + mo, own[j]);
    wgt[j] = m.w[min(max(N2 - ar, 0), N2)];
    se[j] = strip_elem(g, NX, sg.mnx, z, x);
    if ((MIG || ADJ) && se[j] >= 0) ring[j] = strip_get(a.st, shot, a.k, se[j]);
  }

  CoefRow<NFD> cw[CPT], crr[NR];
  if (!edge || MIG || ADJ) {
#pragma unroll
    for (int j = 0; j < CPT; ++j) cw[j].load(m.ctab, ko[j]);
  }
  if (edge) {
#pragma unroll
    for (int i = 0; i < NR; ++i) crr[i].load(m.ctab, kr[i]);
  }
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int e = tid + i * NT;
    if (e < LH * LW) {
      su1[e] = lu[i];
      if (TWO) sq1[e] = lq[i];
    }
  }
  __syncthreads();

  // tap sum of the cell at LDS position c (Add / BKAdd, kernel.cu:46-80,
  // 339-380); v(l), l = -NFD .. NFD: its column
  const auto taps = [&](const float* s, int c, const CoefRow<NFD>& cf, auto v) {
    float w1 = (float)(cf.c0d(m.h1) * (double)v(0));
#pragma unroll
    for (int l = 1; l <= NFD; ++l) {
      float t = v(-l) + v(l);
      t = __builtin_fmaf(t, m.hzx2_1, s[c - l]);
      t = t + s[c + l];
      w1 = __builtin_fmaf(cf.c(l), t, w1);
    }
    return w1;
  };
  // the transposed stencil (per-cell rows): each tap with the coefficient of
  // the cell it reads, from the neighbour-tap planes
  const auto taps_t = [&](const float* s, int c, const CoefRow<NFD>& cf, unsigned o, auto v) {
    const float* tp = m.tp + (long long)sg.win * m.tpstride;
    const unsigned fb = (unsigned)g.fstride * 4u;
    float w1 = (float)(cf.c0d(m.h1) * (double)v(0));
#pragma unroll
    for (int l = 1; l <= NFD; ++l) {
      const unsigned p = o + (unsigned)(4 * (l - 1)) * fb;
      const float cu = ldg(tp, p), cd = ldg(tp, p + fb);
      const float cl = ldg(tp, p + 2u * fb), cr = ldg(tp, p + 3u * fb);
      const float vs = __builtin_fmaf(cu, v(-l), cd * v(l));
      float t = __builtin_fmaf(vs, m.hzx2_1, cl * s[c - l]);
      t = __builtin_fmaf(cr, s[c + l], t);
      w1 = w1 + t;
    }
    return w1;
  };
  // pre-blend values of cell (zz, xx): u of the forward field, q of the
  // second; vu, vq: the columns of the two fields
  const auto values = [&](int zz, int xx, int c, const CoefRow<NFD>& cf, float p, float c_u0,
                          float c_q0, unsigned o, float ex, bool rcv, auto vu, auto vq, float* Tu,
                          float* Tq) {
    const bool in = is_inner(zz, xx);
    if (FWD) {
      *Tu = combine_p(vu(0), c_u0, p, taps(su1, c, cf, vu), a.f64comb != 0);
      *Tu = (zz == sg.r_u && xx == sg.r_x) ? *Tu + a.wav : *Tu;
    }
    if (BORN) {  // scattering source m * D2u(k) on the interior, where u(k) = Tu
      float t = combine_p(vq(0), c_q0, p, taps(sq1, c, cf, vq), a.f64comb != 0);
      const float d2u = (*Tu - 2.0f * vu(0)) + c_u0;
      *Tq = in ? __builtin_fmaf(ex, d2u, t) : t;
    }
    if (MIG) {
      const float t = combine_p(vq(0), c_q0, p, taps(sq1, c, cf, vq), false);
      *Tq = (rcv && ex != 0.0f) ? ex : t;
    }
    if (ADJ) {
      float w1;
      if (a.adjt != 0 && in) w1 = taps_t(sq1, c, cf, o, vq);
      else w1 = taps(sq1, c, cf, vq);
      const float t = combine_p(vq(0), c_q0, p, w1, false);
      *Tq = rcv ? t + p * ex : t;
    }
  };
  const int lc0 = (wv * CPT + R) * LW + lane + R, rc0 = (wv * CPT + 1) * RW + lane + 1;
  float nu[CPT] = {}, nq[CPT] = {};  // new values of the own cells
  if (edge) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int e = tid + i * NT;
      if (e < RH * RW) {
        const int c = (rz[i] - z0 + R) * LW + rx[i] - x0 + R;
        float Tu = 0.f, Tq = 0.f;
        if (rz[i] >= 0 && rz[i] < NZ && rx[i] >= 0 && rx[i] < NX)
          values(rz[i], rx[i], c, crr[i], prm[i], pu0[i], pq0[i], ro[i], ext[i], isr[i],
                 [&](int l) { return su1[c + l * LW]; },
                 [&](int l) { return TWO ? sq1[c + l * LW] : 0.f; }, &Tu, &Tq);
        if (FWD) { tu[e] = Tu; tu0[e] = pu0[i]; }
        if (TWO) { tq[e] = Tq; tq0[e] = pq0[i]; }
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      const int z = zw + j, rc = rc0 + j * RW, lc = lc0 + j * LW;
      if (!cell[j]) continue;
      if (inner[j]) {
        if (FWD) nu[j] = tu[rc];
        if (TWO) nq[j] = tq[rc];
        continue;
      }
      // one-way value and blend (Hybrid1/Hybrid2, kernel.cu:116-183)
      const int ar = min(min(z, x), min(NZ - 1 - z, NX - 1 - x));  // ring
      const bool topc = z == ar, botc = !topc && z == NZ - 1 - ar, side = !topc && !botc;
      const bool inr = x == ar;  // side cell with its inner neighbour to the right
      const int br = NZ - 1 - ar, crn = NX - 1 - ar;
      const bool corner = ((z - ar <= 1) || (br - z <= 1)) && ((x - ar <= 1) || (crn - x <= 1));
      const int dz = topc ? 1 : (botc ? -1 : 0), dx = side ? (inr ? 1 : -1) : 0;
      const auto blend = [&](const float* s1, const float* T, const float* s0) {
        const float T0 = T[rc], U0z = s0[rc], U1z = s1[lc];
        const int ri = rc + dz * RW + dx, lat = side ? RW : 1;
        const float Tx = (x - ar <= 1) ? T[rc + 1] : T[rc - 1];
        const float Tz = (z - ar <= 1) ? T[rc + RW] : T[rc - RW];
        const float num_c = U1z + r1v[j] * (Tx + Tz);
        const float den_c = 2.0f * r1v[j] + 1.0f;
        const float Ti = T[ri], U0i = s0[ri], U1i = s1[lc + dz * LW + dx];
        const float tv = m.taoh * vp[j];
        const float t1 = tv * ((Ti - U0i) + U0z);
        const float t2 = ((((-2.0f * U1z) + U0z) + Ti) - 2.0f * U1i) + U0i;
        const float lap = ((((T[ri + lat] - 2.0f * Ti) + T[ri - lat]) + s0[rc + lat]) - 2.0f * U0z) +
                          s0[rc - lat];
        const float t3 = fsv[j] * lap;
        const float num_s = (t1 - t2) + t3;
        const float den_s = tv + 1.0f;
        const float O = (1.0f / (corner ? den_c : den_s)) * (corner ? num_c : num_s);
        return (1.0f - wgt[j]) * T0 + wgt[j] * O;
      };
      if (FWD) nu[j] = blend(su1, tu, tu0);
      if (TWO) nq[j] = blend(sq1, tq, tq0);
    }
  }
  if (!edge || ((MIG || ADJ) && has_inner)) {
    // the columns of the thread's cells, read once
    float cu[CPT + 2 * NFD], cq[TWO ? CPT + 2 * NFD : 1];
#pragma unroll
    for (int i = 0; i < CPT + 2 * NFD; ++i) {
      cu[i] = su1[lc0 + (i - NFD) * LW];
      if (TWO) cq[i] = sq1[lc0 + (i - NFD) * LW];
    }
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      const int z = zw + j, lc = lc0 + j * LW;
      const auto vu = [&](int l) { return cu[j + NFD + l]; };
      const auto vq = [&](int l) { return TWO ? cq[j + NFD + l] : 0.f; };
      if (!edge)
        values(z, x, lc, cw[j], pm[j], u0[j], q0[j], own[j], ext[j], isr[j], vu, vq, &nu[j], &nq[j]);
      if (MIG || ADJ) {  // BKAdd_EFF (kernel.cu:246-320): u(k), kept on the interior
        const float t = combine_p(vu(0), u0[j], pm[j], taps(su1, lc, cw[j], vu), true);
        nu[j] = (z == sg.r_u && x == sg.r_x) ? t + a.wav : t;
      }
    }
  }

#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const int z = zw + j, lc = lc0 + j * LW;
    if (!cell[j]) continue;
    if (FWD || inner[j]) stg(a.u2 + so, own[j], nu[j]);
    if (TWO) stg(a.q2 + so, own[j], nq[j]);
    // strips: saved by the forward pass (Hybrid3, kernel.cu:184-208), restored
    // into the rings of the reconstructed field (BKEqual, 222-245)
    if (FWD && a.save_strips && se[j] >= 0) strip_put(a.st, shot, a.k, se[j], nu[j]);
    if ((MIG || ADJ) && se[j] >= 0) stg(a.u2 + so, own[j], ring[j]);
    int s = 0;  // the receiver records of u(k), of dU(k) in a Born pass
    if (FWD && a.rec && z == rr.s_z && is_receiver(x, rr, &s))
      a.rec[((long long)shot * a.nt + a.k) * rr.n + s] = BORN ? nq[j] : nu[j];
    if (MIG && a.nimg > 0 && inner[j]) {  // imaging of steps k+nimg-1 .. k, in that order
      const auto image = [&](float u, float q) {
        ssu[j] = a.icompen ? ssu[j] + u : u;
        ssq[j] = a.icompen ? ssq[j] + q : q;
        si1[j] = __builtin_fmaf(ssq[j], ssu[j], si1[j]);
        si2[j] = __builtin_fmaf(u, u, si2[j]);
      };
      if (a.nimg >= 3) image(u0[j], q0[j]);
      if (a.nimg >= 2) image(su1[lc], sq1[lc]);
      image(nu[j], nq[j]);
      stg(i1, own[j], si1[j]);
      stg(i2, own[j], si2[j]);
      if (a.icompen) {
        stg(su, own[j], ssu[j]);
        stg(sq, own[j], ssq[j]);
      }
    }
    if (ADJ && inner[j]) {  // G += D2u(k+1) * mu(k+2)
      const float d2u = (u0[j] - 2.0f * su1[lc]) + nu[j];
      stg(i1, own[j], __builtin_fmaf(d2u, q0[j], si1[j]));
    }
  }
}

template <int CPT>
static void go(int pass, dim3 grid, const TileArgs& a, hipStream_t s) {
  constexpr int N = RTM_NFD;
  const dim3 block(512);
  if (pass == TILE_FWD) hipLaunchKernelGGL((k_tile<N, TILE_FWD, CPT>), grid, block, 0, s, a);
  else if (pass == TILE_MIG) hipLaunchKernelGGL((k_tile<N, TILE_MIG, CPT>), grid, block, 0, s, a);
  else if (pass == TILE_BORN) hipLaunchKernelGGL((k_tile<N, TILE_BORN, CPT>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((k_tile<N, TILE_ADJ, CPT>), grid, block, 0, s, a);
}

template <>
hipError_t TileOps<RTM_NFD>::tile(int pass, int cpt, dim3 grid, const TileArgs& a, hipStream_t s) {
  if (cpt == 1) go<1>(pass, grid, a, s);
#if RTM_NFD <= TILE_CPT2_MAX_NFD
  else if (cpt == 2) go<2>(pass, grid, a, s);
#endif
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace rtm
