// rtm_plan.h -- index rules of the launches, free of HIP types so that a CPU
// build can enumerate them (tests/test_plan.py).  Internal header.
#pragma once

#ifdef __HIPCC__
#define RTM_HD __host__ __device__
#else
#define RTM_HD
#endif

namespace rtm {

// k_tile: a tile of th rows by 64 columns at (z0, x0) stages the field on the
// tile and on this many cells around it: the taps of the tile's own cells and,
// where it holds frame cells, of the ring of cells whose pre-blend values they
// read.
RTM_HD constexpr int tile_halo(int nfd) { return nfd + 1; }
// The tile takes the path of tiles with frame cells (n2 deep on an nz x nx grid):
// clamped loads.  The others load without clamps, so what they stage has to lie
// on the grid: where n2 == nfd a tile beside the frame reaches a cell past it and
// takes the clamped path as well.
RTM_HD inline bool tile_edge(int z0, int x0, int th, int nfd, int n2, int nz, int nx) {
  const int e = n2 > tile_halo(nfd) ? n2 : tile_halo(nfd);
  return z0 < e || z0 + th > nz - e || x0 < e || x0 + 64 > nx - e;
}

}  // namespace rtm
