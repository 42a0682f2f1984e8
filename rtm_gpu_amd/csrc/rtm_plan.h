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
// The tile holds cells of the frame (n2 deep on an nz x nx grid).
RTM_HD inline bool tile_edge(int z0, int x0, int th, int n2, int nz, int nx) {
  return z0 < n2 || z0 + th > nz - n2 || x0 < n2 || x0 + 64 > nx - n2;
}
// All that the tile stages lies on the grid.  A tile without frame cells reaches
// a cell past it where n2 == nfd: the outermost ring, of which it uses nothing.
RTM_HD inline bool tile_inside(int z0, int x0, int th, int nfd, int nz, int nx) {
  const int r = tile_halo(nfd);
  return z0 >= r && z0 + th + r <= nz && x0 >= r && x0 + 64 + r <= nx;
}
// Such a tile loads without clamps, every other one through the outer mirror.
RTM_HD inline bool tile_direct(int z0, int x0, int th, int nfd, int n2, int nz, int nx) {
  return !tile_edge(z0, x0, th, n2, nz, nx) && tile_inside(z0, x0, th, nfd, nz, nx);
}

}  // namespace rtm
