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

// ---- which kernels a batch takes ----------------------------------------------
// What the kernels work on in a step of a batch, in millions of cells, padding
// included.
struct BatchWork {
  double tile_inner = 0, tile_edge = 0;  // k_tile: tiles without and with frame cells
  double wave = 0, wave_two = 0;         // waves of k_interior (256 columns), of k_two
  double inner = 0, frame = 0;           // cells of the interior, of the frame
  double quad = 1;                       // shots of full blocks of four per shot
  double windows = 0;                    // cells times distinct model windows per shot
  double lines = 0;                      // cells times coefficient lines per cell
  // a shot of an nz x nx grid; two_cols: columns of a wave of k_two; line_share:
  // 128-byte lines of the coefficient table that 256 cells of a row touch, per cell
  void add(int nz, int nx, int n2, int two_cols, double line_share) {
    const int mnz = nz - 2 * n2, mnx = nx - 2 * n2;
    const auto split = [n2](int n, int t, double* all, double* in) {  // tiles of t along n cells
      *all = (n + t - 1) / t;
      const int lo = (n2 + t - 1) / t, hi = (n - n2) / t;  // those from n2 to n - n2
      *in = hi > lo ? hi - lo : 0;
    };
    double az, iz, ax, ix;
    split(nz, 8, &az, &iz);
    split(nx, 64, &ax, &ix);
    tile_inner += iz * ix * 512e-6;
    tile_edge += (az * ax - iz * ix) * 512e-6;
    wave += (mnx + 255) / 256 * 256 * 1e-6 * mnz;
    wave_two += (mnx + two_cols - 1) / two_cols * 256 * 1e-6 * mnz;
    inner += 1e-6 * mnz * mnx;
    frame += 1e-6 * nz * nx - 1e-6 * mnz * mnx;
    lines += line_share * 1e-6 * nz * nx;
  }
};

// Microseconds of a forward and a backward step by half-length 1..12, fitted to
// 1500 timed batches: ten grids of 75 to 2400 columns, 2 to 93 M cells,
// least-squares rows up to half-length 5, Taylor rows above.  A marching wave
// spends 0.5 to 1 us on each of its 20 to 30 rows whatever the batch, pads the
// interior to 256 columns and gathers a coefficient row per cell, which costs by
// the lines that its cells touch (a tenth of a line per cell in a smooth model,
// 0.6 to 0.8 in a rough one: then it takes up to 1.7 times as long); k_tile is two
// memory accesses deep but bound by instruction issue, the more the longer the
// operator and the more of its tiles hold frame cells; k_two reads planes and takes
// two steps per pass over memory.  The sums are within 25% of the times; the kernel
// with the smallest one took on average 0.6% longer than the fastest, at worst 1.2
// times as long.  One line on the cells times the half-length, which knows neither
// the grid's shape nor the model, was 5% off on average and up to twice as slow: 171
// shots of 261 x 133 at half-length 8, 60 steps each way, 16.7 ms by k_tile, 10.0 by
// the marching kernels.
namespace cost {
constexpr int kN = 12;
constexpr double kTile[kN][3] = {  // per launch, tiles without, with frame cells
    {3, 14.6, 18.3}, {1, 15.6, 19.4}, {1, 16.1, 20.4}, {1, 17.1, 21.7}, {1, 17.7, 22.6}, {4, 18.6, 23.0},
    {4, 19.5, 26.7}, {6, 21.7, 30.8}, {7, 22.1, 31.8}, {8, 22.9, 33.6}, {9, 22.8, 33.8}, {10, 23.6, 34.0}};
constexpr double kMarch[kN][4] = {  // per launch, waves, frame cells, interior cells
    {37, 4.7, 16, 5.9}, {40, 4.7, 16, 5.8}, {40, 4.8, 16, 5.6}, {48, 4.9, 18, 7.6}, {48, 6.2, 15, 6.2},
    {56, 6.8, 10, 4.7}, {62, 6.5, 11, 4.5}, {70, 6.9, 10, 4.2}, {79, 6.9, 11, 3.2}, {86, 6.6, 14, 2.3},
    {97, 5.9, 13, 2.6}, {109, 5.7, 11, 1.0}};
constexpr double kTwo[5][4] = {{30, 3.8, 14.4, 3.1}, {35, 4.3, 14.9, 2.6}, {46, 5.3, 14.0, 2.1},
                               {52, 5.4, 18.0, 1.3}, {65, 7.5, 17.5, 0.5}};
// the same of a Born and an adjoint step (half-lengths 7, 9, 11 between their
// neighbours)
constexpr double kTile2[kN][3] = {
    {10, 17.4, 19.8}, {1, 20.7, 23.5}, {1, 21.4, 25.2}, {1, 24.8, 27.1}, {1, 27.9, 34.0}, {1, 25.4, 33.8},
    {4, 25.6, 34.7}, {7, 25.9, 35.6}, {9, 31, 51}, {11, 35.7, 66}, {13, 36.6, 66}, {15, 37.5, 66}};
constexpr double kMarch2[kN][4] = {
    {17, 7.5, 33, 10.8}, {26, 8.3, 31, 11.2}, {46, 9.0, 29, 10.8}, {62, 9.8, 33, 13}, {95, 11.3, 25, 12.4},
    {75, 9.9, 25, 7}, {90, 10.6, 25, 6.3}, {105, 11.4, 24, 5.5}, {119, 12, 27, 3}, {133, 12.5, 31, 0.3},
    {147, 11.7, 31, 0.2}, {161, 10.8, 31, 0}};

// Coefficient lines beyond those of the fitted models, in millions.
inline double more_lines(const BatchWork& w, int nfd) {
  return w.lines - (nfd <= 5 ? 0.1 : 0.004) * (w.inner + w.frame);
}
inline double tile(const BatchWork& w, int nfd, bool both, bool ls) {
  const double* k = both ? kTile2[nfd - 1] : kTile[nfd - 1];
  const double win = !both ? 2.0 : ls ? 2.3 + 1.9 * nfd : 2.5;  // a window's planes from memory
  return k[0] + k[1] * w.tile_inner + k[2] * w.tile_edge + win * w.windows +
         (both ? 4.2 : 2.6) * more_lines(w, nfd);
}
inline double march(const BatchWork& w, int nfd, bool both, bool ls) {
  const double* k = both ? kMarch2[nfd - 1] : kMarch[nfd - 1];
  const double win = !both ? 3.2 : ls ? 7 + 2.6 * nfd : 5.0;
  return k[0] + k[1] * w.wave + k[2] * w.frame + k[3] * w.inner + win * w.windows +
         (both ? 16.0 : 12.7) * more_lines(w, nfd);
}
inline double two(const BatchWork& w, int nfd) {  // windows: shared by four shots at least
  const double* k = kTwo[nfd - 1];
  return k[0] + k[1] * w.wave_two * w.quad + k[2] * w.frame * w.quad + k[3] * w.inner;
}
}  // namespace cost

}  // namespace rtm
