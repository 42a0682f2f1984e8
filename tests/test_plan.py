"""Index rules of the launches (rtm_gpu_amd/csrc/rtm_plan.h), enumerated on the
CPU: the header compiled by itself."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rtm_gpu_amd", "csrc")

SHIM = r"""
#include "rtm_plan.h"
using namespace rtm;
// Tiles of an nz x nx grid that load without clamps and whose staged cells
// leave it.  e: the depth up to which a tile counts as one of the frame (0: the
// kernel's rule).
extern "C" int tiles_outside(int nz, int nx, int n2, int nfd, int th, int e) {
  int bad = 0;
  const int r = tile_halo(nfd);
  for (int z0 = 0; z0 < nz; z0 += th)
    for (int x0 = 0; x0 < nx; x0 += 64) {
      if (e ? z0 < e || z0 + th > nz - e || x0 < e || x0 + 64 > nx - e
            : tile_edge(z0, x0, th, nfd, n2, nz, nx)) continue;
      const int zl = z0 - r, zh = z0 + th + r - 1, xl = x0 - r, xh = x0 + 64 + r - 1;
      bad += zl < 0 || zh >= nz || xl < 0 || xh >= nx;
    }
  return bad;
}
extern "C" int edge_tile(int z0, int x0, int th, int nfd, int n2, int nz, int nx) {
  return tile_edge(z0, x0, th, nfd, n2, nz, nx);
}
extern "C" void tile_work(int nz, int nx, int n2, double* inner, double* edge) {
  BatchWork w;
  w.add(nz, nx, n2, 224, 0.1);
  *inner = w.tile_inner;
  *edge = w.tile_edge;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src, so = d / "plan.cpp", d / "plan.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC,
                    str(src), "-o", str(so)], check=True)
    return C.CDLL(str(so))


@pytest.mark.parametrize("nfd", range(1, 13))
def test_tiles_stage_cells_of_the_grid_only(plan, nfd):
    heights = range(2, 140)
    widths = [w for m in (64, 128, 192) for w in range(m - 3, m + 4)] + [16]
    for n2 in (nfd, nfd + 1, nfd + 5, 32):
        for th in (8, 16):
            for h in heights:
                for w in widths:
                    nz, nx = h + 2 * n2, w + 2 * n2
                    assert plan.tiles_outside(nz, nx, n2, nfd, th, 0) == 0, (nz, nx, n2, th)


def test_a_frame_as_deep_as_the_operator_needs_the_clamp(plan):
    """Row -1 (a tile that starts at n2 == nfd) and row nz (one that ends at
    nz - n2) are what a tile without frame cells would load there."""
    assert plan.tiles_outside(136, 186, 8, 8, 8, 8) > 0
    for nfd in range(1, 13):
        nz = 96 + nfd  # nz - n2 = 96
        assert plan.tiles_outside(nz, 186, nfd, nfd, 8, nfd) > 0, nfd
        assert plan.tiles_outside(nz, 186, nfd, nfd, 16, nfd) > 0, nfd


def test_tiles_with_and_without_frame_cells_are_counted(plan):
    inner, edge = C.c_double(), C.c_double()
    for n2 in (1, 8, 12, 20, 30, 66):
        for nz, nx in ((2 * n2 + 2, 2 * n2 + 2), (261, 233), (411, 1761), (700, 175), (152, 192)):
            plan.tile_work(nz, nx, n2, C.byref(inner), C.byref(edge))
            n = [0, 0]
            for z0 in range(0, nz, 8):
                for x0 in range(0, nx, 64):
                    n[plan.edge_tile(z0, x0, 8, n2 - 1, n2, nz, nx)] += 1
            assert [round(inner.value / 512e-6), round(edge.value / 512e-6)] == n, (nz, nx, n2)
