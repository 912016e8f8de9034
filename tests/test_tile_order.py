"""CPU check of the tile order of the fused VIV passes (``window_tiles`` and
``tile_of_block`` of csrc/viv2d.hpp, compiled for the host): with one window
origin, the blocks of a launch take every tile once.  With the origin of a
later step in some of the blocks they do not, so what a pass takes its origin
from must not change while the pass runs."""

import os
import subprocess

from vivsim_amd import _build

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "step_impl.hpp"
#include "viv2d.hpp"
using namespace vsx;

// how often each tile is taken when the blocks before `split` use origin (a0, a1), the others (b0, b1)
static int missed(const Tiles &T, int S, int a0, int a1, int b0, int b1, int split) {
  std::vector<int> hits(T.ntx * T.nty, 0);
  int r[2][4];
  window_tiles(T, a0 - 2, a1 - 2, S + 4, r[0][0], r[0][1], r[0][2], r[0][3]);
  window_tiles(T, b0 - 2, b1 - 2, S + 4, r[1][0], r[1][1], r[1][2], r[1][3]);
  for (int p = 0; p < T.ntx * T.nty; ++p) {
    const int *w = r[p < split ? 0 : 1];
    int tx, ty;
    bool in_win;
    tile_of_block(p, T, w[0], w[1], w[2], w[3], tx, ty, in_win);
    if (tx < 0 || tx >= T.ntx || ty < 0 || ty >= T.nty) return -1;
    if (in_win != (tx >= w[0] && tx <= w[1] && ty >= w[2] && ty <= w[3])) return -1;
    ++hits[tx * T.nty + ty];
  }
  int n = 0;
  for (int h : hits) n += h == 0;
  return n;
}

int main() {
  const int grids[][2] = {{160, 120}, {1031, 777}, {2052, 2000}, {64, 1500}};
  for (auto &g : grids) {
    Tiles T;
    T.TY = (g[1] + 63) / 64 * 64 > 256 ? 256 : (g[1] + 63) / 64 * 64;
    T.TX = kTileCells / T.TY;
    T.ntx = (g[0] + T.TX - 1) / T.TX;
    T.nty = (g[1] + T.TY - 1) / T.TY;
    for (int S : {4, 28, 52})
      for (int x = 2; x + S + 2 <= g[0]; x += x < 20 || x + S + 22 > g[0] ? 1 : 7)
        for (int y = 2; y + S + 2 <= g[1]; y += y < 20 || y + S + 22 > g[1] ? 1 : 61)
          if (missed(T, S, x, y, x, y, 0)) { printf("grid %d x %d window %d at %d, %d\n", g[0], g[1], S, x, y); return 1; }
  }
  // the rows before the window are taken in order, counted from its number of tiles
  const Tiles T = {4, 256, 1024, 16};
  const int n = missed(T, 60, 1021, 2018, 1022, 2018, 2000);
  printf("two origins: %d tiles missed\n", n);
  return n > 0 ? 0 : 1;
}
"""


def test_blocks_take_every_tile_once(tmp_path):
    src, exe = tmp_path / "tiles.hip", tmp_path / "tiles"
    src.write_text(PROGRAM)
    subprocess.run([_build.HIPCC, *_build.FLAGS, "--offload-host-only", "-O1", "-I", _build.CSRC, "-c", str(src),
                    "-o", str(tmp_path / "tiles.o")], check=True, capture_output=True)
    capi = os.path.join(_build.HERE, "libvivsim_amd.so")
    subprocess.run([_build.HIPCC, str(tmp_path / "tiles.o"), capi, "-o", str(exe), f"-Wl,-rpath,{_build.HERE}"],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
