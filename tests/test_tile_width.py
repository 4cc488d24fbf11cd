"""Widths of the host-built tiles (tile_width.hpp), compiled for the CPU: a kernel
with one lane to a quartet always gets tiles of 64, and the gradient's tile list
asks for the widths of its own kernels, not of the tensor's."""
import os
import re
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rchem_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "tile_width.hpp"
using namespace rchem;
int main() {
  const double waves[] = {0.25, 1, 2, 100, 1023, 1024, 1025, 2048, 4096, 4097, 8192, 1e6, 1e9};
  for (double w : waves)
    for (int np = 1; np <= 64; ++np) {
      if (tile_shift(TileEngine::kLane, w, np) != 0) return 1;
      const int lanes = tile_shift(TileEngine::kLanes, w, np), wave = tile_shift(TileEngine::kWave, w, np);
      if ((1 << lanes) > np || lanes > 3 || wave > 3 || lanes > wave) return 2;
      // narrowed no further than 8192 tiles
      if ((lanes && w * (1 << lanes) > 8192.0) || (wave && w * (1 << wave) > 8192.0)) return 3;
    }
  if (tile_shift(TileEngine::kLanes, 1024, 8) != 3 || tile_shift(TileEngine::kLanes, 1025, 8) != 2) return 4;
  if (tile_shift(TileEngine::kLanes, 1, 3) != 1 || tile_shift(TileEngine::kWave, 1, 1) != 3) return 5;
  return 0;
}
"""


def test_shifts(tmp_path):
    (tmp_path / "main.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-o", exe, str(tmp_path / "main.cpp")], check=True)
    assert subprocess.run([exe]).returncode == 0


def test_gradient_asks_for_its_own_kernels():
    with open(os.path.join(CSRC, "rchem_api.cpp")) as fh:
        text = fh.read()
    grad = text[text.index("int rchem_rhf_gradient("):]
    assert re.search(r"prepare_host_tiles\(ctx, tau, kTilesGradient\)", grad)
    tiles = text[text.index("int prepare_host_tiles("):]
    tiles = tiles[:tiles.index("\n}")]
    assert "eri_grad_launcher(" in tiles and "ctx->tiles_use == use" in tiles
