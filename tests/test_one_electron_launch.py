"""The one-electron kernels' launch arithmetic (one_electron_launch.hpp), compiled
for the CPU: every shell pair of a class is taken, by all of its lanes and once,
for any number of pairs that fits the pair list's 32-bit index."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rchem_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "one_electron_launch.hpp"
using namespace rchem;
int main(int argc, char** argv) {
  const long long pairs = std::atoll(argv[1]), blocks = one_el_blocks(pairs);
  const unsigned b = static_cast<unsigned>(blocks);
  // a launch takes fewer than 2^31 workgroups and 2^32 threads
  if (blocks < 1 || blocks * kOneElBlock >= (1ll << 32)) return 1;
  const long long step = one_el_step(b);
  // the threads' first pairs are 0 .. step - 1, eight threads to each and in order
  if (one_el_first(0, 0) != 0 || one_el_first(b - 1, kOneElBlock - 1) != step - 1) return 2;
  if (pairs < (1 << 20)) {
    std::vector<int> lanes(pairs, 0);
    for (unsigned k = 0; k < b; ++k)
      for (unsigned t = 0; t < kOneElBlock; ++t)
        for (long long p = one_el_first(k, t); p < pairs; p += step)
          lanes[p] |= 1 << t % kOneElLanes;
    for (int x : lanes)
      if (x != (1 << kOneElLanes) - 1) return 3;
  } else {
    // the last pair: its thread reaches it in whole steps
    const long long last = pairs - 1, first = last % step;
    const unsigned k = static_cast<unsigned>(first / (kOneElBlock / kOneElLanes));
    const unsigned t = static_cast<unsigned>(first % (kOneElBlock / kOneElLanes)) * kOneElLanes;
    if (one_el_first(k, t) != first || (last - first) % step != 0) return 4;
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("launch")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-o", str(d / "main"), str(d / "main.cpp")],
                   check=True)
    return str(d / "main")


@pytest.mark.parametrize("pairs", [
    1, 31, 32, 33, 255, 256, 257, 1000,
    65536 * 32 - 1, 65536 * 32, 65536 * 32 + 1,  # the largest grid's pairs
    (1 << 28) - 1, 1 << 28, (1 << 28) + 1,       # lanes at 2^31
    (1 << 29) - 1, 1 << 29,                      # lanes at 2^32
    32768 * 32769 // 2, (1 << 31) - 1])
def test_every_pair_is_taken(program, pairs):
    assert subprocess.run([program, str(pairs)]).returncode == 0


def test_grid_and_index_come_from_it():
    """The kernel takes its pairs, and its launch the grid, from these functions."""
    with open(os.path.join(CSRC, "one_electron.hip")) as fh:
        text = fh.read()
    assert "dim3(static_cast<unsigned>(one_el_blocks(cnt)))" in text
    assert "p += one_el_step(gridDim.x)" in text and "* kOneElLanes" not in text
