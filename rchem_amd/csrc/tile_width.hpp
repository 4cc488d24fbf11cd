// Widths of the host-built tiles (64 >> shift quartets).
#pragma once

namespace rchem {

// How a kernel works through a tile's quartets.
enum class TileEngine {
  kLane,   // one lane to a quartet: a narrower tile only leaves lanes idle
  kLanes,  // 1 << Tile::pad lanes to a quartet (kModeTensor, kModeDiag)
  kWave    // the wave takes one quartet after the other
};

// At most 8 lanes to a quartet, and no more tiles than give a class (or a bucket
// of it) 8 waves to a SIMD.  A lane's chain of primitive quartets was the time of
// a small tensor's kernels: (H2O)_3 6-31G (ss|ss) 0.289 -> 0.080 ms, all classes
// 0.89 -> 0.23, the call 2.35 -> 1.66; of the bounds of (H2O)_8, (ss|ss) and
// (ps|ps): 0.42 and 0.14 -> 0.07 and 0.03 ms.
constexpr int kTileMaxShift = 3;
constexpr double kTileMaxWaves = 8192.0;

// The shift for `waves` tiles of 64 quartets; np: primitive pairs of the ket, a
// lane's least share (kLanes).
constexpr int tile_shift(TileEngine engine, double waves, int np) {
  if (engine == TileEngine::kLane) return 0;
  int sh = 0;
  while (sh < kTileMaxShift && waves * (2 << sh) <= kTileMaxWaves &&
         (engine == TileEngine::kWave || (2 << sh) <= np))
    ++sh;
  return sh;
}

}  // namespace rchem
