// Which thread of the one-electron kernels takes which shell pair: kOneElLanes
// lanes to a pair, every thread a pair of its own and then, where a class has
// more pairs than the largest grid, those a grid's pairs further on.  All of it
// in 64 bits: a class has up to 2^31 pairs, its lanes are eight times as many.
#pragma once

namespace rchem {

constexpr int kOneElLanes = 8;
constexpr int kOneElBlock = 256;
constexpr long long kOneElMaxBlocks = 65536;  // 2^24 threads, two million pairs at once

constexpr long long one_el_blocks(long long pairs) {
  const long long per = kOneElBlock / kOneElLanes, blocks = (pairs + per - 1) / per;
  return blocks < kOneElMaxBlocks ? blocks : kOneElMaxBlocks;
}
// A thread's first pair of the class, and how far it is to the next.
constexpr long long one_el_first(unsigned block, unsigned thread) {
  return (static_cast<long long>(block) * kOneElBlock + thread) / kOneElLanes;
}
constexpr long long one_el_step(unsigned blocks) {
  return static_cast<long long>(blocks) * (kOneElBlock / kOneElLanes);
}

}  // namespace rchem
