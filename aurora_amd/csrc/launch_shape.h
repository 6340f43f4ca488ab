// Launch shape of the persistent traversals: the LDS of a block.  Host arithmetic
// only.
#pragma once

#include <cstddef>
#include <cstdint>

namespace aur {

// LDS is allocated in granules of 1280 bytes.  Sizes are rounded up to them here:
// the occupancy query divides the CU's 160 KB by the size as given, and a grid of
// its blocks is then too large, so that some start when the others have ended (a
// batch of trees of 17 levels with every row, 16 KB: 10 blocks per CU said, 9
// resident; 21.2 ms, 17.4 with a grid of 9).
constexpr size_t kLdsGranule = 1280;
inline size_t lds_granules(size_t bytes) { return (bytes + kLdsGranule - 1) / kLdsGranule * kLdsGranule; }

// LDS of a block so that at most `blocks` of them reside on a CU: `need`, or
// that share of its 160 KB (a granule less).
inline size_t lds_for_blocks(size_t need, uint32_t blocks) {
  const size_t share = (163840 - kLdsGranule) / blocks / kLdsGranule * kLdsGranule;
  return lds_granules(need > share ? need : share);
}

}  // namespace aur
