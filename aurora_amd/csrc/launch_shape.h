// Launch shape of the persistent traversals: the LDS of a block and the rows of
// each lane's stack that live in it.  Host arithmetic only.
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

struct StackShape {
  uint32_t rows, maxrows;  // rows in LDS; rows a tree needs
  size_t lds;              // bytes per block
};

// Stack of a tree of `levels` (at most levels - 1 deferred entries, float2 rows)
// for blocks of `block` threads.  want: rows to keep in LDS (0: every row).
// cu_waves: waves that a CU is to hold at most (0: as many as fit).  A window of
// fewer rows than the tree needs that the caller chose (chosen) is there to let
// more waves reside, so it is not limited; otherwise what the limit reserves
// anyway holds further rows.
inline StackShape stack_shape(uint32_t levels, uint32_t want, bool chosen, uint32_t block, uint32_t cu_waves) {
  StackShape s{};
  s.maxrows = levels > 1 ? levels - 1 : 1;
  s.rows = want == 0 || want >= s.maxrows ? s.maxrows : want;
  const size_t row = (size_t)block * 8;
  s.lds = lds_granules(s.rows * row);
  if (cu_waves == 0 || (chosen && s.rows < s.maxrows)) return s;
  s.lds = lds_for_blocks(s.lds, cu_waves * 64 / block);
  if (s.rows < s.maxrows) s.rows = s.lds / row < s.maxrows ? (uint32_t)(s.lds / row) : s.maxrows;
  return s;
}

}  // namespace aur
