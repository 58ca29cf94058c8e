// A block of device memory that is kept between calls and grows when one needs more.
#pragma once
#include <algorithm>
#include <cstddef>

namespace ughip {

enum class Grown { YES, NO_MEMORY, FAILED };

// Hip: synchronize() and free(p), true where that went well, and allocate(&p, bytes), YES where it did and NO_MEMORY where there was none.  FAILED is any
// other error, also one that an earlier launch left: it is the caller's to report, whatever could be done without the block.  After NO_MEMORY there is
// no block.
template <typename Hip>
Grown grow_block(Hip&& hip, void** block, size_t* have, size_t bytes, size_t least) {
  if (bytes <= *have) return Grown::YES;
  if (!hip.synchronize()) return Grown::FAILED;  // earlier launches may still read the old block
  if (*block && !hip.free(*block)) return Grown::FAILED;
  *block = nullptr;
  *have = 0;
  const size_t want = std::max(bytes, least);
  const Grown g = hip.allocate(block, want);
  if (g == Grown::YES) *have = want;
  else *block = nullptr;
  return g;
}

}  // namespace ughip
