// The candidate indices a quad's walk loads, step by step.
#pragma once

#include <cstdint>

namespace rtp {

// Positions past the last that a neighbour walk's loads of four, or a quad's of sixteen, may read
// (and drop).
constexpr uint32_t kPosPad = 16;

// Lane u of a quad in its walk over the nr index ranges rl (first with a code above INDEX_MASK's
// bits, last), sixteen candidates a step: the lane's are e, e + 4, e + 8 and e + 12, those at most
// hi are the range's.  The wave steps until its longest quad is done.  A quad without a range left
// (or without one at all) stays at e = 1, hi = 0, so a lane never loads past e + 12 <= hi + 15 of
// a range in use, or 13 without one: with every hi below the number of positions, less than
// kPosPad past them.
template <class Range, uint32_t INDEX_MASK = 0xffffffffu>
struct QuadScan {
  const Range* rl;
  uint32_t nr, u;
  uint32_t ri = 0, e = 1u, hi = 0u, code = 0u;

  __device__ __forceinline__ QuadScan(const Range* ranges, uint32_t count, uint32_t lane)
    : rl(ranges), nr(count), u(lane)
  {
    if (nr > 0u)
      open();
  }
  __device__ __forceinline__ bool more() const { return ri < nr; }
  __device__ __forceinline__ void open()
  {
    const Range r = rl[ri];
    e = (r.x & INDEX_MASK) + u;
    code = r.x & ~INDEX_MASK;
    hi = r.y;
  }
  __device__ __forceinline__ void next()
  {
    e += 16u;
    if (e - u > hi) {  // always without a range
      e = 1u;
      hi = 0u;
      code = 0u;
      if (++ri < nr)
        open();
    }
  }
};

}  // namespace rtp
