// A CPU model of the quad walks' loads: waves of sixteen quads whose range lists differ as much as
// they can (none, one, 27 of up to the cell cap's length), stepped as the walks step, until the
// wave's longest quad is done.  Every loaded index stays below maxN + kPosPad, and the candidates
// tested are the ranges' own, in order.
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

#define __device__
#define __forceinline__ inline
#include "rtp_quad_scan.hpp"

namespace {

struct Range {
  uint32_t x, y;
};
constexpr uint32_t kMask = (1u << 28) - 1u;

template <uint32_t MASK>
bool run_wave(const std::vector<std::vector<Range>>& quads, uint32_t maxN)
{
  using Scan = rtp::QuadScan<Range, MASK>;
  const uint32_t limit = maxN + rtp::kPosPad;
  std::vector<Scan> lanes;
  std::vector<std::vector<uint32_t>> seen(quads.size());
  for (const auto& q : quads)
    for (uint32_t u = 0; u < 4u; ++u)
      lanes.emplace_back(q.data(), (uint32_t)q.size(), u);
  const auto inside = [&]() {
    for (const Scan& s : lanes)
      if (s.e + 12u >= limit) {
        std::printf("index %u of %u positions\n", s.e + 12u, limit);
        return false;
      }
    return true;
  };
  const auto more = [&]() {
    for (const Scan& s : lanes)
      if (s.more())
        return true;
    return false;
  };
  if (!inside())  // the first loads
    return false;
  do {
    for (int half = 0; half < 2; ++half) {  // two steps between the tests of the loop
      for (size_t q = 0; q < quads.size(); ++q)
        for (uint32_t j = 0; j < 4u; ++j)
          for (uint32_t u = 0; u < 4u; ++u) {
            const Scan& s = lanes[4u * q + u];
            if ((int32_t)(s.hi - s.e) >= 4 * (int32_t)j)
              seen[q].push_back((s.e + 4u * j) | s.code);
          }
      for (Scan& s : lanes)
        s.next();
      if (!inside())
        return false;
    }
  } while (more());
  for (size_t q = 0; q < quads.size(); ++q) {
    std::vector<uint32_t> want;
    for (const Range& r : quads[q])
      for (uint32_t e = r.x & MASK; e <= r.y; ++e)
        want.push_back(e | (r.x & ~MASK));
    if (want != seen[q]) {
      std::printf("quad %zu of %zu: %zu candidates, %zu wanted\n", q, quads.size(), seen[q].size(), want.size());
      return false;
    }
  }
  return true;
}

template <uint32_t MASK>
bool run_all(uint32_t maxN, std::mt19937& rng)
{
  const auto upto = [&](uint32_t n) { return (uint32_t)(rng() % n); };
  for (int trial = 0; trial < 40; ++trial) {
    std::vector<std::vector<Range>> quads(16);
    for (auto& q : quads) {
      const uint32_t counts[] = { 0u, 1u, 9u, 27u, upto(28u) };
      const uint32_t n = counts[upto(5u)];
      for (uint32_t k = 0; k < n; ++k) {
        const uint32_t len = 1u + upto(upto(2u) ? 100u : 12u);  // a column of capped cells: 300
        const uint32_t lo = upto(maxN), hi = lo + len - 1u < maxN ? lo + len - 1u : maxN - 1u;
        q.push_back(Range{ lo | (upto(16u) << 28 & ~MASK), hi });
      }
    }
    if (trial == 0)  // wrapping columns: 27 ranges beside quads without any
      for (size_t k = 0; k < quads.size(); ++k)
        quads[k].assign(k == 5 ? 27 : 0, Range{ maxN - 1u - upto(maxN < 10u ? maxN : 10u), maxN - 1u });
    if (!run_wave<MASK>(quads, maxN)) {
      std::printf("maxN %u, trial %d\n", maxN, trial);
      return false;
    }
  }
  return true;
}

}  // namespace

int main()
{
  std::mt19937 rng(1);
  for (uint32_t maxN : { 1u, 2u, 15u, 16u, 17u, 80u, 300u, 4096u })
    if (!run_all<0xffffffffu>(maxN, rng) || !run_all<kMask>(maxN, rng))
      return 1;
  std::printf("ok\n");
  return 0;
}
