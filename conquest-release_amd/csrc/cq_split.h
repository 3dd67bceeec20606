// Launch units (tiles; uniform sizes: quadrants of tiles) to the eight XCDs.
#pragma once

#include <algorithm>
#include <cstdint>

namespace cq {

constexpr int kXcds = 8;
constexpr int kWorkParts = 64;

// Work of one product's launch units (record words, k-steps or entries) and the
// units where each 64th of it begins; at[64] = the number of units.
struct WorkParts {
  int64_t work = 0;
  int32_t at[kWorkParts + 1] = {};
};

// Units [xcd[x], xcd[x + 1]) of n products, numbered one product after the other,
// run on XCD x: consecutive units, which share an L2, of equal work. Units are
// unequal (truncated tiles, the diagonal tiles of symmetric plans, species), and
// with equal counts or fixed runs per XCD the last XCD decides. An eighth of the
// units each / runs of 8192 / equal work: 13x13 1024 atoms symmetric 15.8 / 13.5
// / 13.1 ms, 4/9/13 mixes of 4096 atoms 27.5 / 26.8 / 26.9, of 8192 atoms 54.0 /
// 55.0 / 53.9, of 2048 atoms symmetric 3.90 / 3.90 / 3.11 ms. Within a product the
// bounds are exact to a 64th, between two of them taken in proportion. At most
// `at_once` units, which all run at the same time, are split by count where their
// mean work is at most `brief`: there the fullest compute unit decides.
inline void xcd_split(const WorkParts *const *p, int n, int32_t at_once, int32_t brief, int32_t xcd[kXcds + 1]) {
  int32_t total = 0;
  int64_t work = 0;
  for (int j = 0; j < n; ++j) {
    total += p[j]->at[kWorkParts];
    work += p[j]->work;
  }
  if (total <= at_once && work <= (int64_t)total * brief) {
    const int32_t each = (total + kXcds - 1) / kXcds;
    for (int x = 0; x <= kXcds; ++x) xcd[x] = std::min(total, x * each);
    return;
  }
  double all = 0.0, before = 0.0;
  for (int j = 0; j < n; ++j) all += (double)p[j]->work;
  int32_t base = 0;
  int x = 0;
  for (int j = 0; j < n; ++j) {
    const double work = (double)p[j]->work;
    for (; x < kXcds && all * x / kXcds < before + work; ++x) {
      const double part = std::max(0.0, (all * x / kXcds - before) / work * kWorkParts);
      const int k = std::min((int)part, kWorkParts - 1);
      const int32_t *at = p[j]->at;
      xcd[x] = base + std::min(at[k] + (int32_t)((part - k) * (at[k + 1] - at[k])), at[kWorkParts]);
    }
    before += work;
    base += p[j]->at[kWorkParts];
  }
  for (; x <= kXcds; ++x) xcd[x] = base;
  xcd[0] = 0;
}

}  // namespace cq
