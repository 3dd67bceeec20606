// Reads the number of products, the units that run at once, the work of a brief one,
// and each product's work and units where its 64ths begin; prints the bounds of the eight XCDs' units (tests/test_xcd_split.py).
#include <cstdio>
#include <vector>

#include "cq_split.h"

int main() {
  int n = 0, at_once = 0, brief = 0;
  if (std::scanf("%d %d %d", &n, &at_once, &brief) != 3 || n < 1) return 1;
  std::vector<cq::WorkParts> parts(n);
  std::vector<const cq::WorkParts *> p;
  for (cq::WorkParts &w : parts) {
    long long work;
    if (std::scanf("%lld", &work) != 1) return 1;
    w.work = work;
    for (int32_t &u : w.at)
      if (std::scanf("%d", &u) != 1) return 1;
    p.push_back(&w);
  }
  int32_t xcd[cq::kXcds + 1];
  cq::xcd_split(p.data(), n, at_once, brief, xcd);
  for (int32_t u : xcd) std::printf("%d ", u);
  return 0;
}
