// The deal of the W4A16 grouped GEMMs' work (gemm_items.hpp): every block of
// every row tile is taken once, and no XCD gets more than its share, for lists
// of tiles as the routing kernel orders them (most sub-tiles first).  Built and
// run by tests/test_gemm_items.py; prints "ok".
#include <algorithm>
#include <cstdio>
#include <vector>

#include "gemm_items.hpp"

using namespace mimoe;

static bool check(const std::vector<unsigned>& subs, unsigned nb) {
  const unsigned n = (unsigned)subs.size(), grid = (n + kXcds - 1) / kXcds * kXcds * nb;
  std::vector<int> taken(n * nb, 0);
  long load[kXcds] = {}, total = 0;
  for (unsigned b = 0; b < grid; ++b) {
    const unsigned first = gemm_item(b, nb, false).tile / kXcds * kXcds, last = std::min(first + kXcds, n) - 1;
    const GemmItem it = gemm_item(b, nb, gemm_even(first, n, subs[first], subs[last]));
    if (it.tile / kXcds != first / kXcds || it.blk >= nb) return false;
    if (it.tile >= n) continue;
    ++taken[it.tile * nb + it.blk];
    load[b % kXcds] += subs[it.tile];
    total += subs[it.tile];
  }
  for (int c : taken)
    if (c != 1) return false;
  // a tile spread over the XCDs gives one of them at most one block (of at
  // most 4 sub-tiles) more than the mean; equal tiles give each the same
  long over = 0;
  for (unsigned first = 0; first < n; first += kXcds) {
    const unsigned last = std::min(first + kXcds, n) - 1;
    if (last - first + 1 < kXcds || subs[first] != subs[last])
      for (unsigned t = first; t <= last; ++t) over += subs[t];
  }
  for (long l : load)
    if (l * (long)kXcds > total + (long)kXcds * over) return false;
  return true;
}

int main() {
  for (unsigned nb : {1u, 2u, 3u, 6u, 7u, 8u, 12u, 16u, 24u, 112u})
    for (unsigned n = 1; n <= 200; n = n < 40 ? n + 1 : n + 13)
      for (unsigned heavy = 0; heavy <= n; heavy = heavy < 10 ? heavy + 1 : 2 * heavy)
        for (unsigned mid = 0; mid <= 9 && heavy + mid <= n; mid += 3) {
          std::vector<unsigned> subs(n, 1);
          for (unsigned t = 0; t < heavy + mid; ++t) subs[t] = t < heavy ? 4 : 2;
          if (!check(subs, nb)) {
            printf("nb %u, %u tiles, %u of 4 and %u of 2 sub-tiles\n", nb, n, heavy, mid);
            return 1;
          }
        }
  printf("ok\n");
  return 0;
}
