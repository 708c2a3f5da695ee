// gemm_items.hpp -- which block of which row tile a workgroup of the W4A16
// grouped GEMMs takes.  Plain C++: used by the kernels and by a host check.
#pragma once

namespace mimoe {

constexpr unsigned kXcds = 8;   // workgroup b runs on XCD b % 8

struct GemmItem {
  unsigned tile, blk;   // row tile, block (of nb) of output rows
};

// Work item of workgroup b.  The 8 * nb workgroups of a group of 8 consecutive
// tiles give each XCD one tile (even), or spread every tile over all XCDs (a
// tile's workgroups are consecutive).
constexpr GemmItem gemm_item(unsigned b, unsigned nb, bool even) {
  const unsigned t = b / nb, first = t - t % kXcds, w = b - first * nb;
  return even ? GemmItem{first + w % kXcds, w / kXcds} : GemmItem{t, b - t * nb};
}

// Whether the group of 8 tiles that starts at tile `first` of ntiles is dealt
// one tile to an XCD: it is whole, and its first and last tile have the same
// number of sub-tiles (s0, s7), so all have, as the list is ordered by it.
constexpr bool gemm_even(unsigned first, unsigned ntiles, unsigned s0, unsigned s7) {
  return first + kXcds <= ntiles && s0 == s7;
}

}  // namespace mimoe
