// dtm_box.h — launches with a lane per cell of a box, plane after plane.
#pragma once
#include <algorithm>

namespace dtm {

// The box is cut into units of m whole x planes: one, or of small planes as many
// as make kBoxUnit cells, so that few lanes are left over at a unit's end.  A
// launch runs blocks [b0, b0 + nblk) of each of some units from u0 on.
struct BoxUnits {
  unsigned nblk, m, u0, b0;
};
constexpr unsigned kBoxBlock = 256;  // lanes
constexpr unsigned kBoxUnit = 2048;

// Plane ip and cell loc of a lane in a box of ni planes of pl cells; false: none.
__host__ __device__ __forceinline__ bool box_lane(const BoxUnits& B, unsigned ni, unsigned long long pl, unsigned block,
                                                  unsigned lane, unsigned& ip, unsigned long long& loc) {
  const unsigned u = block / B.nblk;
  loc = (B.b0 + block - u * B.nblk) * (unsigned long long)kBoxBlock + lane;
  ip = B.u0 + u;
  if (B.m > 1) {  // (32 bits: a unit holds less than 2 kBoxUnit cells)
    const unsigned dp = (unsigned)loc / (unsigned)pl;
    loc = (unsigned)loc - dp * (unsigned)pl;
    ip = dp < B.m ? ip * B.m + dp : ni;
  }
  return loc < pl && ip < ni;
}

// go(units, blocks) for each launch.  The device takes launches of less than 2^32
// lanes (one of more is refused, or runs its blocks modulo 2^32 / kBoxBlock).
template <typename Go>
void box_launches(unsigned ni, unsigned long long pl, Go go, unsigned long long most = (1u << 24) - 1) {
  BoxUnits B{};
  B.m = pl < kBoxUnit ? (unsigned)((kBoxUnit - 1 + pl) / pl) : 1u;
  const unsigned long long blocks = (pl * B.m + kBoxBlock - 1) / kBoxBlock, units = (ni + B.m - 1) / B.m;
  for (unsigned long long b = 0; b < blocks; b += B.nblk) {
    B.b0 = (unsigned)b;
    B.nblk = (unsigned)std::min(blocks - b, most);
    const unsigned long long per = most / B.nblk;
    for (unsigned long long q = 0; q < units; q += per) {
      B.u0 = (unsigned)q;
      go(B, B.nblk * (unsigned)std::min(per, units - q));
    }
  }
}

}  // namespace dtm
