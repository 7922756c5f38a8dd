/*
 * packed_walk.h - which blocks a workgroup of the usual packed kernels moves (hip_layer.h: cuttHipPackedWalk).  Plain integer
 * code: the kernels compile it for the device, tests for the host.
 */
#ifndef CUTT_PACKED_WALK_H
#define CUTT_PACKED_WALK_H

#include "tile_walk.h"

namespace cutt {

// Block number `n`, the i-th one of a workgroup -> slab class, Mbar position, and what the slabs add to the block's base offsets; false: no
// block.  Every constant is there from the start (in registers, or in memory at addresses that are), the divisions are multiply-high
// ones on the scalar unit.  ONE: blocks are numbered as workgroups.
template <bool ONE, typename Walk>
CUTT_DEVICE bool packedWalkSlabs(uint32_t n, uint32_t i, uint32_t shifts, uint32_t items, uint32_t num0, uint32_t mul0, uint32_t num1, uint32_t mul1,
                                 const Walk& a, uint32_t& cls, uint32_t& m, uint32_t& offIn, uint32_t& offOut) {
  if (n >= items) return false;
  const uint32_t t = walkDivide(n, mul0, shifts & 31), s0 = n - t * num0;
  m = walkDivide(t, mul1, (shifts >> 5) & 31);
  const uint32_t s1 = t - m * num1;
  if constexpr (!ONE) {
    m = m * a.mulM + i * a.stepM;
    if (m >= a.volMbar) return false;
  }
  cls = (s0 < a.slab[0].rem ? 1u : 0u) + (s1 < a.slab[1].rem ? 2u : 0u);
  const uint32_t e0 = s0 < a.slab[0].rem ? s0 : a.slab[0].rem, e1 = s1 < a.slab[1].rem ? s1 : a.slab[1].rem;
  offIn = s0 * a.slab[0].stepIn + e0 * a.slab[0].strideIn + s1 * a.slab[1].stepIn + e1 * a.slab[1].strideIn;
  offOut = s0 * a.slab[0].stepOut + e0 * a.slab[0].strideOut + s1 * a.slab[1].stepOut + e1 * a.slab[1].strideOut;
  return true;
}

// What Mbar position m adds.
template <typename Walk>
CUTT_DEVICE void packedWalkMbar(const Walk& a, uint32_t m, uint32_t& offIn, uint32_t& offOut) {
  auto ranks = [&](int from) __attribute__((always_inline)) {
#pragma unroll
    for (int k = from; k < from + 4; k++) {  // (unused ranks have zeros everywhere)
      const uint32_t q = walkDivide(m, a.rank[k].mul, a.rank[k].shift);
      const uint32_t i = m - q * a.rank[k].extent;
      offIn += i * a.rank[k].strideIn;
      offOut += i * a.rank[k].strideOut;
      m = q;
    }
  };
  ranks(0);
  static_assert(CUTT_PACKED_RANKS == 12, "three steps of four ranks");
  if (a.n > 4) {
    ranks(4);
    if (a.n > 8) ranks(8);
  }
}

}  // namespace cutt

#endif  // CUTT_PACKED_WALK_H
