/*
 * tile_walk.h - which tile a workgroup takes, for the numberings that are decoded without a branch or a division by a variable
 * (hip_layer.h: cuttHipTileWalk), and how the XCDs share the workgroups.  Plain integer code: the kernels compile it for the
 * device, tests for the host.
 */
#ifndef CUTT_TILE_WALK_H
#define CUTT_TILE_WALK_H

#include <cstdint>
#include <type_traits>

#include "hip_layer.h"

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define CUTT_DEVICE __device__ __forceinline__
#else
#define CUTT_DEVICE inline
#endif

namespace cutt {

constexpr uint32_t kNumXcd = 8;

// Workgroup index -> logical position (cuttHipTiledArgs.xcdChunk, xcdGroup).
CUTT_DEVICE uint32_t xcdPosition(uint32_t bid, uint32_t chunk, uint32_t group) {
  const uint32_t q = bid / kNumXcd, x = bid % kNumXcd;
  if (group) {
    const uint32_t g = group - 1;
    return ((((q >> g) * kNumXcd) + x) << g) + (q & ((1u << g) - 1));
  }
  return chunk ? x * chunk + q : bid;
}

CUTT_DEVICE uint32_t walkMulHi(uint32_t a, uint32_t b) {
#ifdef __HIPCC__
  return __umulhi(a, b);
#else
  return (uint32_t)(((uint64_t)a * b) >> 32);
#endif
}

// n / d for n < 2^31 (constants of cuttHipTileWalk).
CUTT_DEVICE uint32_t walkDivide(uint32_t n, uint32_t mul, uint32_t shift) { return walkMulHi(2 * n, mul) >> shift; }

// Workgroup index -> position: chunk and bits 15 and up of `shifts` as in cuttHipTileWalk.
CUTT_DEVICE uint32_t walkPosition(uint32_t bid, uint32_t chunk, uint32_t shifts) {
  const uint32_t xs = (shifts >> 15) & 3, g = ((shifts >> 17) - 1) & 31;  // 3: XCD b % 8 has positions of its own; in groups of 2^g (31: no groups)
  const uint32_t q = bid >> xs;
  return (bid & ((1u << xs) - 1)) * chunk + (q & ((1u << g) - 1)) + (((q >> g) << g) << 3);
}

// What every workgroup of a walk (cuttHipTileWalk) decodes its index with.
struct WalkHead {
  uint32_t chunk, superM, stripMul, fullMul, lastMul, shifts;
};

// The Mbar part of a walk for launches without one.
struct NoMbar {};

// Workgroup `bid` -> tile and offsets of its Mbar position, as tile_order.h's locateTile, for a numbering in walk form:
// multiply-high divisions on the scalar unit, whose constants are all there from the start (in registers, or in memory at
// addresses that are), and no branch but the test for the end - where locateTile waits for the order's number, its
// parameters, two to seven divisions by variables and the Mbar table one after the other.
template <typename MB>
CUTT_DEVICE bool walkTile(uint32_t bid, const WalkHead& h, const MB& mb, uint32_t tilesM, uint32_t tilesK, uint32_t& tm, uint32_t& tk, uint32_t& offIn, uint32_t& offOut) {
  constexpr bool kMbar = !std::is_same_v<MB, NoMbar>;
  uint32_t l = walkPosition(bid, h.chunk, h.shifts), m = 0, perStrip = tilesK;
  const uint32_t tiles = tilesM * tilesK;
  offIn = offOut = 0;
  if constexpr (kMbar) {
    if (l >= tiles * mb.volMbar) return false;
    m = walkDivide(l, mb.outerMul, mb.shifts & 31);
    l -= m * tiles;
    perStrip *= mb.stripMbar;
  } else {
    if (l >= tiles) return false;
  }
  const uint32_t first = walkDivide(l, h.stripMul, h.shifts & 31) * h.superM;  // the strip's first tile along Mm
  const uint32_t width = h.superM < tilesM - first ? h.superM : tilesM - first;
  const bool full = width == h.superM;
  l -= first * perStrip;  // (all strips before are full ones)
  if constexpr (kMbar) {
    const uint32_t mi = walkDivide(l, full ? mb.innerMul[0] : mb.innerMul[1], (full ? mb.shifts >> 5 : mb.shifts >> 10) & 31);
    l -= mi * (width * tilesK);
    m += mi;
  }
  tk = walkDivide(l, full ? h.fullMul : h.lastMul, (full ? h.shifts >> 5 : h.shifts >> 10) & 31);
  tm = first + (l - tk * width);
  if constexpr (kMbar) {
    auto ranks = [&](int from) __attribute__((always_inline)) {
#pragma unroll
      for (int k = from; k < from + 4; k++) {  // (unused ranks have zeros everywhere)
        const uint32_t q = walkDivide(m, mb.rank[k].mul, mb.rank[k].shift);
        const uint32_t i = m - q * mb.rank[k].extent;
        offIn += i * mb.rank[k].strideIn;
        offOut += i * mb.rank[k].strideOut;
        m = q;
      }
    };
    ranks(0);
    static_assert(CUTT_WALK_RANKS == 8, "two steps of four ranks");
    if (mb.n > 4) ranks(4);
  }
  return true;
}

// Offset of row `i` of a tile axis, per lane.
CUTT_DEVICE uint32_t walkRowOffset(const cuttHipWalkRows& r, uint32_t i) {
  uint32_t q = walkDivide(i, r.mul[0], r.shift[0]);
  uint32_t off = (i - q * r.extent[0]) * r.stride[0];
  if (r.n > 2) {
#pragma unroll
    for (int k = 1; k < 3; k++) {
      const uint32_t q2 = walkDivide(q, r.mul[k], r.shift[k]);
      off += (q - q2 * r.extent[k]) * r.stride[k];
      q = q2;
    }
    return off + q * r.stride[3];
  }
  return off + q * r.stride[1];
}

}  // namespace cutt

#endif  // CUTT_TILE_WALK_H
