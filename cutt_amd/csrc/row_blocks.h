/*
 * row_blocks.h - device code shared by the row-gathering kernel and the kernel that replays its
 * address stream: which output elements a workgroup writes and where their rows lie in the input.
 */
#ifndef CUTT_ROW_BLOCKS_H
#define CUTT_ROW_BLOCKS_H

#include <hip/hip_runtime.h>

#include "hip_layer.h"
#include "mbar_decode.h"

namespace cutt {

constexpr int kRowThreads = 256;
constexpr int kRowElems = CUTT_ROW_BLOCK / kRowThreads;  // elements per lane

struct RowBlock {
  int64_t first;        // output element of the block's slot 0 (negative in block 0 of a buffer off the line grid)
  uint32_t lo, hi;      // slots [lo, hi) hold elements of the tensor
  uint32_t row0, col0;  // row and column of slot lo
  uint32_t rows;        // rows the block meets
};

// Block of this workgroup when the output starts `shift` elements past a 128-byte line; false if it lies beyond the tensor.
__device__ __forceinline__ bool locateRows(const cuttHipRowArgs& a, uint32_t shift, RowBlock& b) {
  uint32_t l = blockIdx.x;
  if (a.xcdGroup) {
    const uint32_t g = (uint32_t)a.xcdGroup - 1, q = l >> 3;
    l = ((((q >> g) << 3) + (l & 7)) << g) + (q & ((1u << g) - 1));
  }
  b.first = (int64_t)l * CUTT_ROW_BLOCK - shift;
  if (b.first >= (int64_t)a.volume) return false;
  b.lo = b.first < 0 ? shift : 0u;
  b.hi = (uint32_t)min((int64_t)CUTT_ROW_BLOCK, (int64_t)a.volume - b.first);
  const uint32_t e0 = (uint32_t)(b.first + b.lo);
  b.row0 = e0 / a.rowLen;
  b.col0 = e0 - b.row0 * a.rowLen;
  b.rows = fastDivide(b.col0 + (b.hi - b.lo) - 1, a.rowDiv.mul, a.rowDiv.shift, a.rowDiv.add) + 1;
  return true;
}

// Input offset of output row o.
__device__ __forceinline__ uint32_t rowInputOffset(const cuttHipRowArgs& a, uint32_t o) {
  uint32_t off = 0;
  for (int k = 0; k + 1 < a.n; k++) {
    const cuttHipRowRank d = a.rank[k];
    const uint32_t q = fastDivide(o, d.mul, d.ctl & 0xff, d.ctl >> 8);
    off += (o - q * d.extent) * d.stride;
    o = q;
  }
  return off + o * a.rank[a.n - 1].stride;
}

}  // namespace cutt

#endif  // CUTT_ROW_BLOCKS_H
