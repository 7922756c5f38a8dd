/*
 * line_windows.h - device code shared by the Tiled kernel with line-aligned stores and the kernel that
 * replays its address stream: the part of the tensor a workgroup handles.
 */
#ifndef CUTT_LINE_WINDOWS_H
#define CUTT_LINE_WINDOWS_H

#include <hip/hip_runtime.h>

#include "hip_layer.h"
#include "tile_order.h"

namespace cutt {

constexpr int kWindow = kTile;  // elements of an output run that one tile row stores

// Elements per 128-byte line, input rows along Mk that a tile may need, and the lanes of its workgroup.
template <typename T>
constexpr int kLineElems = 128 / (int)sizeof(T);
template <typename T>
constexpr int kLineRows = kWindow + kLineElems<T> - 1;
template <typename T>
constexpr int kLineMaxWidth = sizeof(T) == 8 ? CUTT_LINE_WIDTH : 2 * CUTT_LINE_WIDTH;

struct LineTile {
  uint32_t m0, width;   // columns [m0, m0 + width) along Mm
  uint32_t pitch;       // elements between tile rows in LDS (odd: a column read meets every bank once)
  int32_t kWin;         // the window of a row that starts s elements past a line is [kWin - s, kWin - s + 64)
  int32_t kLo;          // first of the `rows` rows along Mk that some window of the tile needs
  uint32_t rows;        // 0: every window lies beyond the ends of the runs
};

// `outWord` is the element address of the Mbar position's first output element, counted from a line boundary.
template <typename T>
__device__ __forceinline__ LineTile lineTile(const cuttHipTiledArgs& a, uint32_t tm, uint32_t tk, uint32_t outWord) {
  constexpr uint32_t LE = kLineElems<T>;
  LineTile t;
  t.m0 = tm * (uint32_t)a.lineWidth;
  t.width = min((uint32_t)a.lineWidth, (uint32_t)a.volMm - t.m0);
  t.pitch = (uint32_t)a.lineWidth | 1u;
  t.kWin = (int32_t)(tk * kWindow);
  // The rows start s = s0 + j g (mod LE) elements past a line, g = the largest power of two that divides every
  // stride of the Mm axis: the windows together cover [kWin - sMax, kWin - sMin + 64).
  uint32_t bits = LE;
  if (a.rowsM.n > 0)
    for (int k = 0; k < a.rowsM.n; k++) bits |= a.rowsM.stride[k];
  else
    bits |= a.strideOutM;
  const uint32_t g = bits & (0u - bits);
  const uint32_t sMin = outWord & (g - 1), sMax = sMin + (LE - g);
  t.kLo = max(t.kWin - (int32_t)sMax, 0);
  const int32_t hi = min(t.kWin - (int32_t)sMin + kWindow, (int32_t)a.volMk);
  t.rows = hi > t.kLo ? (uint32_t)(hi - t.kLo) : 0u;
  return t;
}

// Row k of the Mk axis -> input offset, row m of the Mm axis -> output offset.
template <bool FUSED>
__device__ __forceinline__ uint32_t lineRowIn(const cuttHipTiledArgs& a, uint32_t k) {
  return FUSED && a.rowsK.n > 0 ? rowOffset(a.rowsK, k) : k * a.strideInK;
}
template <bool FUSED>
__device__ __forceinline__ uint32_t lineRowOut(const cuttHipTiledArgs& a, uint32_t m) {
  return FUSED && a.rowsM.n > 0 ? rowOffset(a.rowsM, m) : m * a.strideOutM;
}

// The tile's input elements are read in order of rows and columns: element p (< rows * width) is column c of row r;
// `widthDiv` divides by the width of a whole tile.
__device__ __forceinline__ void lineElem(const cuttHipTiledArgs& a, const cuttHipDivisor& widthDiv, const LineTile& t, uint32_t p, uint32_t& r, uint32_t& c) {
  // (the last tile along Mm may be narrower than the constants' divisor)
  r = t.width == (uint32_t)a.lineWidth ? fastDivide(p, widthDiv.mul, widthDiv.shift, widthDiv.add) : p / t.width;
  c = p - r * t.width;
}

}  // namespace cutt

#endif  // CUTT_LINE_WINDOWS_H
