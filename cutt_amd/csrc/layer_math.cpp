/*
 * layer_math.cpp - the part of the C-ABI layer (hip_layer.h) that is plain arithmetic: division
 * constants, the Mbar table's derived fields, LDS bytes and register counts of the packed kernel.
 * No HIP header and no runtime call, so the host planner can be linked and tested without the
 * device side (the kernels check their arguments with the same functions).
 */
#include "hip_layer.h"

#include <cstdint>
#include <cstring>

extern "C" cuttHipDivisor cuttHipMakeDivisor(uint32_t d) {
  cuttHipDivisor dv = {0u, 0u, 1u};  // d <= 1: n / 1
  if (d >= 2) {
    uint32_t shift = 0;
    while ((1ull << (shift + 1)) < d) shift++;  // ceil(log2 d) - 1
    const uint64_t pow2 = 1ull << (32 + shift);
    dv.mul = (uint32_t)((pow2 + d - 1) / d);
    dv.shift = shift;
    dv.add = 0;
  }
  return dv;
}

extern "C" uint32_t cuttHipDivide(uint32_t n, cuttHipDivisor dv) {
  const uint32_t hi = (uint32_t)(((uint64_t)n * dv.mul) >> 32);
  return (hi + n * dv.add) >> dv.shift;
}

extern "C" int cuttHipFinishMbar(cuttHipMbar* mb) {
  if (!mb || mb->n < 0 || mb->n > CUTT_MAX_RANK) return -1;
  uint64_t below = 1;
  for (int k = 0; k < CUTT_MAX_RANK; k++) {
    cuttHipMbarDim& d = mb->d[k];
    if (k >= mb->n) {
      d.belowMul = d.extentMul = d.ctl = 0;  // quotients 0: no contribution
      continue;
    }
    if (d.extent == 0 || below * d.extent >= (1ull << 31)) return -1;
    const cuttHipDivisor b = cuttHipMakeDivisor((uint32_t)below), e = cuttHipMakeDivisor(d.extent);
    d.belowMul = b.mul;
    d.extentMul = e.mul;
    d.ctl = b.shift | (e.shift << 8) | (b.add << 16) | (e.add << 17);
    below *= d.extent;
  }
  return 0;
}

extern "C" uint64_t cuttHipRowGrid(const cuttHipRowArgs* a) {
  uint64_t blocks = ((uint64_t)a->volume + 128 / a->elemSize - 1 + CUTT_ROW_BLOCK - 1) / CUTT_ROW_BLOCK;
  if (a->xcdGroup) {
    const uint64_t unit = 8ull << (a->xcdGroup - 1);  // a group per XCD
    blocks = (blocks + unit - 1) / unit * unit;
  }
  return blocks <= 0x7fffffffull && blocks * 256 <= CUTT_HIP_MAX_GRID_LANES ? blocks : 0;
}

static int finishTileDigits(cuttHipTileDigits* dg, const cuttHipMbar* mb);

extern "C" int cuttHipFinishTileDigits(cuttHipTileDigits* dg, const cuttHipMbar* mb) {
  if (!dg || !mb) return -1;
  finishTileDigits(dg, mb);
  if (!dg->lanes) {  // not decodable in one step: no half-filled table
    dg->total = 0;
    for (int i = 0; i < CUTT_MAX_TILE_DIGITS; i++) dg->lane[i] = cuttHipDigitLane{0u, 0u, 0u, 1u, 0u, 0u, 0u, 0u};
  }
  return 0;
}

static int finishTileDigits(cuttHipTileDigits* dg, const cuttHipMbar* mb) {
  dg->lanes = 0;
  dg->total = 0;
  for (int i = 0; i < CUTT_MAX_TILE_DIGITS; i++) dg->lane[i] = cuttHipDigitLane{0u, 0u, 0u, 1u, 0u, 0u, 0u, 0u};
  if (dg->n < 1 || dg->n > CUTT_MAX_TILE_DIGITS || mb->n < 0 || mb->n > CUTT_MAX_RANK) return 0;
  uint64_t below = 1, mbarDigits = 1, volMbar = 1;
  for (int k = 0; k < mb->n; k++) volMbar *= mb->d[k].extent;
  for (int i = 0; i < dg->n; i++) {
    const cuttHipTileDigit& d = dg->d[i];
    cuttHipDigitLane& l = dg->lane[i];
    if (d.radix < 1 || d.which > 2 || below * d.radix >= (1ull << 31)) return 0;
    const cuttHipDivisor b = cuttHipMakeDivisor((uint32_t)below), e = cuttHipMakeDivisor(d.radix);
    l.belowMul = b.mul;
    l.radixMul = e.mul;
    l.ctl = b.shift | (e.shift << 8) | (b.add << 16) | (e.add << 17);
    l.radix = d.radix;
    if (d.which == 0) l.stepM = d.weight;
    if (d.which == 1) l.stepK = d.weight;
    if (d.which == 2 && d.radix > 1) {
      // the Mbar rank the digit counts in; it must not reach into the next one
      uint64_t rankBelow = 1;
      int k = 0;
      for (; k < mb->n; rankBelow *= mb->d[k].extent, k++)
        if ((uint64_t)d.weight >= rankBelow && (uint64_t)d.weight < rankBelow * mb->d[k].extent) break;
      if (k == mb->n || (uint64_t)d.weight % rankBelow != 0) return 0;
      const uint64_t u = (uint64_t)d.weight / rankBelow;
      if ((uint64_t)mb->d[k].extent % (u * d.radix) != 0) return 0;
      mbarDigits *= d.radix;
      if (u * mb->d[k].strideIn > 0xffffffffull || u * mb->d[k].strideOut > 0xffffffffull) return 0;
      l.strideIn = (uint32_t)(u * mb->d[k].strideIn);
      l.strideOut = (uint32_t)(u * mb->d[k].strideOut);
    }
    below *= d.radix;
  }
  // (no Mbar position beyond the last one: the kernels do not rebuild the position to check it)
  if (mbarDigits != volMbar) return 0;
  dg->total = (uint32_t)below;
  dg->lanes = 1;
  return 0;
}

namespace {
// mulhi32(2 n, mul) >> shift == n / d for n < 2^31 (d >= 1).
void walkDivisor(uint64_t d, uint32_t& mul, uint32_t& shift) {
  shift = 0;
  while ((1ull << shift) < d) shift++;
  mul = (uint32_t)(((1ull << (31 + shift)) + d - 1) / d);
}

void walkRows(const cuttHipRowRadix& rr, uint32_t stride, cuttHipWalkRows& w) {
  w.n = rr.n > 0 ? (uint32_t)rr.n : 1u;
  w.stride[0] = stride;
  for (int k = 0; k < rr.n; k++) {
    w.stride[k] = rr.stride[k];
    if (k + 1 == rr.n) break;
    w.extent[k] = rr.extent[k];
    walkDivisor(rr.extent[k], w.mul[k], w.shift[k]);
  }
}
}  // namespace

extern "C" void cuttHipFinishTileWalk(cuttHipTiledArgs* a) {
  cuttHipTileWalk& w = a->walk;
  std::memset(&w, 0, sizeof(w));
  const uint64_t tilesM = (uint64_t)a->tilesM, tilesK = (uint64_t)a->tilesK, volMbar = (uint64_t)a->volMbar;
  const bool strips = (a->order == 3 || a->order == 5) && a->superK >= tilesK;
  if (a->tilesM < 1 || a->tilesK < 1 || a->volMbar < 1 || (!strips && a->order != 1 && a->order != 2)) return;
  if (a->mbar.n < 0 || a->mbar.n > CUTT_WALK_RANKS || a->rowsK.n < 0 || a->rowsK.n > CUTT_MAX_TILE_SET || a->rowsM.n < 0 || a->rowsM.n > CUTT_MAX_TILE_SET) return;
  // (every division is of a number below 2^31; two of the factors are)
  const uint64_t tiles = tilesM * tilesK;
  if (tiles > 0x7fffffffull || tiles * volMbar > 0x7fffffffull) return;
  const uint64_t total = tiles * volMbar;
  w.superM = a->order == 1 ? (uint32_t)tilesM : (a->order == 2 ? 1u : (a->superM < tilesM ? a->superM : (uint32_t)tilesM));
  if (w.superM < 1) return;
  const uint64_t stripMbar = a->order == 5 ? volMbar : 1, last = tilesM % w.superM;
  uint32_t strip = 0, full = 0, lastShift = 0;
  walkDivisor(w.superM * tilesK * stripMbar, w.stripMul, strip);
  walkDivisor(w.superM, w.fullMul, full);
  walkDivisor(last ? last : 1, w.lastMul, lastShift);
  const bool perXcd = a->xcdChunk != 0 || a->xcdGroup > 0;
  if (a->xcdGroup < 0 || a->xcdGroup > 20) return;
  if (a->xcdGroup > 0) {
    w.chunk = 1u << (a->xcdGroup - 1);
    const uint64_t unit = 8ull * w.chunk, blocks = (total + unit - 1) / unit * unit;
    if (blocks > 0x7fffffffull) return;
    w.blocks = (uint32_t)blocks;
  } else {
    w.chunk = perXcd ? (uint32_t)((total + 7) / 8) : 0u;
    w.blocks = perXcd ? 8 * w.chunk : (uint32_t)total;
  }
  w.shifts = strip | full << 5 | lastShift << 10 | (perXcd ? 3u : 0u) << 15 | (uint32_t)a->xcdGroup << 17;
  w.kind = volMbar > 1 ? 2 : 1;
  if (w.kind == 2) {
    cuttHipWalkMbar& b = w.mbar;
    b.volMbar = (uint32_t)volMbar;
    b.stripMbar = (uint32_t)stripMbar;
    uint32_t outer = 0, inner[2] = {0, 0};
    if (a->order == 5) {
      walkDivisor(w.superM * tilesK, b.innerMul[0], inner[0]);
      walkDivisor((last ? last : 1) * tilesK, b.innerMul[1], inner[1]);
    } else {
      walkDivisor(tiles, b.outerMul, outer);
    }
    b.shifts = outer | inner[0] << 5 | inner[1] << 10;
    b.n = (uint32_t)a->mbar.n;
    for (int k = 0; k < a->mbar.n; k++) {
      cuttHipWalkRank& r = b.rank[k];
      r.strideIn = a->mbar.d[k].strideIn;
      r.strideOut = a->mbar.d[k].strideOut;
      if (k + 1 == a->mbar.n) break;
      r.extent = a->mbar.d[k].extent;
      walkDivisor(r.extent, r.mul, r.shift);
    }
  }
  walkRows(a->rowsK, a->strideInK, w.rowsK);
  walkRows(a->rowsM, a->strideOutM, w.rowsM);
}

extern "C" int cuttHipTiledTakesWalk(const cuttHipTiledArgs* a) {
  return a->walk.kind != 0 && a->lineWidth == 0 && (a->wide || (!a->grouped && !a->paced)) ? 1 : 0;
}

extern "C" void cuttHipFinishPackedWalk(cuttHipPackedArgs* a) {
  cuttHipPackedWalk& o = a->walk;
  std::memset(&o, 0, sizeof(o));
  const long long numbers = cuttHipPackedItemNumbers(a);
  // (a loop over blocks of few elements per lane is slower this way: (5,4,1374779)/(1,0,2), 8 bytes, one element per lane, 212 -> 254 us)
  // Nor does it help workgroups of 13-16 waves with 8-byte elements: 36 plans of 250-1600 MB per buffer 1.004 in
  // the mean, 0.975 ... 1.024, (1544,426,76,4)/(2,0,1,3) 556 -> 571 us.
  if (a->itemsPerBlock > 1 && (a->elemsPerThread < CUTT_PACKED_LOOP_ELEMS || (a->elemSize == 8 && a->numThreads > 768))) return;
  if (a->itemsPerBlock < 1 || a->wideOffsets || a->mbar.n < 0 || a->mbar.n > CUTT_PACKED_RANKS || a->xcdGroup < 0 || a->xcdGroup > 20 || numbers < 1) return;
  const unsigned long long per = (unsigned long long)a->itemsPerBlock, groups = ((unsigned long long)numbers + per - 1) / per;
  unsigned long long blocks = groups;
  o.perGroup = (uint32_t)per;
  o.volMbar = (uint32_t)a->volMbar;
  o.first = o.stepN = o.mulM = 1;
  if (a->xcdGroup > 0) {
    o.chunk = 1u << (a->xcdGroup - 1);
    blocks = (blocks + 8ull * o.chunk - 1) / (8ull * o.chunk) * (8ull * o.chunk);
  } else if (a->xcdChunk) {
    o.chunk = a->xcdChunk;
    if (8ull * o.chunk < blocks) return;
    blocks = 8ull * o.chunk;
  }
  // (the divisions are of numbers below 2^31; those of padding workgroups only have to stay below 2^32)
  if (blocks > 0x7fffffffull || blocks * per > 0xffffffffull) return;
  o.items = (uint32_t)numbers;
  if (a->itemOrder == 1) {  // the workgroup keeps its slabs
    o.items = (uint32_t)groups;
    o.stepN = 0;
    o.mulM = (uint32_t)per;
    o.stepM = 1;
  } else if (a->itemOrder == 2) {  // the workgroups of a chunk take its blocks in turn
    const bool chunks = a->xcdChunk && !a->xcdGroup;
    o.stepN = chunks ? o.chunk : (uint32_t)blocks;
    if (chunks) o.chunk *= o.perGroup;
  } else {
    o.first = (uint32_t)per;
  }
  uint32_t shift[2];
  for (int i = 0; i < 2; i++) {
    const cuttHipSplitRank& s = a->split[i];
    o.num[i] = (uint32_t)s.numSplit;
    walkDivisor(o.num[i], o.mul[i], shift[i]);
    o.slab[i] = cuttHipPackedWalkSlab{(uint32_t)s.slabRem, (uint32_t)s.slabFloor * s.strideIn, (uint32_t)s.slabFloor * s.strideOut, s.strideIn, s.strideOut};
  }
  o.shifts = shift[0] | shift[1] << 5 | (a->xcdGroup > 0 || a->xcdChunk ? 3u : 0u) << 15 | (uint32_t)a->xcdGroup << 17;
  o.padThreads = (uint32_t)a->padShift | (uint32_t)a->numThreads << 8;
  o.n = (uint32_t)a->mbar.n;
  for (int k = 0; k < a->mbar.n; k++) {
    cuttHipWalkRank& r = o.rank[k];
    r.strideIn = a->mbar.d[k].strideIn;
    r.strideOut = a->mbar.d[k].strideOut;
    if (k + 1 == a->mbar.n) break;
    r.extent = a->mbar.d[k].extent;
    walkDivisor(r.extent, r.mul, r.shift);
  }
  const unsigned char* const first = (const unsigned char*)a->cls[0].rowIn;
  for (int c = 0; c < 4; c++) {
    if (((c & 1) && a->split[0].slabRem == 0) || ((c & 2) && a->split[1].slabRem == 0)) continue;
    const cuttHipPackedClass& k = a->cls[c];
    const void* const table[3] = {k.rowIn, k.rowOut, k.shIdx};
    uint32_t at[3];
    for (int i = 0; i < 3; i++) {
      const uintptr_t d = (uintptr_t)table[i] - (uintptr_t)first;
      if (!table[i] || d > 0x7fffffffu) return;  // (one piece of memory, class 0 first)
      at[i] = (uint32_t)d;
    }
    if (k.vol < 1 || k.inCont < 1 || k.outCont < 1) return;
    cuttHipPackedWalkClass& w = o.cls[c];
    uint32_t inShift = 0, outShift = 0;
    walkDivisor((uint64_t)k.inCont, w.inMul, inShift);
    walkDivisor((uint64_t)k.outCont, w.outMul, outShift);
    w.last = (uint32_t)k.vol - 1;
    w.inCont = (uint32_t)k.inCont;
    w.outCont = (uint32_t)k.outCont;
    w.shifts = inShift | outShift << 5;
    w.rowIn = at[0];
    w.rowOut = at[1];
    w.shIdx = at[2];
  }
  o.blocks = (uint32_t)blocks;
}

extern "C" long long cuttHipPackedItemNumbers(const cuttHipPackedArgs* a) {
  const unsigned long long slabs = (unsigned long long)a->split[0].numSplit * (unsigned long long)a->split[1].numSplit;
  unsigned long long n = (unsigned long long)a->volMbar * slabs;
  if (a->itemOrder == 1) {
    const unsigned long long ipb = (unsigned long long)a->itemsPerBlock;
    n = (((unsigned long long)a->volMbar + ipb - 1) / ipb) * slabs * ipb;
  }
  return n > 0x7fffffffull ? -1 : (long long)n;
}

extern "C" int cuttHipDecodeItem(const cuttHipPackedArgs* a, uint32_t w, uint32_t* m, uint32_t* s0, uint32_t* s1, int* cls) {
  const uint32_t ns0 = (uint32_t)a->split[0].numSplit, ns1 = (uint32_t)a->split[1].numSplit;
  uint32_t slab = w, mi = 0, ipb = 1;
  if (a->itemOrder == 1) {
    ipb = (uint32_t)a->itemsPerBlock;
    slab = w / ipb;
    mi = w - slab * ipb;
  }
  const uint32_t t = cuttHipDivide(slab, a->split[0].div);
  *s0 = slab - t * ns0;
  const uint32_t mb = cuttHipDivide(t, a->split[1].div);
  *s1 = t - mb * ns1;
  *m = mb * ipb + mi;
  *cls = (*s0 < (uint32_t)a->split[0].slabRem ? 1 : 0) + (*s1 < (uint32_t)a->split[1].slabRem ? 2 : 0);
  return *m < (uint32_t)a->volMbar;
}

extern "C" size_t cuttHipPackedLdsBytes(const cuttHipPackedArgs* a) {
  const size_t b = (size_t)a->ldsElems * a->elemSize;
  return (b + 15) & ~(size_t)15;
}

// Registers per lane of packedKernel<T, E, *, WIDE> as compiled for gfx950 (the cache policy does
// not change the count).  Rows: E = 1, 2, 4, 8, 16.
extern "C" int cuttHipPackedRegsPerLane(int elemSize, int elemsPerThread, int wideOffsets) {
  static const int narrow4[5] = {15, 23, 38, 68, 124}, wide4[5] = {17, 27, 40, 72, 128};
  static const int narrow8[5] = {15, 25, 43, 73, 0}, wide8[5] = {18, 28, 48, 88, 0};
  int row = 0;
  while (row < 5 && (1 << row) != elemsPerThread) row++;
  if (row == 5 || (elemSize != 4 && elemSize != 8)) return 0;
  return elemSize == 4 ? (wideOffsets ? wide4 : narrow4)[row] : (wideOffsets ? wide8 : narrow8)[row];
}

extern "C" int cuttHipLinesMaxWidth(int elemSize) { return elemSize == 8 ? CUTT_LINE_WIDTH : 2 * CUTT_LINE_WIDTH; }

// 8-byte elements and wide tiles of 4-byte ones take 512 lanes.
extern "C" int cuttHipLinesThreads(int elemSize, int tileWidth) { return elemSize == 8 || tileWidth > CUTT_LINE_WIDTH ? 512 : 256; }

extern "C" size_t cuttHipLinesLdsBytes(int elemSize, int tileWidth) {
  return (size_t)(64 + 128 / elemSize - 1) * (size_t)(tileWidth | 1) * (size_t)elemSize;
}
