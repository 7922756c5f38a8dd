/*
 * kernels.hip - transpose kernels for gfx950 (64-lane wavefronts) and their
 * launch functions.
 *
 * Four data paths, matching the reference's method set
 * (reference src/cuttkernel.cu:38-118 Tiled, :123-222 Packed, :230-347
 * PackedSplit, :356-426 TiledCopy), written for CDNA4 rather than translated:
 *
 *  - every kernel moves opaque 4- or 8-byte words (uint32_t / uint64_t), one
 *    word per lane per access, so a wavefront touches 256 or 512 contiguous
 *    bytes per instruction when the run is long enough;
 *  - the per-rank decomposition of a workgroup's Mbar position is wave-uniform:
 *    lane k owns rank k, divides by precomputed multiply-high constants and the
 *    wavefront sums the contributions with DPP adds (mbar_decode.h);
 *  - Tiled stages a 64x64 tile in LDS padded to 65 columns (conflict-free for
 *    both 4- and 8-byte words); each lane keeps 16 loads in flight; edges are handled by
 *    clamping indices, not by branches, so the memory instructions stay back to back;
 *  - Packed/PackedSplit take their index remap from tables the planner precomputed in device
 *    memory (one input offset per contiguous input run, one output offset per contiguous output
 *    run, an LDS gather slot per staged element); a workgroup takes one block (packedOnceKernel), or it derives
 *    its lanes' offsets once and keeps them in registers while it loops over its blocks, so the loop body is load, LDS
 *    write, LDS read, store (packedLoopKernel; packedKernel where the blocks cannot be decoded as a walk);
 *    the LDS buffer is skewed by one slot per 2^padShift to break power-of-two bank strides;
 *  - workgroups are short-lived and small (a tile, or a few Mbar positions),
 *    thousands are in flight: on this chip that streams faster than a
 *    persistent grid-stride loop.
 *
 * All offsets are unsigned 32-bit element offsets from the pointers of the launch (one launch
 * spans fewer than 2^32 elements on either side - a larger tensor comes in pieces -; every true
 * offset is below that span, so the modular sums are exact); the packed kernel turns them into
 * 32-bit byte offsets from a wave-uniform base when the span is below 4 GB.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <tuple>
#include <type_traits>

#include "hip_layer.h"
#include "line_windows.h"
#include "mbar_decode.h"
#include "packed_items.h"
#include "packed_walk.h"
#include "row_blocks.h"
#include "tile_order.h"

using namespace cutt;

namespace {

// Cache policy of the global accesses, a kernel template parameter NT: bit 0 = non-temporal
// (streaming) loads, bit 1 = non-temporal stores.  The input is read once, so streaming loads keep
// the L2 free for the output lines that neighbouring workgroups still have to complete; streaming
// stores pay off only when every written run covers whole 128-byte lines.
template <int NT, typename T>
__device__ __forceinline__ T ldg(const T* p) {
  if constexpr (NT & 1) return __builtin_nontemporal_load(p);
  else return *p;
}
template <int NT, typename T>
__device__ __forceinline__ void stg(T* p, T v) {
  if constexpr (NT & 2) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// Blocks the wave until its outstanding global loads have returned and its stores have been
// acknowledged (the vector memory counter reaches zero); also a barrier for the compiler.
__device__ __forceinline__ void waitForGlobalAccesses() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// ---------------------------------------------------------------------------
// Tiled: 64x64 tile through padded LDS.
// ---------------------------------------------------------------------------
// GROUPED: the four row groups of a lane go one after the other - request 4 rows, wait, stage them,
// request the next 4; store 4 rows, wait, store the next 4 - instead of all 16 rows at once.  That
// quarters what a wave has in flight.  When tile rows start off the 128-byte grid (4-byte
// elements, large tensors) it is 3-11 % faster: the neighbouring tiles' requests for a shared line
// then arrive while the line is still in the L2.  On aligned or cache-resident tensors it is up to
// 10 % slower, so the planner decides (cuttHipTiledArgs.grouped).
//
// FUSED: a tile axis runs over several fused ranks (the ranks that lead the input on the Mm side, the
// ranks that lead the output on the Mk side), so the rows of a tile are not equally far apart.  Lane l
// derives the offset of row l of either axis with a short mixed-radix decode (tileRowOffsets) and the
// wave picks a row's offset out of that lane; the elements of a row are contiguous as before.
template <typename T, int NT, bool FUSED, typename Args>
__device__ __forceinline__ void moveTile(const TileLanes& t, const Args& a, const T* __restrict__ in, T* __restrict__ out) {
  __shared__ T tile[kTile][kTile + 1];
  const uint32_t wave = threadIdx.x >> 6;

  // One straight piece of code per number of row groups (4 for a whole tile, fewer at an edge): all loads go out back to back, where tests
  // between the groups would keep them apart or even, in a function like this one, make them wait for each other (tiledKernel).  WHOLE: all
  // 64 rows are there, no index needs clamping.
  auto read = [&](auto groups, auto whole) __attribute__((always_inline)) {  // lanes run along the input-contiguous axis (Mm), rows along Mk
    constexpr int kRows = decltype(groups)::value * kGroupRows;
    const uint32_t lastRow = decltype(whole)::value ? kTile - 1u : t.wK;
    T v[kRows];
#pragma unroll
    for (int j = 0; j < kRows; j++) v[j] = ldg<NT>(in + tileReadElem<FUSED>(t, a, wave, j, lastRow));
#pragma unroll
    for (int j = 0; j < kRows; j++) tile[min(wave + kWaves * j, lastRow)][t.cx] = v[j];
  };
  auto write = [&](auto groups, auto whole) __attribute__((always_inline)) {  // lanes run along the output-contiguous axis (Mk), rows along Mm
    constexpr int kRows = decltype(groups)::value * kGroupRows;
    const uint32_t lastRow = decltype(whole)::value ? kTile - 1u : t.wM;
    T v[kRows];
#pragma unroll
    for (int j = 0; j < kRows; j++) v[j] = tile[t.ck][min(wave + kWaves * j, lastRow)];
#pragma unroll
    for (int j = 0; j < kRows; j++) stg<NT>(out + tileWriteElem<FUSED>(t, a, wave, j, lastRow), v[j]);
  };
  auto byGroups = [](uint32_t lastRow, auto&& f) __attribute__((always_inline)) {
    if (lastRow == kTile - 1) f(std::integral_constant<int, 4>{}, std::true_type{});
    else if (lastRow >= 48) f(std::integral_constant<int, 4>{}, std::false_type{});
    else if (lastRow >= 32) f(std::integral_constant<int, 3>{}, std::false_type{});
    else if (lastRow >= 16) f(std::integral_constant<int, 2>{}, std::false_type{});
    else f(std::integral_constant<int, 1>{}, std::false_type{});
  };
  static_assert(kRowGroups == 4 && kGroupRows * kWaves == 16, "row groups of 16 tile rows");
  byGroups(t.wK, read);
  __syncthreads();
  byGroups(t.wM, write);
}

// The same with a test for every row in one piece of code, whose loads the compiler makes wait for each other.  For 4-byte elements with
// non-temporal stores in numberings that have no walk (address bits, mostly): (1024,64,1024)/(2,1,0) 103.5 us with paced loads, 103.1 here,
// (1024,16,1024,12)/(2,1,0,3) 278.2 / 275.4, (256,1024,512)/(2,1,0) 197.8 / 195.4; eight such tensors 0.4 % in the mean.
template <typename T, int NT, bool FUSED, typename Args>
__device__ __forceinline__ void moveTileTested(const TileLanes& t, const Args& a, const T* __restrict__ in, T* __restrict__ out) {
  __shared__ T tile[kTile][kTile + 1];
  const uint32_t wave = threadIdx.x >> 6;
  T v[kTileRows];
#pragma unroll
  for (int j = 0; j < kTileRows; j++)
    if ((uint32_t)(j / kGroupRows) < t.groupsK) v[j] = ldg<NT>(in + tileReadElem<FUSED>(t, a, wave, j, t.wK));
#pragma unroll
  for (int j = 0; j < kTileRows; j++)
    if ((uint32_t)(j / kGroupRows) < t.groupsK) tile[min(wave + kWaves * j, t.wK)][t.cx] = v[j];
  __syncthreads();
  T u[kTileRows];
#pragma unroll
  for (int j = 0; j < kTileRows; j++)
    if ((uint32_t)(j / kGroupRows) < t.groupsM) u[j] = tile[t.ck][min(wave + kWaves * j, t.wM)];
#pragma unroll
  for (int j = 0; j < kTileRows; j++)
    if ((uint32_t)(j / kGroupRows) < t.groupsM) stg<NT>(out + tileWriteElem<FUSED>(t, a, wave, j, t.wM), u[j]);
}

// How tiledKernel's loads leave: row group by row group without waiting, row group by row group waiting for each, as in moveTileTested.
enum { kLoadsPaced, kLoadsGrouped, kLoadsTested };

// Any numbering of the workgroups (tile_order.h: locateTile).
template <typename T, int NT, int LOADS, bool FUSED>
__global__ __launch_bounds__(kTileThreads) void tiledKernel(const cuttHipTiledArgs a,
                                                            const T* __restrict__ in,
                                                            T* __restrict__ out) {
  uint32_t tm, tk, offIn, offOut;
  if (!locateTile(a, tm, tk, offIn, offOut)) return;
  // tile geometry, clamped edges, skipped row groups: tile_order.h
  const TileLanes t = tileLanes<FUSED>(a, tm, tk, offIn, offOut, threadIdx.x & 63, threadIdx.x >> 6);
  if constexpr (LOADS != kLoadsTested) {
    // Rows in groups, or paced loads (cuttHipTiledArgs.paced): one piece of code whose row groups are tested one after the
    // other.  Without GROUPED a group's loads go out while the next one's addresses are computed, and no load is waited for before all are
    // out.  All sixteen at once (moveTile), what a small tensor needs, cost large ones up to 10 %, since neighbouring tiles no
    // longer find shared lines in the L2.
    // Written out here: as a function of its own, forced inline, the compiler keeps a lane's rows in one register tuple and merges it behind every
    // test with copies that wait for the loads: (777,111,1000)/(1,0,2), 8 bytes, 246.7 us here, 252.5 that way, (633,147,1602)/(1,0,2) 442.5 / 453.4,
    // (9,7,23,7,46,11,5,3)/(4,7,0,6,3,1,5,2), 4 bytes, 157.1 / 160.3; 24 such tensors 0.9 % in the mean, -1.5 ... +2.4 %.  With rows in
    // groups a straight piece of code per number of row groups costs 3.5-5.5 % instead: 16411 x 9377, 4 bytes, 282.4 us here, 296.3 that way.
    constexpr bool GROUPED = LOADS == kLoadsGrouped;
    const uint32_t wave = threadIdx.x >> 6;
    __shared__ T tile[kTile][kTile + 1];
    {
      T v[kTileRows];
#pragma unroll
      for (int g = 0; g < kRowGroups; g++) {
        if ((uint32_t)g < t.groupsK) {
#pragma unroll
          for (int j = g * kGroupRows; j < (g + 1) * kGroupRows; j++) v[j] = ldg<NT>(in + tileReadElem<FUSED>(t, a, wave, j, t.wK));
          if constexpr (GROUPED) {
            waitForGlobalAccesses();
#pragma unroll
            for (int j = g * kGroupRows; j < (g + 1) * kGroupRows; j++) tile[min(wave + kWaves * j, t.wK)][t.cx] = v[j];
          }
        }
      }
      if constexpr (!GROUPED) {
#pragma unroll
        for (int g = 0; g < kRowGroups; g++) {
          if ((uint32_t)g < t.groupsK) {
#pragma unroll
            for (int j = g * kGroupRows; j < (g + 1) * kGroupRows; j++) tile[min(wave + kWaves * j, t.wK)][t.cx] = v[j];
          }
        }
      }
    }
    __syncthreads();
    T v[kTileRows];
#pragma unroll
    for (int g = 0; g < kRowGroups; g++) {
      if ((uint32_t)g < t.groupsM) {
#pragma unroll
        for (int j = g * kGroupRows; j < (g + 1) * kGroupRows; j++) v[j] = tile[t.ck][min(wave + kWaves * j, t.wM)];
        if constexpr (GROUPED) {
#pragma unroll
          for (int j = g * kGroupRows; j < (g + 1) * kGroupRows; j++) stg<NT>(out + tileWriteElem<FUSED>(t, a, wave, j, t.wM), v[j]);
          waitForGlobalAccesses();
        }
      }
    }
    if constexpr (!GROUPED) {
#pragma unroll
      for (int g = 0; g < kRowGroups; g++) {
        if ((uint32_t)g < t.groupsM) {
#pragma unroll
          for (int j = g * kGroupRows; j < (g + 1) * kGroupRows; j++) stg<NT>(out + tileWriteElem<FUSED>(t, a, wave, j, t.wM), v[j]);
        }
      }
    }
  } else {
    moveTileTested<T, NT, FUSED>(t, a, in, out);
  }
}

// The numberings of cuttHipTileWalk.  The arguments up to `shifts`, 14 words, are in scalar registers when a wave starts
// (the Makefile's kernarg-preload-count), so that a plain matrix transpose waits for nothing before its first load;
// MB and ROWS hold what launches with Mbar positions and with fused axes need besides.
// Bound by latency up to some 20 MB, by memory beyond.  Against the kernel above, with
// its loads in groups of four: 2011 x 1163, 4 bytes, 5.94 -> 4.38 us; (24,32,36,43)/(3,1,2,0), 8 bytes, 5.99 -> 4.86;
// 4297 x 1731, 8 bytes, 28.2 -> 25.5; (7,149,21,189)/(3,2,1,0), 4 bytes, 9.5 -> 7.8; (96,75,96,75)/(2,1,3,0), 8 bytes, 161.7 -> 159.0,
// 157.7 in XCD groups.
template <typename T, int NT, typename MB, typename ROWS>
__global__ __launch_bounds__(kTileThreads) void tiledWalkKernel(const T* __restrict__ in, T* __restrict__ out, uint32_t volMm, uint32_t volMk,
                                                                uint32_t strideInK, uint32_t strideOutM, uint32_t chunk, uint32_t superM,
                                                                uint32_t stripMul, uint32_t fullMul, uint32_t lastMul, uint32_t shifts,
                                                                const MB mb, const ROWS rows) {
  constexpr bool kFused = std::is_same_v<ROWS, WalkAxes>;
  uint32_t tm, tk, offIn, offOut;
  if (!walkTile(blockIdx.x, WalkHead{chunk, superM, stripMul, fullMul, lastMul, shifts}, mb, (volMm + kTile - 1) / kTile, (volMk + kTile - 1) / kTile, tm, tk, offIn, offOut)) return;
  const WalkShape<ROWS> shape{volMm, volMk, strideInK, strideOutM, rows};
  const TileLanes t = tileLanes<kFused>(shape, tm, tk, offIn, offOut, threadIdx.x & 63, threadIdx.x >> 6);
  moveTile<T, NT, kFused>(t, shape, in, out);
}

// Tiles of 128x128 4-byte elements, whole ones only, numbered by a walk.
// Bound by the memory channels: a 64x64 tile touches 256 bytes of a row at a time, and with rows a power of two apart the
// pieces in flight crowd into few channels.  512 bytes of each row on both sides spread them: 8192 x 8192 101 (64x64) -> 95 us,
// 16384 x 8192 214 -> 176, 8192 x 16384 213 -> 185, 10240 x 10240 163 -> 147.  1024 lanes with 16 loads each, two workgroups per CU
// (66 KB of LDS); reading and writing the same pieces without transposing is 2 % slower with 512 lanes, 5-20 % with tiles of 256x64 or 64x256.
template <int NT, typename MB>
__global__ __launch_bounds__(CUTT_WIDE_THREADS, 8) void wideTileKernel(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, uint32_t volMm, uint32_t volMk,
                                                                   uint32_t strideInK, uint32_t strideOutM, uint32_t chunk, uint32_t superM,
                                                                   uint32_t stripMul, uint32_t fullMul, uint32_t lastMul, uint32_t shifts,
                                                                   const MB mb) {
  constexpr uint32_t kEdge = CUTT_WIDE_TILE, kStep = CUTT_WIDE_THREADS / kEdge;
  constexpr int kRows = kEdge / kStep;
  __shared__ uint32_t tile[kEdge][kEdge + 1];
  uint32_t tm, tk, offIn, offOut;
  if (!walkTile(blockIdx.x, WalkHead{chunk, superM, stripMul, fullMul, lastMul, shifts}, mb, volMm / kEdge, volMk / kEdge, tm, tk, offIn, offOut)) return;
  const uint32_t c = threadIdx.x % kEdge, r = threadIdx.x / kEdge;
  const uint32_t rd = offIn + tm * kEdge + c + (tk * kEdge + r) * strideInK, wr = offOut + tk * kEdge + c + (tm * kEdge + r) * strideOutM;
  uint32_t v[kRows];
#pragma unroll
  for (int j = 0; j < kRows; j++) v[j] = ldg<NT>(in + (rd + j * kStep * strideInK));
#pragma unroll
  for (int j = 0; j < kRows; j++) tile[r + j * kStep][c] = v[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kRows; j++) stg<NT>(out + (wr + j * kStep * strideOutM), tile[c][r + j * kStep]);
}

// ---------------------------------------------------------------------------
// Tiled with line-aligned stores.
// ---------------------------------------------------------------------------
// Bound by memory bandwidth.  When the output rows (runs along Mk) start off the 128-byte grid, the 64-wide store
// of a tile row covers the lines at its two ends partly, and the tile next door completes them later.  Here every
// row of a tile takes its own window of 64 elements along Mk: row m, whose output run starts s_m elements past a
// line boundary, stores the elements [64 tk - s_m, 64 tk - s_m + 64) of its run, so a store of a wave is whole
// lines (except at the two ends of a run) and can go past the caches.  The windows of the rows of a tile differ by
// up to one line, so the workgroup reads up to 64 + (elements per line - 1) rows along Mk into a taller LDS tile;
// the rows in the fringe are also read by the tile next door, from the L2, which is why the loads are temporal.
//
// 23425 x 8538, 8 bytes: 675 us with ordinary tiles (4.75 TB/s) -> 605 us, 560 (5.7 TB/s) since the XCDs share the
// workgroups in groups; 16411 x 9377, 4 bytes: 282 -> 241, 227; (132,11,3,47,14,2,35)/(2,1,3,6,5,0,4), 4 bytes: 358 -> 323, 315
// (buffers in rotation).  One workgroup for two to nine windows in turn, which reads no fringe row twice, is 0-10 % slower with
// 8-byte elements and 10-50 % with 4-byte ones.  Read from beyond the
// L2: 1.21 times the tensor's bytes on the first (ordinary tiles 1.03), 1.00 times on the third and on
// (200000,2,500)/(2,1,0), where every fringe row hits the L2; written 1.000-1.002 times (1.007-1.054).  The same windows
// with ordinary stores gain half of that, ordinary tiles with non-temporal stores lose 20-40 % (their partial lines go
// to memory twice).  512 lanes for 8-byte elements keep 11 loads per lane in flight, 256 for narrow tiles of 4-byte
// ones 26; twice the lanes with half the loads each are 1-2 % slower, four times 10-60 %.
//
// A tile is lineWidth columns wide along Mm (plan.cpp: lineTileWidth): its elements are read in order of rows and
// columns, so that a width of 33 or 66 leaves no lane of a request idle.
template <typename T, int TH>
constexpr int kLineLoads = sizeof(T) == 8 ? 11 : 26;  // per lane: rows * width / TH, rounded up

template <typename T, int TH, int NT, bool FUSED>
__global__ __launch_bounds__(TH) void tiledLinesKernel(const cuttHipTiledArgs a, const cuttHipDivisor widthDiv, const T* __restrict__ in, T* __restrict__ out) {
  constexpr uint32_t LE = kLineElems<T>;
  constexpr int LOADS = kLineLoads<T, TH>;
  static_assert(kLineRows<T> * (TH == 256 ? CUTT_LINE_WIDTH : kLineMaxWidth<T>) <= LOADS * TH, "the loads reach every element of a tile");
  extern __shared__ __align__(16) unsigned char ldsRaw[];
  __shared__ uint32_t rowIn[FUSED ? kLineRows<T> : 1], rowOut[FUSED ? TH : 1];
  T* const tile = reinterpret_cast<T*>(ldsRaw);

  uint32_t tm, tk, offIn, offOut;
  if (!locateTile<true>(a, tm, tk, offIn, offOut)) return;
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t outWord = (uint32_t)(reinterpret_cast<uintptr_t>(out) / sizeof(T)) + offOut;
  const LineTile t = lineTile<T>(a, tm, tk, outWord);
  if (t.rows == 0) return;
  if constexpr (FUSED) {
    if (tid < t.rows) rowIn[tid] = lineRowIn<true>(a, (uint32_t)t.kLo + tid);
    if (tid < t.width) rowOut[tid] = lineRowOut<true>(a, t.m0 + tid);
    __syncthreads();
  }
  {
    const uint32_t n = t.rows * t.width;
    const uint32_t base = offIn + t.m0 + (FUSED ? 0u : (uint32_t)t.kLo * a.strideInK);
    T v[LOADS];
    uint32_t slot[LOADS];
#pragma unroll
    for (int j = 0; j < LOADS; j++) {
      if ((uint32_t)(j * TH) < n) {  // uniform over the workgroup
        uint32_t r, c;
        lineElem(a, widthDiv, t, min(tid + j * TH, n - 1), r, c);
        slot[j] = r * t.pitch + c;
        v[j] = ldg<NT>(in + (base + (FUSED ? rowIn[r] : r * a.strideInK) + c));
      }
    }
#pragma unroll
    for (int j = 0; j < LOADS; j++)
      if ((uint32_t)(j * TH) < n) tile[slot[j]] = v[j];
  }
  __syncthreads();
  // Write: lanes run along Mk inside the row's own window.
#pragma unroll 8
  for (uint32_t r = tid >> 6; r < t.width; r += TH / 64) {
    const uint32_t rowStart = offOut + (FUSED ? rowOut[r] : (t.m0 + r) * a.strideOutM);
    const uint32_t s = (outWord - offOut + rowStart) & (LE - 1);
    const int32_t k = t.kWin - (int32_t)s + (int32_t)lane;
    if (k >= 0 && k < a.volMk) stg<NT>(out + (rowStart + (uint32_t)k), tile[(uint32_t)(k - t.kLo) * t.pitch + r]);
  }
}

// ---------------------------------------------------------------------------
// TiledCopy: rank 0 stays in front; rows are copied through registers.
// ---------------------------------------------------------------------------
template <typename T, int NT>
__global__ __launch_bounds__(kTileThreads) void tiledCopyKernel(const cuttHipCopyTiles a,
                                                                const T* __restrict__ in,
                                                                T* __restrict__ out) {
  uint32_t tm, tk, offIn, offOut;
  if (!locateTile(a, tm, tk, offIn, offOut)) return;

  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = threadIdx.x >> 6;
  const uint32_t m0 = tm * kTile, k0 = tk * kTile;
  // Clamped indices instead of branches, as in the tiled kernel.
  const uint32_t cx = min(lane, min((uint32_t)kTile, (uint32_t)a.volMm - m0) - 1);
  const uint32_t wK = min((uint32_t)kTile, (uint32_t)a.volMk - k0) - 1;
  const T* src = in + (offIn + m0 + cx);
  T* dst = out + (offOut + m0 + cx);

  // Row groups that lie beyond the tile's valid rows are skipped, as in the tiled kernel.
  const uint32_t groupsK = (wK >> 4) + 1;
  T v[kTileRows];
#pragma unroll
  for (int g = 0; g < kRowGroups; g++) {
    if ((uint32_t)g < groupsK) {
#pragma unroll
      for (int j = g * kGroupRows; j < (g + 1) * kGroupRows; j++) {
        const uint32_t r = min(wave + kWaves * j, wK);
        v[j] = ldg<NT>(src + (k0 + r) * a.strideInK);
      }
    }
  }
#pragma unroll
  for (int g = 0; g < kRowGroups; g++) {
    if ((uint32_t)g < groupsK) {
#pragma unroll
      for (int j = g * kGroupRows; j < (g + 1) * kGroupRows; j++) {
        const uint32_t r = min(wave + kWaves * j, wK);
        stg<NT>(dst + (k0 + r) * a.strideOutK, v[j]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// TiledCopy, dense tensors: the output written front to back.
// ---------------------------------------------------------------------------
// Bound by memory bandwidth.  What the 64x64 copy tiles and the packed kernel lose on such tensors is lost on
// the write side: their requests start off the 128-byte lines wherever a row does, so that lines are written in
// two parts.  Here the unit of work is a piece of the output instead - CUTT_ROW_BLOCK elements from one line
// boundary to another, whatever rows they belong to -, every store of a wave is whole lines, which can then go
// past the caches (non-temporal), and only the loads start anywhere.  (1305,599,88)/(0,2,1) of 4-byte elements,
// 550 MB moved: 120 us (packed kernel, 4.6 TB/s) -> 97 us (5.7 TB/s; a linear copy takes 84); 8-byte elements
// 226 -> 187 us; (115340,289,6)/(0,2,1), 4 bytes: 336 -> 265 us; (84,700,500)/(0,2,1), 4 bytes: 56 -> 48 us (buffers
// in rotation).  Four elements per lane: two are 30 % slower for 4-byte elements, eight 1-3 % slower.
template <typename T, int NT>
__global__ __launch_bounds__(kRowThreads) void rowGatherKernel(const cuttHipRowArgs a, const T* __restrict__ in,
                                                               T* __restrict__ out) {
  __shared__ uint32_t rowIn[CUTT_ROW_TABLE];
  const uint32_t tid = threadIdx.x;
  // the block's first element, counted from the output's first element: a 128-byte line starts there
  const uint32_t s = (uint32_t)(reinterpret_cast<uintptr_t>(out) / sizeof(T)) & (kLineElems<T> - 1);
  RowBlock b;
  if (!locateRows(a, s, b)) return;
  if (tid < b.rows) rowIn[tid] = rowInputOffset(a, b.row0 + tid);
  __syncthreads();
  T v[kRowElems];
#pragma unroll
  for (int j = 0; j < kRowElems; j++) {
    const uint32_t p = b.col0 + (min(max(tid + kRowThreads * j, b.lo), b.hi - 1) - b.lo);
    const uint32_t r = fastDivide(p, a.rowDiv.mul, a.rowDiv.shift, a.rowDiv.add);
    v[j] = ldg<NT>(in + (rowIn[r] + (p - r * a.rowLen)));
  }
  T* dst = out + b.first;
  if (b.lo == 0 && b.hi == CUTT_ROW_BLOCK) {
#pragma unroll
    for (int j = 0; j < kRowElems; j++) stg<NT>(dst + (tid + kRowThreads * j), v[j]);
  } else {  // first or last block of the tensor
#pragma unroll
    for (int j = 0; j < kRowElems; j++) {
      const uint32_t i = tid + kRowThreads * j;
      if (i >= b.lo && i < b.hi) dst[i] = v[j];
    }
  }
}

// ---------------------------------------------------------------------------
// Packed / PackedSplit: stage a block of Mmk through LDS with remap tables.
// ---------------------------------------------------------------------------

// The general kernel: 64-bit offsets, more than twelve Mbar ranks, loops of fewer than four elements per lane and 8-byte loops of 13-16
// waves (cuttHipFinishPackedWalk).  Bound by memory.
// E = elements per lane.  Every lane keeps its E table entries in registers, so that the loop
// over work items does no index arithmetic beyond adding the item's base offsets; the loop is
// software-pipelined (an item's loads are in flight while the previous one is gathered and stored).
// WIDE = false: the tensor is smaller than 4 GB, so the lanes keep 32-bit byte offsets and every
// access is "uniform 64-bit base + 32-bit lane offset" (no per-access 64-bit address registers).  WIDE = true:
// element offsets and 64-bit address arithmetic.
// (The 8-byte instance with 8 elements per lane sits at the edge of a register granule: it is held to the 80
// registers that let six of its waves share a SIMD; the other instances get what the compiler gives them.)
template <typename T, int E, bool WIDE>
constexpr int kPackedMinWaves = (sizeof(T) == 8 && E == 8 && !WIDE) ? 6 : 1;

template <typename T, int E, int NT, bool WIDE>
__global__ __launch_bounds__(1024, (kPackedMinWaves<T, E, WIDE>)) void packedKernel(const cuttHipPackedArgs a, const T* __restrict__ in,
                             T* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char ldsRaw[];
  constexpr uint32_t kScale = WIDE ? 1u : (uint32_t)sizeof(T);

  const uint32_t tid = threadIdx.x;
  const uint32_t nt = blockDim.x;
  // which work items this workgroup handles, and where an item lies: packed_items.h
  const PackedItems items = packedItems(a);
  const uint32_t count = items.count;
  const int padShift = a.padShift;

  // Lanes whose element index lies beyond the block repeat the block's last element (same
  // addresses, same value), so that the code below has no branches and every lane's E loads go
  // out back to back.
  uint32_t inOff[E], outOff[E];  // global offsets: bytes (narrow) or elements (wide)
  uint32_t shSlot[E];            // byte offset of the LDS slot an output element is taken from
  uint32_t last = 0;             // last element index of the class whose data is being loaded
  const MbarLane mbarLane = loadMbarLane(a.mbar, tid & 63);

  auto locate = [&](uint32_t i, int& c, uint32_t& offIn, uint32_t& offOut) __attribute__((always_inline)) {
    packedLocate(a, items, mbarLane, i, c, offIn, offOut);
  };
  // The lane's table entries of class c: the read side (input offsets, element count) and the
  // write side (output offsets, LDS gather slots) are fetched separately, because the next item's
  // loads go out while the current item's stores are still to come.
  auto loadReadSide = [&](int c) __attribute__((always_inline)) {
    const cuttHipPackedClass& k = a.cls[c];
    last = (uint32_t)k.vol - 1;
#pragma unroll
    for (int j = 0; j < E; j++) inOff[j] = packedInElem(k, min(tid + j * nt, last)) * kScale;
  };
  auto loadWriteSide = [&](int c) __attribute__((always_inline)) {
    const cuttHipPackedClass& k = a.cls[c];
    const uint32_t lastP = (uint32_t)k.vol - 1;
    const uint16_t* gSh = k.shIdx;
#pragma unroll
    for (int j = 0; j < E; j++) {
      const uint32_t p = min(tid + j * nt, lastP);
      const uint32_t sh = *reinterpret_cast<const uint16_t*>(reinterpret_cast<const unsigned char*>(gSh) + p * 2u);
      outOff[j] = packedOutElem(k, p) * kScale;
      shSlot[j] = sh * (uint32_t)sizeof(T);
    }
  };
  T v[E];  // data on its way in: global memory -> registers -> LDS
  auto issueLoads = [&](uint32_t offIn) __attribute__((always_inline)) {
    const unsigned char* srcB = reinterpret_cast<const unsigned char*>(in + offIn);  // wave-uniform base
#pragma unroll
    for (int j = 0; j < E; j++) {
      if (WIDE)
        v[j] = ldg<NT>(reinterpret_cast<const T*>(srcB) + inOff[j]);
      else
        v[j] = ldg<NT>(reinterpret_cast<const T*>(srcB + inOff[j]));
    }
  };
  // The slot of element p is p + (p >> padShift).  It is recomputed for every item from a value
  // the compiler cannot see through, so that it does not park E more registers.
  auto stage = [&]() __attribute__((always_inline)) {
    uint32_t tv = tid;
    asm volatile("" : "+v"(tv));
#pragma unroll
    for (int j = 0; j < E; j++) {
      const uint32_t p = min(tv + j * nt, last);
      *reinterpret_cast<T*>(ldsRaw + (p + (p >> padShift)) * (uint32_t)sizeof(T)) = v[j];
    }
  };
  auto gatherAndStore = [&](uint32_t offOut) __attribute__((always_inline)) {
    unsigned char* dstB = reinterpret_cast<unsigned char*>(out + offOut);
    T u[E];
#pragma unroll
    for (int j = 0; j < E; j++) u[j] = *reinterpret_cast<const T*>(ldsRaw + shSlot[j]);
#pragma unroll
    for (int j = 0; j < E; j++) {
      if (WIDE)
        stg<NT>(reinterpret_cast<T*>(dstB) + outOff[j], u[j]);
      else
        stg<NT>(reinterpret_cast<T*>(dstB + outOff[j]), u[j]);
    }
  };

  // Software pipeline over the workgroup's items: the loads of item w+1 are issued before the LDS
  // gather and the stores of item w, so they overlap, and the wait for them (the memory counter
  // counts loads and stores in issue order) does not also wait for those stores to complete.
  if (count == 0) return;
  uint32_t w = 0, offIn, offOut;  // index of the item among the workgroup's own
  int cls;
  locate(w, cls, offIn, offOut);
  loadReadSide(cls);
  issueLoads(offIn);
  loadWriteSide(cls);  // after the data loads are out: its latency hides behind theirs
  stage();
  for (;;) {
    if (w + 1 >= count) {  // last item: nothing to fetch ahead
      __syncthreads();
      gatherAndStore(offOut);
      break;
    }
    int clsNext;
    uint32_t offInNext, offOutNext;
    locate(w + 1, clsNext, offInNext, offOutNext);
    // the slab class changes at most a few times per workgroup (wave-uniform tests)
    if (clsNext != cls) loadReadSide(clsNext);
    issueLoads(offInNext);
    __syncthreads();  // item w is complete in the LDS buffer
    gatherAndStore(offOut);
    if (clsNext != cls) {
      loadWriteSide(clsNext);
      cls = clsNext;
    }
    __syncthreads();  // every lane has taken its elements of item w out of the buffer
    stage();
    w++;
    offOut = offOutNext;
  }
}

// The usual packed kernels (cuttHipPackedWalk): below 4 GB, up to twelve Mbar ranks.  The arguments up to `padThreads`, 14 words, are in scalar
// registers when a wave starts (the Makefile's kernarg-preload-count), the others are read at addresses known from the start, and
// the table reads go out before the Mbar position is decoded: the kernel above waits for some ten reads, one after the other, before its first load.
//
// One block per workgroup.  Bound by latency up to some 10 MB per buffer, by memory and the table reads (three of them per element, from the L2)
// beyond.  Against the kernel above, 100 tensors of 4-90 MB per buffer: 0.91 of the time in the mean, 0.73-1.05; (4,2,40,2,14,9,14)/(2,0,3,4,5,6,1),
// 4 bytes, 4.6 -> 3.8 us; (24,32,16,36,9)/(4,1,3,2,0), 8 bytes, 12.9 -> 11.7; (13,509,1082)/(1,0,2), 4 bytes, 16.5 -> 12.0: 56
// registers instead of 72 leave room for a second workgroup of 13 waves.  Tables with every lane's offsets ready, read 16 bytes at a time, are 5 %
// faster below 6 MB and 2-20 % slower beyond (10 bytes per element from the L2); run tables read by the scalar unit 20 % slower there.
template <typename T, int E, int NT>
__global__ __launch_bounds__(1024) void packedOnceKernel(const T* __restrict__ in, T* __restrict__ out, const unsigned char* __restrict__ tables, uint32_t chunk,
                                                         uint32_t shifts, uint32_t items, uint32_t num0, uint32_t mul0, uint32_t num1, uint32_t mul1,
                                                         uint32_t padThreads, const cuttHipPackedWalk a) {
  extern __shared__ __align__(16) unsigned char ldsRaw[];
  T* const tile = reinterpret_cast<T*>(ldsRaw);
  uint32_t c, m, offIn, offOut;
  if (!packedWalkSlabs<true>(walkPosition(blockIdx.x, chunk, shifts), 0, shifts, items, num0, mul0, num1, mul1, a, c, m, offIn, offOut)) return;
  const uint32_t tid = threadIdx.x, nt = padThreads >> 8, padShift = padThreads & 31;
  const cuttHipPackedWalkClass k = a.cls[c];
  // Lanes beyond the block's end repeat its last element (same addresses, same value).
  uint32_t rowIn[E], rowOut[E], sh[E];
  T v[E];
#pragma unroll
  for (int j = 0; j < E; j++) {
    const uint32_t p = min(tid + j * nt, k.last), r = walkDivide(p, k.inMul, k.shifts & 31);
    rowIn[j] = *reinterpret_cast<const uint32_t*>(tables + (k.rowIn + r * 4u)) + (p - r * k.inCont);
  }
#pragma unroll
  for (int j = 0; j < E; j++) {
    const uint32_t p = min(tid + j * nt, k.last), r = walkDivide(p, k.outMul, k.shifts >> 5);
    sh[j] = *reinterpret_cast<const uint16_t*>(tables + (k.shIdx + p * 2u));
    rowOut[j] = *reinterpret_cast<const uint32_t*>(tables + (k.rowOut + r * 4u)) + (p - r * k.outCont);
  }
  packedWalkMbar(a, m, offIn, offOut);
  const unsigned char* const src = reinterpret_cast<const unsigned char*>(in + offIn);  // wave-uniform base, 32-bit byte offsets
  unsigned char* const dst = reinterpret_cast<unsigned char*>(out + offOut);
#pragma unroll
  for (int j = 0; j < E; j++) v[j] = ldg<NT>(reinterpret_cast<const T*>(src + rowIn[j] * (uint32_t)sizeof(T)));
#pragma unroll
  for (int j = 0; j < E; j++) {
    const uint32_t p = min(tid + j * nt, k.last);
    tile[p + (p >> padShift)] = v[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < E; j++) v[j] = tile[sh[j]];
#pragma unroll
  for (int j = 0; j < E; j++) stg<NT>(reinterpret_cast<T*>(dst + rowOut[j] * (uint32_t)sizeof(T)), v[j]);
}

// Where the walk lies among the arguments of the kernel below: behind three pointers and eight words.
constexpr uint32_t kPackedWalkAt = 3 * 8 + 8 * 4;
static_assert(alignof(cuttHipPackedWalk) == 4, "no gap in front of it");

// Several blocks per workgroup (4-byte elements beyond some 60 MB, where the table reads weigh most, and 8-byte ones in more than 12000 blocks), in a software pipeline: a block's loads
// are issued before the LDS gather and the stores of the one before, so they overlap, and the wait for them (the memory counter counts loads and
// stores in issue order) does not also wait for those stores to complete.  Bound by memory.  Against packedKernel, 70 tensors of 90-700 MB per
// buffer: 0.7 % faster in the mean, (6,18,5,14,8,24,17)/(0,5,1,6,2,3,4), 4 bytes, 42.3 -> 39.2 us, (15,2842,3021)/(1,0,2), 4 bytes, 193 -> 188.
// (The instances with 8 elements per lane are held to the 72 and 80 registers that let seven and six of their waves share a SIMD.  64, and eight
// waves, cost the 4-byte one 1 % in the mean over 70 tensors, up to 7 %: what is in flight then crowds the L2, which has to hold the lines
// that neighbouring blocks complete.)
template <typename T, int E>
constexpr int kLoopMinWaves = E == 8 ? (sizeof(T) == 4 ? 7 : 6) : 1;

template <typename T, int E, int NT>
__global__ __launch_bounds__(1024, (kLoopMinWaves<T, E>)) void packedLoopKernel(const T* __restrict__ in, T* __restrict__ out, const unsigned char* __restrict__ tables, uint32_t chunk,
                                                         uint32_t shifts, uint32_t items, uint32_t num0, uint32_t mul0, uint32_t num1, uint32_t mul1,
                                                         uint32_t padThreads, const cuttHipPackedWalk a) {
  extern __shared__ __align__(16) unsigned char ldsRaw[];
  T* const tile = reinterpret_cast<T*>(ldsRaw);
  const uint32_t tid = threadIdx.x, nt = padThreads >> 8, padShift = padThreads & 31;
  const uint32_t first = walkPosition(blockIdx.x, chunk, shifts) * a.first;
  uint32_t c, m, offIn, offOut;
  if (!packedWalkSlabs<false>(first, 0, shifts, items, num0, mul0, num1, mul1, a, c, m, offIn, offOut)) return;
  // Lanes beyond the block's end repeat its last element (same addresses, same value).
  uint32_t rd[E], wr[E];  // byte offsets
  uint32_t sh[(E + 1) / 2];  // LDS slots, two to a register
  uint32_t last = 0;  // last element of the class whose data is being loaded
  auto readSide = [&](uint32_t cls) __attribute__((always_inline)) {
    const cuttHipPackedWalkClass k = a.cls[cls];
    last = k.last;
#pragma unroll
    for (int j = 0; j < E; j++) {
      const uint32_t p = min(tid + j * nt, k.last), r = walkDivide(p, k.inMul, k.shifts & 31);
      rd[j] = (*reinterpret_cast<const uint32_t*>(tables + (k.rowIn + r * 4u)) + (p - r * k.inCont)) * (uint32_t)sizeof(T);
    }
  };
  auto writeSide = [&](uint32_t cls) __attribute__((always_inline)) {
    const cuttHipPackedWalkClass k = a.cls[cls];
#pragma unroll
    for (int j = 0; j < E; j++) {
      const uint32_t p = min(tid + j * nt, k.last), r = walkDivide(p, k.outMul, k.shifts >> 5);
      const uint32_t slot = *reinterpret_cast<const uint16_t*>(tables + (k.shIdx + p * 2u));
      sh[j / 2] = j % 2 ? sh[j / 2] | slot << 16 : slot;
      wr[j] = (*reinterpret_cast<const uint32_t*>(tables + (k.rowOut + r * 4u)) + (p - r * k.outCont)) * (uint32_t)sizeof(T);
    }
  };
  T v[E];  // data on its way in: global memory -> registers -> LDS
  auto request = [&](uint32_t off) __attribute__((always_inline)) {
    const unsigned char* const src = reinterpret_cast<const unsigned char*>(in + off);
#pragma unroll
    for (int j = 0; j < E; j++) v[j] = ldg<NT>(reinterpret_cast<const T*>(src + rd[j]));
  };
  // (computed for every block from a value the compiler cannot see through, so that the slots do not take E more registers)
  auto stage = [&]() __attribute__((always_inline)) {
    uint32_t tv = tid;
    asm volatile("" : "+v"(tv));
#pragma unroll
    for (int j = 0; j < E; j++) {
      const uint32_t p = min(tv + j * nt, last);
      tile[p + (p >> padShift)] = v[j];
    }
  };
  auto gatherAndStore = [&](uint32_t off) __attribute__((always_inline)) {
    unsigned char* const dst = reinterpret_cast<unsigned char*>(out + off);
    T u[E];
#pragma unroll
    for (int j = 0; j < E; j++) u[j] = tile[j % 2 ? sh[j / 2] >> 16 : sh[j / 2] & 0xffffu];
#pragma unroll
    for (int j = 0; j < E; j++) stg<NT>(reinterpret_cast<T*>(dst + wr[j]), u[j]);
  };
  readSide(c);
  packedWalkMbar(a, m, offIn, offOut);
  request(offIn);
  writeSide(c);  // its latency hides behind the data's
  stage();
  for (uint32_t i = 1;; i++) {
    // The arguments are read again for every block, from where the launch put them (the cache of the scalar unit, that is): kept, they take
    // all scalar registers, and some to memory.
    typedef const __attribute__((address_space(4))) unsigned char* KernelArguments;
    KernelArguments args = (KernelArguments)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    const auto& w = *reinterpret_cast<const __attribute__((address_space(4))) cuttHipPackedWalk*>(args + kPackedWalkAt);
    uint32_t next, offInNext, offOutNext;
    if (i >= w.perGroup || !packedWalkSlabs<false>(first + i * w.stepN, i, shifts, items, num0, mul0, num1, mul1, w, next, m, offInNext, offOutNext)) break;
    packedWalkMbar(w, m, offInNext, offOutNext);
    if (next != c) readSide(next);  // (wave-uniform; at most a few times per workgroup)
    request(offInNext);
    __syncthreads();  // the block is complete in LDS
    gatherAndStore(offOut);
    if (next != c) {
      writeSide(next);
      c = next;
    }
    __syncthreads();  // every lane has taken its elements out
    stage();
    offOut = offOutNext;
  }
  __syncthreads();
  gatherAndStore(offOut);
}

// The table must carry the division constants cuttHipFinishMbar derives from its extents.
bool mbarOk(const cuttHipMbar& mb) {
  cuttHipMbar want = mb;
  if (cuttHipFinishMbar(&want) != 0) return false;
  for (int k = 0; k < CUTT_MAX_RANK; k++)
    if (want.d[k].belowMul != mb.d[k].belowMul || want.d[k].extentMul != mb.d[k].extentMul ||
        want.d[k].ctl != mb.d[k].ctl)
      return false;
  return true;
}

bool divisorOk(const cuttHipDivisor& dv, uint32_t d) {
  const cuttHipDivisor want = cuttHipMakeDivisor(d);
  return dv.mul == want.mul && dv.shift == want.shift && dv.add == want.add;
}

// Number of workgroups of a tiled launch; checks the ordering parameters.
bool tileGrid(int order, int tilesM, int tilesK, int volMbar, uint32_t xcdChunk, int xcdGroup, uint32_t superM,
              uint32_t superK, const cuttHipTileDigits& dg, const cuttHipMbar& mbar, uint64_t& blocks, uint64_t threads = kTileThreads) {
  uint64_t logical = (uint64_t)tilesM * tilesK * (uint64_t)volMbar;
  if (order == 7) {
    if (dg.n < 1 || dg.n > CUTT_MAX_TILE_DIGITS) return false;
    logical = 1;
    for (int i = 0; i < dg.n; i++) {
      const cuttHipTileDigit& d = dg.d[i];
      if (d.radix < 1 || d.which > 2 || !divisorOk(d.div, d.radix)) return false;
      logical *= d.radix;
      if (logical > 0x7fffffffull) return false;  // the decode divides 31-bit numbers
    }
    // per coordinate the digits, taken by growing weight, must be a mixed-radix number that reaches the extent
    const uint64_t extent[3] = {(uint64_t)tilesM, (uint64_t)tilesK, (uint64_t)volMbar};
    for (uint32_t w = 0; w < 3; w++) {
      uint64_t span = 1;
      for (;;) {
        int next = -1;
        for (int i = 0; i < dg.n; i++)
          if (dg.d[i].which == w && dg.d[i].weight == span && dg.d[i].radix > 1 && (next < 0 || dg.d[i].radix > dg.d[next].radix)) next = i;
        if (next < 0) break;
        span *= dg.d[next].radix;
      }
      uint64_t all = 1;
      for (int i = 0; i < dg.n; i++)
        if (dg.d[i].which == w && dg.d[i].radix > 1) all *= dg.d[i].radix;
      if (span != all || span < extent[w]) return false;
    }
    // what the kernels decode with must be what cuttHipFinishTileDigits derives from the list
    // (a list without lanes is decoded digit by digit, which needs none of this)
    if (dg.lanes) {
      cuttHipTileDigits want = dg;
      if (cuttHipFinishTileDigits(&want, &mbar) != 0 || want.lanes != 1 || want.total != dg.total ||
          std::memcmp(want.lane, dg.lane, sizeof(dg.lane)) != 0)
        return false;
    }
  } else if (order >= 3) {
    if (superM < 1 || superK < 1) return false;
    logical = (uint64_t)((tilesM + superM - 1) / superM) * ((tilesK + superK - 1) / superK) * superM * superK *
              (uint64_t)volMbar;
  }
  blocks = logical;
  if (xcdGroup < 0 || xcdGroup > 20 || (xcdGroup && order == 7)) return false;
  if (xcdGroup) {
    const uint64_t unit = (uint64_t)kNumXcd << (xcdGroup - 1);
    blocks = (logical + unit - 1) / unit * unit;
  } else if (xcdChunk) {
    if ((uint64_t)xcdChunk * kNumXcd < logical) return false;
    blocks = (uint64_t)xcdChunk * kNumXcd;
  }
  return blocks > 0 && blocks <= 0x7fffffffull && blocks * threads <= CUTT_HIP_MAX_GRID_LANES;
}

// The rows of a tile axis over fused ranks: the extents must multiply to the axis' length.
bool rowRadixOk(const cuttHipRowRadix& rr, int count) {
  if (rr.n == 0) return true;
  if (rr.n < 0 || rr.n > CUTT_MAX_TILE_SET) return false;
  uint64_t vol = 1;
  for (int k = 0; k < rr.n; k++) {
    if (rr.extent[k] < 1 || !divisorOk(rr.div[k], rr.extent[k])) return false;
    vol *= rr.extent[k];
    if (vol > 0x7fffffffull) return false;
  }
  return vol == (uint64_t)count;
}

bool rowsOk(const cuttHipRowArgs& a, int elemSize) {
  if (a.elemSize != elemSize || a.n < 1 || a.n > CUTT_MAX_RANK || a.rowLen < 1 || a.cachePolicy < 0 || a.cachePolicy > 3 ||
      a.xcdGroup < 0 || a.xcdGroup > 20 || CUTT_ROW_BLOCK / a.rowLen + 2 > CUTT_ROW_TABLE || !divisorOk(a.rowDiv, a.rowLen))
    return false;
  uint64_t rows = 1;
  for (int k = 0; k < a.n; k++) {
    const cuttHipRowRank& d = a.rank[k];
    if (d.extent < 1 || !divisorOk(cuttHipDivisor{d.mul, d.ctl & 0xff, d.ctl >> 8}, d.extent)) return false;
    rows *= d.extent;
    if (rows > 0x7fffffffull) return false;  // (rows are divided as 31-bit numbers)
  }
  return rows == a.numRows && rows * a.rowLen == a.volume && cuttHipRowGrid(&a) > 0;
}

// Allow dynamic LDS up to the device limit for a kernel (once per process and kernel).
template <typename K>
int allowLargeLds(K kernel, size_t bytes) {
  return (int)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// The same for the packed kernels whose arguments are decoded as a walk; loops over few elements per lane have none (cuttHipFinishPackedWalk).
template <typename T, int E, int NT>
int allowLargeLdsWalks(size_t bytes) {
  int r = allowLargeLds(packedOnceKernel<T, E, NT>, bytes);
  if constexpr (E >= CUTT_PACKED_LOOP_ELEMS)
    if (r == 0) r = allowLargeLds(packedLoopKernel<T, E, NT>, bytes);
  return r;
}

// ---------------------------------------------------------------------------
// Trivial method: a plain copy, 16 bytes per lane and one 4-KB piece per workgroup, so that the
// hardware dispatcher spreads the pieces and every wave has exactly one load and one store in
// flight.  Measured against the runtime's device-to-device copy: the same below 128 MB, 20-33 %
// faster from 256 MB on with streaming loads (6.4-7.0 against 4.9-5.4 TB/s).
// The last (bytes % 16) / 4 words are copied by the first lanes of workgroup 0.
typedef unsigned int Vec16 __attribute__((ext_vector_type(4)));
constexpr int kCopyThreads = 256;

template <int NT>
__global__ __launch_bounds__(kCopyThreads) void copyKernel(const Vec16* __restrict__ in, Vec16* __restrict__ out,
                                                           uint64_t n16, uint32_t tailWords) {
  const uint64_t i = (uint64_t)blockIdx.x * kCopyThreads + threadIdx.x;
  if (i < n16) stg<NT>(out + i, ldg<NT>(in + i));
  if (blockIdx.x == 0 && threadIdx.x < tailWords) {
    const uint32_t* in32 = (const uint32_t*)(in + n16);
    uint32_t* out32 = (uint32_t*)(out + n16);
    out32[threadIdx.x] = in32[threadIdx.x];
  }
}

}  // namespace

extern "C" int cuttHipPackedRegsPerLaneLoaded(int elemSize, int elemsPerThread, int wideOffsets) {
  const void* f = nullptr;
#define CUTT_PICK(T, E)                                                                       \
  f = wideOffsets ? reinterpret_cast<const void*>(packedKernel<T, E, 0, true>)               \
                  : reinterpret_cast<const void*>(packedKernel<T, E, 0, false>)
  if (elemSize == 4) {
    switch (elemsPerThread) {
      case 1: CUTT_PICK(uint32_t, 1); break;
      case 2: CUTT_PICK(uint32_t, 2); break;
      case 4: CUTT_PICK(uint32_t, 4); break;
      case 8: CUTT_PICK(uint32_t, 8); break;
      case 16: CUTT_PICK(uint32_t, 16); break;
      default: return -1;
    }
  } else if (elemSize == 8) {
    switch (elemsPerThread) {
      case 1: CUTT_PICK(uint64_t, 1); break;
      case 2: CUTT_PICK(uint64_t, 2); break;
      case 4: CUTT_PICK(uint64_t, 4); break;
      case 8: CUTT_PICK(uint64_t, 8); break;
      default: return -1;
    }
  } else {
    return -1;
  }
#undef CUTT_PICK
  hipFuncAttributes attr;
  if (hipFuncGetAttributes(&attr, f) != hipSuccess) return -1;
  return attr.numRegs;
}

namespace {

// A launch reports the launch call's own result.  (hipGetLastError after a launch would also report
// - and clear - an error that an earlier, unrelated call of the application left behind on this
// thread, such as hipErrorNotReady from a stream query.)
template <typename... KArgs, typename... Args>
hipError_t launchKernel(void (*kernel)(KArgs...), dim3 grid, dim3 block, size_t lds, hipStream_t s, Args... args) {
  static_assert(sizeof...(KArgs) == sizeof...(Args), "one argument per kernel parameter");
  std::tuple<std::remove_const_t<KArgs>...> held{args...};
  void* ptrs[sizeof...(KArgs)];
  int i = 0;
  std::apply([&](auto&... v) { ((ptrs[i++] = (void*)&v), ...); }, held);
  return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, ptrs, lds, s);
}

}  // namespace

static bool copyTileGrid(const cuttHipCopyTiles& t, uint64_t& blocks) {
  return tileGrid(t.order, t.tilesM, t.tilesK, t.volMbar, t.xcdChunk, 0, t.superM, t.superK, t.digits, t.mbar, blocks);
}

// Lanes of a workgroup of these arguments.
static uint32_t tiledThreads(const cuttHipTiledArgs& a) {
  return a.lineWidth ? (uint32_t)cuttHipLinesThreads(a.elemSize, a.lineWidth) : (a.wide ? CUTT_WIDE_THREADS : (uint32_t)kTileThreads);
}

extern "C" long long cuttHipTiledGrid(const cuttHipTiledArgs* a) {
  uint64_t blocks = 0;
  if (!a || !tileGrid(a->order, a->tilesM, a->tilesK, a->volMbar, a->xcdChunk, a->xcdGroup, a->superM, a->superK, a->digits, a->mbar, blocks, tiledThreads(*a)))
    return 0;
  return (long long)blocks;
}

extern "C" long long cuttHipTiledCopyGrid(const cuttHipTiledCopyArgs* a) {
  uint64_t blocks = 0;
  if (!a || !copyTileGrid(a->tiles, blocks)) return 0;
  return (long long)blocks;
}

extern "C" int cuttHipValidateTiled(const cuttHipTiledArgs* a) {
  if (!a) return (int)hipErrorInvalidValue;
  if ((a->elemSize != 4 && a->elemSize != 8) || a->volMm < 1 || a->volMk < 1 || a->volMbar < 1)
    return (int)hipErrorInvalidValue;
  if ((a->wide != 0 && a->wide != 1) || (a->wide && (a->elemSize != 4 || a->lineWidth || a->grouped || a->rowsK.n > 0 || a->rowsM.n > 0 ||
                                                     a->volMm % CUTT_WIDE_TILE || a->volMk % CUTT_WIDE_TILE || a->walk.kind == 0)))
    return (int)hipErrorInvalidValue;
  const int edge = a->wide ? CUTT_WIDE_TILE : kTile;
  const int width = a->lineWidth ? a->lineWidth : edge, fringe = a->lineWidth ? 128 / a->elemSize - 1 : 0;
  if (width < 1 || (a->lineWidth && (width > cuttHipLinesMaxWidth(a->elemSize) || a->volMk > 0x7fffffff - 2 * kTile ||
                                     a->volMm > 0x7fffffff - 2 * kTile)) ||
      a->tilesM != (a->volMm + width - 1) / width || a->tilesK != (a->volMk + fringe + edge - 1) / edge ||
      a->order < 0 || a->order > 7 || !mbarOk(a->mbar) || (a->grouped != 0 && a->grouped != 1) || (a->paced != 0 && a->paced != 1) ||
      !rowRadixOk(a->rowsK, a->volMk) || !rowRadixOk(a->rowsM, a->volMm))
    return (int)hipErrorInvalidValue;
  uint64_t blocks = 0;
  if (!tileGrid(a->order, a->tilesM, a->tilesK, a->volMbar, a->xcdChunk, a->xcdGroup, a->superM, a->superK, a->digits, a->mbar, blocks, tiledThreads(*a)))
    return (int)hipErrorInvalidConfiguration;
  if (a->cachePolicy < 0 || a->cachePolicy > 3) return (int)hipErrorInvalidValue;
  if (a->walk.kind != 0) {  // the walk must be the one that follows from the other arguments
    cuttHipTiledArgs want = *a;
    cuttHipFinishTileWalk(&want);
    if (std::memcmp(&want.walk, &a->walk, sizeof(want.walk)) != 0) return (int)hipErrorInvalidValue;
  }
  return 0;
}

// Line-aligned stores: 8-byte elements and wide tiles of 4-byte ones take 512 lanes.
static int launchLines(const cuttHipTiledArgs& a, const void* in, void* out, uint32_t blocks, hipStream_t s) {
  const uint32_t threads = tiledThreads(a);
  const dim3 grid(blocks), block(threads);
  const size_t lds = cuttHipLinesLdsBytes(a.elemSize, a.lineWidth);
  const cuttHipDivisor widthDiv = cuttHipMakeDivisor((uint32_t)a.lineWidth);
  const bool fused = a.rowsK.n > 0 || a.rowsM.n > 0;
#define CUTT_LAUNCH_LINES(T, TH, NT)                                                                              \
  return (int)(fused ? launchKernel(tiledLinesKernel<T, TH, NT, true>, grid, block, lds, s, a, widthDiv, (const T*)in, (T*)out) \
                     : launchKernel(tiledLinesKernel<T, TH, NT, false>, grid, block, lds, s, a, widthDiv, (const T*)in, (T*)out))
#define CUTT_LAUNCH_LINES_NT(T, TH)           \
  switch (a.cachePolicy) {                    \
    case 0: CUTT_LAUNCH_LINES(T, TH, 0);      \
    case 1: CUTT_LAUNCH_LINES(T, TH, 1);      \
    case 2: CUTT_LAUNCH_LINES(T, TH, 2);      \
    default: CUTT_LAUNCH_LINES(T, TH, 3);     \
  }
  if (a.elemSize == 8) {
    CUTT_LAUNCH_LINES_NT(uint64_t, 512)
  } else if (threads == 512) {
    CUTT_LAUNCH_LINES_NT(uint32_t, 512)
  } else {
    CUTT_LAUNCH_LINES_NT(uint32_t, 256)
  }
#undef CUTT_LAUNCH_LINES_NT
#undef CUTT_LAUNCH_LINES
}

// Tiles in the sequence of a walk.
template <typename T, int NT, typename MB, typename ROWS>
static int launchWalkOf(const cuttHipTiledArgs& a, const MB& mb, const ROWS& rows, const void* in, void* out, hipStream_t s) {
  const cuttHipTileWalk& w = a.walk;
  return (int)launchKernel(tiledWalkKernel<T, NT, MB, ROWS>, dim3(w.blocks), dim3(kTileThreads), 0, s, (const T*)in, (T*)out, (uint32_t)a.volMm,
                           (uint32_t)a.volMk, a.strideInK, a.strideOutM, w.chunk, w.superM, w.stripMul, w.fullMul, w.lastMul, w.shifts, mb, rows);
}

template <typename T, int NT>
static int launchWalkNt(const cuttHipTiledArgs& a, const void* in, void* out, hipStream_t s) {
  const bool fused = a.rowsK.n > 0 || a.rowsM.n > 0;
  const WalkAxes axes{a.walk.rowsK, a.walk.rowsM};
  if (a.walk.kind == 1) return fused ? launchWalkOf<T, NT>(a, NoMbar{}, axes, in, out, s) : launchWalkOf<T, NT>(a, NoMbar{}, NoAxes{}, in, out, s);
  return fused ? launchWalkOf<T, NT>(a, a.walk.mbar, axes, in, out, s) : launchWalkOf<T, NT>(a, a.walk.mbar, NoAxes{}, in, out, s);
}

template <typename T>
static int launchWalkOfWidth(const cuttHipTiledArgs& a, const void* in, void* out, hipStream_t s) {
  switch (a.cachePolicy) {
    case 0: return launchWalkNt<T, 0>(a, in, out, s);
    case 1: return launchWalkNt<T, 1>(a, in, out, s);
    case 2: return launchWalkNt<T, 2>(a, in, out, s);
    default: return launchWalkNt<T, 3>(a, in, out, s);
  }
}

template <int NT, typename MB>
static int launchWideOf(const cuttHipTiledArgs& a, const MB& mb, const void* in, void* out, hipStream_t s) {
  const cuttHipTileWalk& w = a.walk;
  return (int)launchKernel(wideTileKernel<NT, MB>, dim3(w.blocks), dim3(CUTT_WIDE_THREADS), 0, s, (const uint32_t*)in, (uint32_t*)out, (uint32_t)a.volMm,
                           (uint32_t)a.volMk, a.strideInK, a.strideOutM, w.chunk, w.superM, w.stripMul, w.fullMul, w.lastMul, w.shifts, mb);
}

static int launchWide(const cuttHipTiledArgs& a, const void* in, void* out, hipStream_t s) {
  const bool single = a.walk.kind == 1;
  switch (a.cachePolicy) {
    case 0: return single ? launchWideOf<0>(a, NoMbar{}, in, out, s) : launchWideOf<0>(a, a.walk.mbar, in, out, s);
    case 1: return single ? launchWideOf<1>(a, NoMbar{}, in, out, s) : launchWideOf<1>(a, a.walk.mbar, in, out, s);
    case 2: return single ? launchWideOf<2>(a, NoMbar{}, in, out, s) : launchWideOf<2>(a, a.walk.mbar, in, out, s);
    default: return single ? launchWideOf<3>(a, NoMbar{}, in, out, s) : launchWideOf<3>(a, a.walk.mbar, in, out, s);
  }
}

static int launchWalk(const cuttHipTiledArgs& a, const void* in, void* out, hipStream_t s) {
  return a.elemSize == 4 ? launchWalkOfWidth<uint32_t>(a, in, out, s) : launchWalkOfWidth<uint64_t>(a, in, out, s);
}

extern "C" int cuttHipLaunchTiled(const cuttHipTiledArgs* a, const void* in, void* out, void* stream) {
  if (!a || !in || !out) return (int)hipErrorInvalidValue;
  uint64_t blocks = 0;
  if (!tileGrid(a->order, a->tilesM, a->tilesK, a->volMbar, a->xcdChunk, a->xcdGroup, a->superM, a->superK, a->digits, a->mbar, blocks, tiledThreads(*a)))
    return (int)hipErrorInvalidConfiguration;
  hipStream_t s = (hipStream_t)stream;
  if (a->lineWidth) return launchLines(*a, in, out, (uint32_t)blocks, s);
  if (cuttHipTiledTakesWalk(a)) return a->wide ? launchWide(*a, in, out, s) : launchWalk(*a, in, out, s);
  if (a->wide) return (int)hipErrorInvalidValue;  // (no other kernel knows such tiles)
  const dim3 grid((uint32_t)blocks), block(kTileThreads);
  const bool fused = a->rowsK.n > 0 || a->rowsM.n > 0;
#define CUTT_LAUNCH_TILED_F(T, NT, LOADS)                                                                        \
  (fused ? launchKernel(tiledKernel<T, NT, LOADS, true>, grid, block, 0, s, *a, (const T*)in, (T*)out)           \
         : launchKernel(tiledKernel<T, NT, LOADS, false>, grid, block, 0, s, *a, (const T*)in, (T*)out))
#define CUTT_LAUNCH_TILED(T, NT)                                                                                 \
  return (int)(a->grouped                                               ? CUTT_LAUNCH_TILED_F(T, NT, kLoadsGrouped) \
               : sizeof(T) == 8 || a->paced || !(a->cachePolicy & 2) ? CUTT_LAUNCH_TILED_F(T, NT, kLoadsPaced)   \
                                                                     : CUTT_LAUNCH_TILED_F(uint32_t, NT | 2, kLoadsTested))
#define CUTT_LAUNCH_TILED_NT(T)                                \
  switch (a->cachePolicy) {                                    \
    case 0: CUTT_LAUNCH_TILED(T, 0);                           \
    case 1: CUTT_LAUNCH_TILED(T, 1);                           \
    case 2: CUTT_LAUNCH_TILED(T, 2);                           \
    default: CUTT_LAUNCH_TILED(T, 3);                          \
  }
  if (a->elemSize == 4) {
    CUTT_LAUNCH_TILED_NT(uint32_t)
  } else {
    CUTT_LAUNCH_TILED_NT(uint64_t)
  }
#undef CUTT_LAUNCH_TILED_NT
#undef CUTT_LAUNCH_TILED
#undef CUTT_LAUNCH_TILED_F
}

extern "C" int cuttHipValidateTiledCopy(const cuttHipTiledCopyArgs* a) {
  if (!a) return (int)hipErrorInvalidValue;
  const cuttHipCopyTiles& t = a->tiles;
  if ((t.elemSize != 4 && t.elemSize != 8) || t.volMm < 1 || t.volMk < 1 || t.volMbar < 1 || t.tilesM != (t.volMm + kTile - 1) / kTile ||
      t.tilesK != (t.volMk + kTile - 1) / kTile || t.order < 0 || t.order > 7 || !mbarOk(t.mbar))
    return (int)hipErrorInvalidValue;
  uint64_t blocks = 0;
  if (!copyTileGrid(t, blocks)) return (int)hipErrorInvalidConfiguration;
  if (t.cachePolicy < 0 || t.cachePolicy > 3) return (int)hipErrorInvalidValue;
  if (a->rowGather && !rowsOk(a->rows, t.elemSize)) return (int)hipErrorInvalidValue;
  return 0;
}

// Rows of a TiledCopy plan gathered in output order.
static int launchRows(const cuttHipRowArgs& a, const void* in, void* out, hipStream_t s) {
  const uint64_t blocks = cuttHipRowGrid(&a);
  if (blocks == 0) return (int)hipErrorInvalidConfiguration;
  const dim3 grid((uint32_t)blocks), block(kRowThreads);
#define CUTT_LAUNCH_ROWS(T, NT) return (int)launchKernel(rowGatherKernel<T, NT>, grid, block, 0, s, a, (const T*)in, (T*)out)
#define CUTT_LAUNCH_ROWS_NT(T)             \
  switch (a.cachePolicy) {                 \
    case 0: CUTT_LAUNCH_ROWS(T, 0);        \
    case 1: CUTT_LAUNCH_ROWS(T, 1);        \
    case 2: CUTT_LAUNCH_ROWS(T, 2);        \
    default: CUTT_LAUNCH_ROWS(T, 3);       \
  }
  if (a.elemSize == 4) {
    CUTT_LAUNCH_ROWS_NT(uint32_t)
  } else {
    CUTT_LAUNCH_ROWS_NT(uint64_t)
  }
#undef CUTT_LAUNCH_ROWS_NT
#undef CUTT_LAUNCH_ROWS
}

extern "C" int cuttHipLaunchTiledCopy(const cuttHipTiledCopyArgs* a, const void* in, void* out,
                                      void* stream) {
  if (!a || !in || !out) return (int)hipErrorInvalidValue;
  if (a->rowGather) return launchRows(a->rows, in, out, (hipStream_t)stream);
  uint64_t blocks = 0;
  if (!copyTileGrid(a->tiles, blocks)) return (int)hipErrorInvalidConfiguration;
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((uint32_t)blocks), block(kTileThreads);
#define CUTT_LAUNCH_TCOPY(T, NT) \
  return (int)launchKernel(tiledCopyKernel<T, NT>, grid, block, 0, s, a->tiles, (const T*)in, (T*)out)
#define CUTT_LAUNCH_TCOPY_NT(T)                                \
  switch (a->tiles.cachePolicy) {                              \
    case 0: CUTT_LAUNCH_TCOPY(T, 0);                           \
    case 1: CUTT_LAUNCH_TCOPY(T, 1);                           \
    case 2: CUTT_LAUNCH_TCOPY(T, 2);                           \
    default: CUTT_LAUNCH_TCOPY(T, 3);                          \
  }
  if (a->tiles.elemSize == 4) {
    CUTT_LAUNCH_TCOPY_NT(uint32_t)
  } else {
    CUTT_LAUNCH_TCOPY_NT(uint64_t)
  }
#undef CUTT_LAUNCH_TCOPY_NT
#undef CUTT_LAUNCH_TCOPY
}

// Plain copy for the Trivial method.  Both pointers 16-byte aligned: copyKernel; otherwise the
// runtime's device-to-device copy.
extern "C" int cuttHipLaunchCopy(const void* in, void* out, size_t bytes, int cachePolicy, void* stream) {
  if (!in || !out || bytes == 0 || bytes % 4 != 0) return (int)hipErrorInvalidValue;
  if (cachePolicy < 0 || cachePolicy > 3) return (int)hipErrorInvalidValue;
  hipStream_t s = (hipStream_t)stream;
  if ((((uintptr_t)in | (uintptr_t)out) & 15) != 0)
    return (int)hipMemcpyAsync(out, in, bytes, hipMemcpyDeviceToDevice, s);
  const uint64_t n16 = bytes / 16;
  const uint32_t tailWords = (uint32_t)((bytes % 16) / 4);
  const uint64_t blocks = std::max<uint64_t>(1, (n16 + kCopyThreads - 1) / kCopyThreads);
  if (blocks > 0x7fffffffull || blocks * kCopyThreads > CUTT_HIP_MAX_GRID_LANES) return (int)hipErrorInvalidConfiguration;
  const dim3 grid((uint32_t)blocks), block(kCopyThreads);
  switch (cachePolicy) {
    case 0: return (int)launchKernel(copyKernel<0>, grid, block, 0, s, (const Vec16*)in, (Vec16*)out, n16, tailWords);
    case 1: return (int)launchKernel(copyKernel<1>, grid, block, 0, s, (const Vec16*)in, (Vec16*)out, n16, tailWords);
    case 2: return (int)launchKernel(copyKernel<2>, grid, block, 0, s, (const Vec16*)in, (Vec16*)out, n16, tailWords);
    default: return (int)launchKernel(copyKernel<3>, grid, block, 0, s, (const Vec16*)in, (Vec16*)out, n16, tailWords);
  }
}

// ---------------------------------------------------------------------------
// Static scratch memory and the kernel that builds a plan's index tables in it.
// ---------------------------------------------------------------------------
// Device memory that exists from the moment the code object is loaded: the entry point that must
// not allocate keeps a packed plan's index tables here.  In host code the array's name is only a
// handle for hipGetSymbolAddress; the address it returns (one per device) is what kernels get.
static __device__ __align__(256) unsigned char scratch[CUTT_HIP_SCRATCH_BYTES];

extern "C" int cuttHipScratch(void** ptr, size_t* bytes) {
  static std::mutex lock;
  static void* perDevice[64] = {};
  if (!ptr || !bytes) return (int)hipErrorInvalidValue;
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= 64) return (int)hipErrorInvalidDevice;
  std::lock_guard<std::mutex> guard(lock);
  if (!perDevice[dev]) {
    void* p = nullptr;
    if (hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)); e != hipSuccess) return (int)e;
    if (!p) return (int)hipErrorInvalidSymbol;
    perDevice[dev] = p;
  }
  *ptr = perDevice[dev];
  *bytes = CUTT_HIP_SCRATCH_BYTES;
  return 0;
}

namespace {
constexpr int kBuildThreads = 256;

// A list of cuttHipTableBuildArgs as the kernel evaluates it: RANKS steps without a test, the divisions by multiply-high.  The slowest
// rank takes what is left (constants and extent zero), the steps behind it contribute nothing.
struct BuildRank {
  uint32_t mul, shift, add, extent, stride;
};
template <int RANKS>
struct BuildLists {
  uint32_t *rowIn, *rowOut;
  uint16_t* shIdx;
  uint32_t count[3];
  int padShift;
  BuildRank rank[3][RANKS];
};
template <int RANKS, int CLASSES>
struct BuildClasses {
  BuildLists<RANKS> cls[CLASSES];
};

template <int RANKS>
__device__ __forceinline__ uint32_t radixSum(const BuildRank (&r)[RANKS], uint32_t i) {
  uint32_t off = 0;
#pragma unroll
  for (int k = 0; k < RANKS; k++) {
    const uint32_t q = fastDivide(i, r[k].mul, r[k].shift, r[k].add);
    off += (i - q * r[k].extent) * r[k].stride;
    i = q;
  }
  return off;
}

// Bound by the dispatch (1.8 us) and what one lane computes in turn.  With a division by a variable per rank and list, each waiting
// for the one before and for its extent, a call with such a build took 16.5 us on
// (24,32,16,36,9)/(4,1,3,2,0), 8 bytes (the transpose itself 13.0), 15.4 with these; (12,13,14,15,16)/(4,3,2,1,0), 8 bytes: 10.5 -> 8.9.
// One launch for all slab classes (blockIdx.y), where a launch for each cost 2 us more per class: (11,5,196,31,4)/(4,1,3,2,0), 8 bytes, two classes,
// 12.3 -> 10.0 us a call; (24,613,532)/(0,2,1), 4 bytes, four, 20.4 -> 14.1; (4,107,5,1475)/(2,0,3,1), 8 bytes, four, 22.0 -> 12.6.
template <int RANKS, int CLASSES>
__global__ __launch_bounds__(kBuildThreads) void buildTablesKernel(const BuildClasses<RANKS, CLASSES> classes) {
  const BuildLists<RANKS>& a = classes.cls[CLASSES > 1 ? blockIdx.y : 0];
  const uint32_t i = blockIdx.x * kBuildThreads + threadIdx.x;
  const uint32_t in = radixSum(a.rank[0], i), out = radixSum(a.rank[1], i), pos = radixSum(a.rank[2], i);
  if (i < a.count[0]) a.rowIn[i] = in;
  if (i < a.count[1]) a.rowOut[i] = out;
  if (i < a.count[2]) a.shIdx[i] = (uint16_t)(pos + (pos >> a.padShift));
}

template <int RANKS, int CLASSES>
hipError_t launchTableBuild(const cuttHipTableBuildArgs* args, int classes, uint32_t entries, hipStream_t s) {
  BuildClasses<RANKS, CLASSES> all = {};
  for (int c = 0; c < classes; c++) {
    const cuttHipTableBuildArgs& a = args[c];
    BuildLists<RANKS>& b = all.cls[c];
    b.rowIn = a.rowIn;
    b.rowOut = a.rowOut;
    b.shIdx = a.shIdx;
    b.padShift = a.padShift;
    for (int l = 0; l < 3; l++) {
      b.count[l] = a.count[l];
      for (int k = 0; k < a.list[l].n; k++) {
        b.rank[l][k].stride = a.list[l].stride[k];
        if (k + 1 == a.list[l].n) break;
        const cuttHipDivisor d = cuttHipMakeDivisor(a.list[l].extent[k]);
        b.rank[l][k].mul = d.mul;
        b.rank[l][k].shift = d.shift;
        b.rank[l][k].add = d.add;
        b.rank[l][k].extent = a.list[l].extent[k];
      }
    }
  }
  return launchKernel(buildTablesKernel<RANKS, CLASSES>, dim3((entries + kBuildThreads - 1) / kBuildThreads, (uint32_t)classes), dim3(kBuildThreads), 0, s, all);
}
}  // namespace

extern "C" int cuttHipLaunchTableBuilds(const cuttHipTableBuildArgs* args, int classes, void* stream) {
  if (!args || classes < 1 || classes > 4) return (int)hipErrorInvalidValue;
  uint32_t most = 0;
  int ranks = 0;
  for (int c = 0; c < classes; c++) {
    const cuttHipTableBuildArgs& a = args[c];
    if (!a.rowIn || !a.rowOut || !a.shIdx || a.padShift < 1 || a.padShift > 31) return (int)hipErrorInvalidValue;
    for (int l = 0; l < 3; l++) {
      if (a.count[l] < 1 || a.count[l] > 65536 || a.list[l].n < 0 || a.list[l].n > CUTT_MAX_RANK) return (int)hipErrorInvalidValue;
      uint64_t span = 1;  // the list must enumerate at least count entries
      for (int k = 0; k < a.list[l].n; k++) {
        if (a.list[l].extent[k] < 1) return (int)hipErrorInvalidValue;
        span *= a.list[l].extent[k];
        if (span > (1ull << 32)) return (int)hipErrorInvalidValue;
      }
      if (span != a.count[l]) return (int)hipErrorInvalidValue;
      most = std::max(most, a.count[l]);
      ranks = std::max(ranks, a.list[l].n);
    }
  }
  const hipStream_t s = (hipStream_t)stream;
  if (classes == 1) {
    if (ranks <= 4) return (int)launchTableBuild<4, 1>(args, 1, most, s);
    if (ranks <= 8) return (int)launchTableBuild<8, 1>(args, 1, most, s);
    if (ranks <= 12) return (int)launchTableBuild<12, 1>(args, 1, most, s);
    return (int)launchTableBuild<CUTT_MAX_RANK, 1>(args, 1, most, s);
  }
  if (ranks <= 4) return (int)launchTableBuild<4, 4>(args, classes, most, s);
  if (ranks <= 8) return (int)launchTableBuild<8, 4>(args, classes, most, s);
  if (ranks <= 12) return (int)launchTableBuild<12, 4>(args, classes, most, s);
  for (int c = 0; c < classes; c++)  // (four classes of 32 ranks each do not fit a launch's arguments)
    if (int e = cuttHipLaunchTableBuilds(args + c, 1, stream); e != 0) return e;
  return 0;
}

// Lets the packed kernels use more than the default 64 KB of dynamic LDS on the current device.
// Called when a packed plan is activated, so that every cuttExecute is a plain kernel launch.
extern "C" int cuttHipPreparePacked(void) {
  // Function attributes are kept per device.  Two threads may both find the flag clear and both
  // make the calls: they are idempotent.
  static std::atomic<bool> ldsOptInDone[64];
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return (int)e;
  const bool tracked = dev >= 0 && dev < 64;
  if (!tracked || !ldsOptInDone[dev]) {
    hipDeviceProp_t prop;
    if (hipError_t e = hipGetDeviceProperties(&prop, dev); e != hipSuccess) return (int)e;
    const size_t m = prop.sharedMemPerBlock;
    int r = 0;
#define CUTT_ALLOW(T, E)                                                  \
  if (r == 0) r = allowLargeLds(packedKernel<T, E, 0, false>, m);         \
  if (r == 0) r = allowLargeLds(packedKernel<T, E, 1, false>, m);         \
  if (r == 0) r = allowLargeLds(packedKernel<T, E, 2, false>, m);         \
  if (r == 0) r = allowLargeLds(packedKernel<T, E, 3, false>, m);         \
  if (r == 0) r = allowLargeLds(packedKernel<T, E, 0, true>, m);          \
  if (r == 0) r = allowLargeLds(packedKernel<T, E, 1, true>, m);          \
  if (r == 0) r = allowLargeLds(packedKernel<T, E, 2, true>, m);          \
  if (r == 0) r = allowLargeLds(packedKernel<T, E, 3, true>, m);          \
  if (r == 0) r = allowLargeLdsWalks<T, E, 0>(m);                         \
  if (r == 0) r = allowLargeLdsWalks<T, E, 1>(m);                         \
  if (r == 0) r = allowLargeLdsWalks<T, E, 2>(m);                         \
  if (r == 0) r = allowLargeLdsWalks<T, E, 3>(m)
    CUTT_ALLOW(uint32_t, 1); CUTT_ALLOW(uint32_t, 2); CUTT_ALLOW(uint32_t, 4); CUTT_ALLOW(uint32_t, 8);
    CUTT_ALLOW(uint32_t, 16);
    CUTT_ALLOW(uint64_t, 1); CUTT_ALLOW(uint64_t, 2); CUTT_ALLOW(uint64_t, 4); CUTT_ALLOW(uint64_t, 8);
#undef CUTT_ALLOW
    if (r != 0) return r;
    if (tracked) ldsOptInDone[dev] = true;
  }
  return 0;
}

// Number of workgroups of a packed launch (0 = the work items do not fit a grid).
static uint64_t packedGrid(const cuttHipPackedArgs* a) {
  const long long items = cuttHipPackedItemNumbers(a);
  if (items < 1) return 0;
  uint64_t blocks = ((uint64_t)items + a->itemsPerBlock - 1) / a->itemsPerBlock;
  if (a->xcdGroup < 0 || a->xcdGroup > 20) return 0;
  if (a->xcdGroup) {
    const uint64_t unit = (uint64_t)kNumXcd << (a->xcdGroup - 1);
    blocks = (blocks + unit - 1) / unit * unit;
  } else if (a->xcdChunk) {
    if ((uint64_t)a->xcdChunk * kNumXcd < blocks) return 0;
    blocks = (uint64_t)a->xcdChunk * kNumXcd;
  }
  return blocks <= 0x7fffffffull && blocks * (uint64_t)a->numThreads <= CUTT_HIP_MAX_GRID_LANES ? blocks : 0;
}

extern "C" long long cuttHipPackedGrid(const cuttHipPackedArgs* a) { return a ? (long long)packedGrid(a) : 0; }

extern "C" int cuttHipValidatePacked(const cuttHipPackedArgs* a) {
  if (!a) return (int)hipErrorInvalidValue;
  if ((a->elemSize != 4 && a->elemSize != 8) || a->numThreads < 64 || a->numThreads > 1024 ||
      (a->numThreads & 63) || a->volMbar < 1 || a->itemsPerBlock < 1 || a->padShift < 1 ||
      a->itemOrder < 0 || a->itemOrder > 2 ||
      (a->elemsPerThread != 1 && a->elemsPerThread != 2 && a->elemsPerThread != 4 &&
       a->elemsPerThread != 8 && !(a->elemsPerThread == 16 && a->elemSize == 4)) ||
      a->cachePolicy < 0 || a->cachePolicy > 3 ||
      a->padShift > 31 || a->ldsElems < 1 || a->ldsElems > 65536 || !mbarOk(a->mbar) || a->volume < 1 ||
      a->volume > 0xffffffffll ||
      // 32-bit byte offsets reach 4 GB
      (!a->wideOffsets && (uint64_t)a->volume * (uint64_t)a->elemSize > (1ull << 32)))
    return (int)hipErrorInvalidValue;
  for (int i = 0; i < 2; i++) {
    const cuttHipSplitRank& sr = a->split[i];
    if (sr.numSplit < 1 || sr.slabRem < 0 || sr.slabRem >= sr.numSplit || sr.slabFloor < 0 ||
        !divisorOk(sr.div, (uint32_t)sr.numSplit))
      return (int)hipErrorInvalidValue;
  }
  for (int c = 0; c < 4; c++) {
    // class c is used only if the split ranks it refers to have slabs of the larger size
    if (((c & 1) && a->split[0].slabRem == 0) || ((c & 2) && a->split[1].slabRem == 0)) continue;
    const cuttHipPackedClass& k = a->cls[c];
    if (k.vol < 1 || k.vol > a->maxVol || (int64_t)a->numThreads * a->elemsPerThread < k.vol || !k.rowIn ||
        !k.rowOut || !k.shIdx || k.inCont < 1 || k.outCont < 1 || k.vol % k.inCont || k.vol % k.outCont ||
        !divisorOk(k.inDiv, (uint32_t)k.inCont) || !divisorOk(k.outDiv, (uint32_t)k.outCont))
      return (int)hipErrorInvalidValue;
    const uint32_t last = (uint32_t)k.vol - 1;
    if ((int)(last + (last >> a->padShift)) >= a->ldsElems) return (int)hipErrorInvalidValue;
  }
  if (packedGrid(a) == 0) return (int)hipErrorInvalidConfiguration;
  if (a->walk.blocks != 0) {  // must be what follows from the other arguments
    cuttHipPackedArgs want = *a;
    cuttHipFinishPackedWalk(&want);
    if (std::memcmp(&want.walk, &a->walk, sizeof(want.walk)) != 0 || want.walk.blocks != packedGrid(a)) return (int)hipErrorInvalidValue;
  }
  return 0;
}

template <typename T, int E, int NT>
static int launchPackedWalk(const cuttHipPackedArgs& a, const void* in, void* out, hipStream_t s) {
  const cuttHipPackedWalk& o = a.walk;
  auto kernel = packedOnceKernel<T, E, NT>;
  if constexpr (E >= CUTT_PACKED_LOOP_ELEMS) {
    if (o.perGroup > 1) kernel = packedLoopKernel<T, E, NT>;
  } else if (o.perGroup > 1) {  // (has no walk)
    return (int)hipErrorInvalidValue;
  }
  return (int)launchKernel(kernel, dim3(o.blocks), dim3(a.numThreads), cuttHipPackedLdsBytes(&a), s, (const T*)in, (T*)out,
                           (const unsigned char*)a.cls[0].rowIn, o.chunk, o.shifts, o.items, o.num[0], o.mul[0], o.num[1], o.mul[1], o.padThreads, o);
}

extern "C" int cuttHipLaunchPacked(const cuttHipPackedArgs* a, const void* in, void* out, void* stream) {
  if (!a || !in || !out) return (int)hipErrorInvalidValue;
  const uint64_t blocks = packedGrid(a);
  if (blocks == 0) return (int)hipErrorInvalidConfiguration;
  const size_t lds = cuttHipPackedLdsBytes(a);
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((uint32_t)blocks), block(a->numThreads);
  const bool wide = a->wideOffsets != 0;
#define CUTT_LAUNCH_PACKED(T, E, NT)                                                                              \
  return a->walk.blocks ? launchPackedWalk<T, E, NT>(*a, in, out, s)                                              \
                        : (int)(wide ? launchKernel(packedKernel<T, E, NT, true>, grid, block, lds, s, *a, (const T*)in, (T*)out)  \
                    : launchKernel(packedKernel<T, E, NT, false>, grid, block, lds, s, *a, (const T*)in, (T*)out))
#define CUTT_LAUNCH_PACKED_NT(T, E)                            \
  switch (a->cachePolicy) {                                    \
    case 0: CUTT_LAUNCH_PACKED(T, E, 0);                       \
    case 1: CUTT_LAUNCH_PACKED(T, E, 1);                       \
    case 2: CUTT_LAUNCH_PACKED(T, E, 2);                       \
    default: CUTT_LAUNCH_PACKED(T, E, 3);                      \
  }
#define CUTT_LAUNCH_PACKED_E(T)                                \
  switch (a->elemsPerThread) {                                 \
    case 1: CUTT_LAUNCH_PACKED_NT(T, 1)                        \
    case 2: CUTT_LAUNCH_PACKED_NT(T, 2)                        \
    case 4: CUTT_LAUNCH_PACKED_NT(T, 4)                        \
    default: CUTT_LAUNCH_PACKED_NT(T, 8)                       \
  }
  if (a->elemSize == 4 && a->elemsPerThread == 16) {
    // 4-byte elements only: 16 per lane stage the same 64 KB as 8 per lane do for 8-byte elements
    CUTT_LAUNCH_PACKED_NT(uint32_t, 16)
  } else if (a->elemSize == 4) {
    CUTT_LAUNCH_PACKED_E(uint32_t)
  } else {
    CUTT_LAUNCH_PACKED_E(uint64_t)
  }
#undef CUTT_LAUNCH_PACKED_NT
#undef CUTT_LAUNCH_PACKED_E
#undef CUTT_LAUNCH_PACKED
}
