"""The walk form of a Tiled launch's numbering (cuttHipTileWalk) against the tile orders it stands for.

A C++ program decodes every workgroup index of random launches with the kernels' own code (tile_walk.h, compiled for the host, and the constants of
cuttHipFinishTileWalk), one chunk per XCD or groups, and compares the sequence of tiles, the Mbar offsets and the rows' offsets with the orders' own
definition, divisions and all; divisors near the limits are checked at the numerators where a wrong rounding shows first.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>
#include "tile_walk.h"
typedef uint32_t u;
struct Pos { u tm, tk, in, out; bool operator!=(const Pos& o) const { return tm != o.tm || tk != o.tk || in != o.in || out != o.out; } };
static void offsets(const cuttHipTiledArgs& a, u m, Pos& p) {
  p.in = p.out = 0;
  for (int k = 0; k < a.mbar.n; k++) {
    const u i = m % a.mbar.d[k].extent;
    m /= a.mbar.d[k].extent;
    p.in += i * a.mbar.d[k].strideIn;
    p.out += i * a.mbar.d[k].strideOut;
  }
}
static std::vector<Pos> byOrder(const cuttHipTiledArgs& a) {  // the orders' definition, padding positions left out
  std::vector<Pos> v;
  const u M = a.tilesM, K = a.tilesK, B = a.volMbar, sm = a.superM, sk = a.superK, nM = (M + sm - 1) / sm, nK = (K + sk - 1) / sk;
  const uint64_t n = a.order < 3 ? (uint64_t)M * K * B : (uint64_t)nM * nK * sm * sk * B;
  for (uint64_t l = 0; l < n; l++) {
    Pos p; u m;
    if (a.order == 1) { p.tm = l % M; p.tk = l / M % K; m = l / M / K; }
    else if (a.order == 2) { p.tk = l % K; p.tm = l / K % M; m = l / K / M; }
    else {
      const u w = l % (sm * sk), t = l / (sm * sk), st = a.order == 5 ? t / B : t % (nM * nK);
      m = a.order == 5 ? t % B : t / (nM * nK);
      p.tm = st % nM * sm + w % sm; p.tk = st / nM * sk + w / sm;
    }
    if (p.tm >= M || p.tk >= K || m >= B) continue;
    offsets(a, m, p);
    v.push_back(p);
  }
  return v;
}
static bool decode(const cuttHipTiledArgs& a, u bid, Pos& p) {
  const cuttHipTileWalk& h = a.walk;
  const cutt::WalkHead head{h.chunk, h.superM, h.stripMul, h.fullMul, h.lastMul, h.shifts};
  return h.kind == 2 ? cutt::walkTile(bid, head, h.mbar, a.tilesM, a.tilesK, p.tm, p.tk, p.in, p.out)
                     : cutt::walkTile(bid, head, cutt::NoMbar{}, a.tilesM, a.tilesK, p.tm, p.tk, p.in, p.out);
}
static size_t position(const cuttHipTiledArgs& a, u bid) {  // what the fields' comments say
  if (!a.xcdChunk) return bid;
  if (!a.xcdGroup) return (size_t)(bid % 8) * a.walk.chunk + bid / 8;
  const u g = 1u << (a.xcdGroup - 1), turn = bid / 8 / g;  // XCD b % 8 takes groups of g in turn
  return (size_t)(turn * 8 + bid % 8) * g + bid / 8 % g;
}
static u rowPlain(const cuttHipRowRadix& rr, u stride, u i) {
  if (rr.n == 0) return i * stride;
  u off = 0;
  for (int k = 0; k < rr.n; k++) { off += (k + 1 < rr.n ? i % rr.extent[k] : i) * rr.stride[k]; i /= rr.extent[k]; }
  return off;
}
int main() {
  std::mt19937 g(5);
  auto r = [&](int lo, int hi) { return lo + (int)(g() % (unsigned)(hi - lo + 1)); };
  long walks = 0;
  for (int t = 0; t < 4000; t++) {
    cuttHipTiledArgs a; std::memset(&a, 0, sizeof(a));
    a.elemSize = r(0, 1) ? 4 : 8;
    a.tilesM = r(1, 40); a.tilesK = r(1, 40);
    a.volMm = a.tilesM * 64 - r(0, 63); a.volMk = a.tilesK * 64 - r(0, 63);
    a.order = r(0, 6); a.superM = r(1, a.tilesM); a.superK = r(0, 3) ? a.tilesK : r(1, a.tilesK);
    a.mbar.n = r(0, 2) ? 0 : r(1, 9); a.volMbar = 1;
    for (int k = 0; k < a.mbar.n; k++) {
      a.mbar.d[k].extent = a.volMbar > 30 ? r(1, 2) : r(1, 7);
      a.mbar.d[k].strideIn = g(); a.mbar.d[k].strideOut = g(); a.volMbar *= a.mbar.d[k].extent;
    }
    const uint64_t logical = (uint64_t)a.tilesM * a.tilesK * a.volMbar;
    a.xcdChunk = logical >= 64 ? (u)((logical + 7) / 8) : 0;
    a.xcdGroup = (int16_t)(a.xcdChunk && r(0, 1) ? r(1, 9) : 0);
    const uint64_t unit = a.xcdGroup ? 8ull << (a.xcdGroup - 1) : (a.xcdChunk ? 8 : 1);
    a.strideInK = g(); a.strideOutM = g();
    for (cuttHipRowRadix* rr : {&a.rowsK, &a.rowsM}) {
      rr->n = r(0, 4);
      if (rr->n == 1) rr->n = 0;
      for (int k = 0; k < rr->n; k++) { rr->extent[k] = r(1, 50); rr->stride[k] = g(); }
    }
    cuttHipFinishTileWalk(&a);
    const bool strips = (a.order == 3 || a.order == 5) && (int)a.superK >= a.tilesK;
    if ((a.walk.kind != 0) != ((strips || a.order == 1 || a.order == 2) && a.mbar.n <= CUTT_WALK_RANKS)) return std::printf("kind %d of order %d\n", a.walk.kind, a.order), 1;
    if (!a.walk.kind) continue;
    walks++;
    const std::vector<Pos> want = byOrder(a);
    if (want.size() != logical || a.walk.blocks != (logical + unit - 1) / unit * unit) return std::printf("%zu positions, %u workgroups\n", want.size(), a.walk.blocks), 1;
    size_t seen = 0;
    for (u b = 0; b < a.walk.blocks; b++) {
      const size_t l = position(a, b);
      if (l != cutt::xcdPosition(b, a.xcdGroup ? a.xcdChunk : a.walk.chunk, a.xcdGroup)) return std::printf("workgroup %u: position\n", b), 1;
      Pos p;
      if (decode(a, b, p) != (l < logical)) return std::printf("workgroup %u: end\n", b), 1;
      if (l >= logical) continue;
      if (p != want[l]) return std::printf("order %d, workgroup %u: tile (%u,%u) instead of (%u,%u)\n", a.order, b, p.tm, p.tk, want[l].tm, want[l].tk), 1;
      seen++;
    }
    if (seen != logical) return std::printf("%zu of %zu tiles\n", seen, (size_t)logical), 1;
    for (int i = 0; i < 300; i++) {
      u k = 1, m = 1;
      for (int j = 0; j < a.rowsK.n; j++) k *= a.rowsK.extent[j];
      for (int j = 0; j < a.rowsM.n; j++) m *= a.rowsM.extent[j];
      k = g() % (a.rowsK.n ? k : 0x7fffffffu); m = g() % (a.rowsM.n ? m : 0x7fffffffu);
      if (cutt::walkRowOffset(a.walk.rowsK, k) != rowPlain(a.rowsK, a.strideInK, k) || cutt::walkRowOffset(a.walk.rowsM, m) != rowPlain(a.rowsM, a.strideOutM, m)) return std::printf("row offsets\n"), 1;
    }
  }
  if (walks < 1000) return std::printf("only %ld walks\n", walks), 1;
  // the divisions at their limits: a row rank's extent may be any number below 2^31
  std::vector<u> ds = {1, 2, 3, 5, 7, 64, 65, 641, 65535, 65536, 65537, 46341, 0x3fffffffu, 0x40000000u, 0x40000001u, 0x7ffffffeu, 0x7fffffffu};
  for (int i = 0; i < 20000; i++) ds.push_back(1u + (g() >> r(1, 31)) % 0x7fffffffu);
  for (u d : ds) {
    cuttHipTiledArgs a; std::memset(&a, 0, sizeof(a));
    a.tilesM = a.tilesK = a.volMbar = 1; a.order = 1; a.rowsK.n = 2; a.rowsK.extent[0] = d; a.rowsK.stride[1] = 1;
    cuttHipFinishTileWalk(&a);
    for (int i = 0; i < 40; i++) {
      const uint64_t q = (g() % (0x7fffffffull / d + 1)) * d;
      for (uint64_t n : {q, q + d - 1, q > 0 ? q - 1 : 0, (uint64_t)0x7fffffff}) {
        if (n > 0x7fffffffull) continue;
        if (cutt::walkRowOffset(a.walk.rowsK, (u)n) != (u)n / d) return std::printf("%llu / %u\n", (unsigned long long)n, d), 1;
      }
    }
  }
  std::printf("ok %ld\n", walks);
  return 0;
}
"""


def test_walks_visit_the_tiles_of_their_orders(tmp_path):
    src = tmp_path / "walk.cpp"
    src.write_text(PROGRAM)
    exe = str(tmp_path / "walk")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "cutt_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
                           str(src), os.path.join(ROOT, "cutt_amd", "csrc", "layer_math.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout
