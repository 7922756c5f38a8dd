"""The packed kernel for one block per workgroup (cuttHipPackedWalk) against the arguments it is derived from.

A C++ program decodes every workgroup index of random launches with the kernel's own code (packed_walk.h, compiled for the host) and compares
slab class and offsets with the work items' definition, and the class's constants with its tables and run lengths.
"""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>
#include "packed_walk.h"
typedef uint32_t u;
#define CHECK(x) do { if (!(x)) { printf("failed: %s (launch %d)\n", #x, t); return 1; } } while (0)
int main() {
  std::mt19937 g(7);
  auto r = [&](int lo, int hi) { return lo + (int)(g() % (unsigned)(hi - lo + 1)); };
  static unsigned char mem[1 << 20];
  long items = 0, classes = 0;
  for (int t = 0; t < 3000; t++) {
    cuttHipPackedArgs a; std::memset(&a, 0, sizeof(a));
    a.elemSize = r(0, 1) ? 4 : 8; a.elemsPerThread = 4; a.itemsPerBlock = r(0, 1) ? 1 : r(2, 9); a.itemOrder = r(0, 2); a.numThreads = 64 * r(1, a.elemSize == 8 && a.itemsPerBlock > 1 ? 12 : 16); a.padShift = r(0, 3) ? 5 : 31;
    a.mbar.n = r(0, CUTT_PACKED_RANKS); a.volMbar = 1;
    for (int k = 0; k < a.mbar.n; k++) {
      a.mbar.d[k].extent = a.volMbar > 100 ? 1 : r(1, 7);
      a.mbar.d[k].strideIn = g(); a.mbar.d[k].strideOut = g();
      a.volMbar *= a.mbar.d[k].extent;
    }
    for (int i = 0; i < 2; i++) {
      cuttHipSplitRank& s = a.split[i];
      s.numSplit = r(0, 1) ? 1 : r(1, 30);
      if (s.numSplit > 1) { s.slabFloor = r(1, 9); s.slabRem = r(0, 1) ? 0 : r(0, s.numSplit - 1); s.strideIn = g(); s.strideOut = g(); }
    }
    const long n = (long)a.volMbar * a.split[0].numSplit * a.split[1].numSplit;
    if (r(0, 2)) a.xcdChunk = (u)(((cuttHipPackedItemNumbers(&a) + a.itemsPerBlock - 1) / a.itemsPerBlock + 7) / 8);
    if (a.xcdChunk && r(0, 1)) a.xcdGroup = r(1, 6);
    size_t at = 64 * r(0, 9);
    for (int c = 0; c < 4; c++) {
      if (((c & 1) && !a.split[0].slabRem) || ((c & 2) && !a.split[1].slabRem)) continue;
      cuttHipPackedClass& k = a.cls[c];
      k.inCont = r(1, 50); k.outCont = r(1, 50); k.vol = k.inCont * k.outCont * r(1, 20);
      k.rowIn = (const u*)(mem + at); at += 16 * r(1, 9); k.rowOut = (const u*)(mem + at); at += 16 * r(1, 9); k.shIdx = (const uint16_t*)(mem + at); at += 16 * r(1, 9);
    }
    cuttHipFinishPackedWalk(&a);
    const cuttHipPackedWalk& o = a.walk;
    CHECK(o.blocks > 0 && (o.padThreads & 31) == (u)a.padShift && (o.padThreads >> 8) == (u)a.numThreads);
    const unsigned char* base = (const unsigned char*)a.cls[0].rowIn;
    for (int c = 0; c < 4; c++) {
      const cuttHipPackedClass& k = a.cls[c];
      if (!k.vol) continue;
      const cuttHipPackedWalkClass& w = o.cls[c];
      CHECK(w.last + 1 == (u)k.vol && w.inCont == (u)k.inCont && w.outCont == (u)k.outCont);
      CHECK(base + w.rowIn == (const unsigned char*)k.rowIn && base + w.rowOut == (const unsigned char*)k.rowOut && base + w.shIdx == (const unsigned char*)k.shIdx);
      for (u p = 0; p < 65536; p += 1 + g() % 97)
        CHECK(cutt::walkDivide(p, w.inMul, w.shifts & 31) == p / w.inCont && cutt::walkDivide(p, w.outMul, w.shifts >> 5) == p / w.outCont);
      classes++;
    }
    std::vector<char> seen(n, 0);
    const u per = a.itemsPerBlock, ns0 = a.split[0].numSplit, ns1 = a.split[1].numSplit, groups = (cuttHipPackedItemNumbers(&a) + per - 1) / per;
    for (u b = 0; b < o.blocks; b++) {
      u l = b;  // the comments of xcdChunk and xcdGroup
      if (a.xcdGroup) { const u q = 1u << (a.xcdGroup - 1), turn = b / 8 / q; l = (turn * 8 + b % 8) * q + b / 8 % q; }
      else if (a.xcdChunk) l = b % 8 * a.xcdChunk + b / 8;
      const u first = cutt::walkPosition(b, o.chunk, o.shifts) * o.first;
      bool more = true;
      for (u i = 0; i < per; i++) {
        // the item orders' definitions: Mbar position mm, slabs s0 and s1
        u w = l * per + i, mm, s0, s1;
        bool want = w < (u)n;
        if (a.itemOrder == 1) {
          s0 = l % ns0; s1 = l / ns0 % ns1; mm = l / ns0 / ns1 * per + i;
          want = l < groups && mm < (u)a.volMbar;
        } else {
          if (a.itemOrder == 2) {
            const u chunk = a.xcdChunk && !a.xcdGroup ? a.xcdChunk : o.blocks, x = l / chunk;
            w = x * chunk * per + (l - x * chunk) + i * chunk;
            want = w < (u)n;
          }
          s0 = w % ns0; s1 = w / ns0 % ns1; mm = w / ns0 / ns1;
        }
        u c, m, in, out;
        const bool some = more && (per == 1 ? cutt::packedWalkSlabs<true>(first, 0, o.shifts, o.items, o.num[0], o.mul[0], o.num[1], o.mul[1], o, c, m, in, out)
                                            : cutt::packedWalkSlabs<false>(first + i * o.stepN, i, o.shifts, o.items, o.num[0], o.mul[0], o.num[1], o.mul[1], o, c, m, in, out));
        CHECK(some == want);
        more = some;
        if (!some) continue;
        cutt::packedWalkMbar(o, m, in, out);
        const size_t id = ((size_t)mm * ns1 + s1) * ns0 + s0;
        CHECK(!seen[id]); seen[id] = 1;
        u wantIn = 0, wantOut = 0;
        const u s[2] = {s0, s1};
        for (int k = 0; k < 2; k++) {
          const cuttHipSplitRank& sr = a.split[k];
          const u at = s[k] * sr.slabFloor + std::min<u>(s[k], sr.slabRem);
          wantIn += at * sr.strideIn; wantOut += at * sr.strideOut;
        }
        for (int k = 0; k < a.mbar.n; k++) {
          wantIn += mm % a.mbar.d[k].extent * a.mbar.d[k].strideIn; wantOut += mm % a.mbar.d[k].extent * a.mbar.d[k].strideOut;
          mm /= a.mbar.d[k].extent;
        }
        CHECK(c == (s0 < (u)a.split[0].slabRem ? 1u : 0u) + (s1 < (u)a.split[1].slabRem ? 2u : 0u) && in == wantIn && out == wantOut);
        items++;
      }
    }
    for (char x : seen) CHECK(x);
    // forms that stay with the general kernel
    if (a.elemSize == 8 && a.itemsPerBlock > 1) { cuttHipPackedArgs b = a; b.numThreads = 832; cuttHipFinishPackedWalk(&b); CHECK(b.walk.blocks == 0); }
    cuttHipPackedArgs b = a; b.itemsPerBlock = 3; b.elemsPerThread = 2; cuttHipFinishPackedWalk(&b); CHECK(b.walk.blocks == 0);
    b = a; b.wideOffsets = 1; cuttHipFinishPackedWalk(&b); CHECK(b.walk.blocks == 0);
    b = a; b.mbar.n = CUTT_PACKED_RANKS + 1; cuttHipFinishPackedWalk(&b); CHECK(b.walk.blocks == 0);
    b = a; b.cls[0].shIdx = nullptr; cuttHipFinishPackedWalk(&b); CHECK(b.walk.blocks == 0);
  }
  printf("ok %ld %ld\n", items, classes);
  return 0;
}
"""


def test_items_and_tables(tmp_path):
    src = tmp_path / "walk.cpp"
    src.write_text(PROGRAM)
    csrc = os.path.join(ROOT, "cutt_amd", "csrc")
    exe = str(tmp_path / "walk")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-include", "algorithm", "-I" + csrc, str(src), os.path.join(csrc, "layer_math.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout + out.stderr


def test_kernel_instances_that_can_be_launched():
    # (a loop over blocks of fewer than four elements per lane has no walk: the general kernel takes it)
    names = subprocess.check_output(["nm", "-C", os.path.join(ROOT, "cutt_amd", "libcutt.so")], text=True)
    for kernel, elems in (("packedOnceKernel", {4: {1, 2, 4, 8, 16}, 8: {1, 2, 4, 8}}), ("packedLoopKernel", {4: {4, 8, 16}, 8: {4, 8}})):
        for size, name in ((4, "unsigned int"), (8, "unsigned long")):
            found = re.findall(kernel + "<%s, (\\d+), (\\d)>" % name, names)
            assert set(found) == {(str(e), str(p)) for e in elems[size] for p in range(4)}, (kernel, size)
