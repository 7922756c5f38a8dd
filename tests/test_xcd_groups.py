"""Workgroups handed to the XCDs in groups: every logical position is visited exactly once, in both forms the kernels decode
(tile_walk.h: xcdPosition and walkTile, the kernels' own code compiled for the host; no GPU)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>
#include "tile_walk.h"
typedef uint32_t u;
int main() {
  for (u tiles : {1u, 7u, 8u, 63u, 64u, 65u, 127u, 128u, 129u, 1000u, 4097u})
    for (u group = 0; group <= 10; group++) {
      cuttHipTiledArgs a;
      std::memset(&a, 0, sizeof(a));
      a.elemSize = 4; a.tilesM = (int)tiles; a.tilesK = 1; a.volMm = (int)tiles * 64; a.volMk = 64; a.volMbar = 1;
      a.order = 1; a.superM = tiles; a.superK = 1; a.xcdChunk = (tiles + 7) / 8; a.xcdGroup = (int16_t)group;
      cuttHipFinishTileWalk(&a);
      if (a.walk.kind != 1 || a.walk.blocks % 8) return std::printf("walk %u %u\n", tiles, group), 1;
      std::vector<int> seen(a.walk.blocks, 0);
      const cutt::WalkHead head{a.walk.chunk, a.walk.superM, a.walk.stripMul, a.walk.fullMul, a.walk.lastMul, a.walk.shifts};
      for (u b = 0; b < a.walk.blocks; b++) {
        const u l = cutt::xcdPosition(b, a.walk.chunk, group);
        u tm = 0, tk = 0, in, out;
        const bool tile = cutt::walkTile(b, head, cutt::NoMbar{}, tiles, 1, tm, tk, in, out);
        if (tile != (l < tiles) || (tile && (tm != l || tk != 0))) return std::printf("two forms differ: %u %u %u\n", tiles, group, b), 1;
        if (l >= a.walk.blocks || seen[l]++) return std::printf("position %u of %u\n", l, a.walk.blocks), 1;
      }
    }
  std::printf("ok\n");
  return 0;
}
"""


def test_every_position_once(tmp_path):
    src = tmp_path / "groups.cpp"
    src.write_text(PROGRAM)
    exe = str(tmp_path / "groups")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "cutt_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
                           str(src), os.path.join(ROOT, "cutt_amd", "csrc", "layer_math.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout
