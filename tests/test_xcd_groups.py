"""Workgroups handed to the XCDs in groups: every logical position is visited exactly once, in both forms the kernels decode
(tile_order.h: xcdPosition and walkTile; no GPU)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>
#include "hip_layer.h"
typedef uint32_t u;
static u position(u bid, u chunk, u group) {  // as tile_order.h: xcdPosition
  const u q = bid / 8, x = bid % 8;
  if (group) { const u g = group - 1; return ((((q >> g) * 8) + x) << g) + (q & ((1u << g) - 1)); }
  return chunk ? x * chunk + q : bid;
}
static u walked(const cuttHipTileWalk& h, u bid) {  // as tile_order.h: walkTile
  const u xs = (h.shifts >> 15) & 3, g = ((h.shifts >> 17) - 1) & 31, q = bid >> xs;
  return (bid & ((1u << xs) - 1)) * h.chunk + (q & ((1u << g) - 1)) + (((q >> g) << g) << 3);
}
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
      for (u b = 0; b < a.walk.blocks; b++) {
        const u l = position(b, a.walk.chunk, group);
        if (l != walked(a.walk, b)) return std::printf("two forms differ: %u %u %u\n", tiles, group, b), 1;
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
