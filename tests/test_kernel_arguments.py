"""The argument blocks of the tile kernels.  The command processor leaves them in memory that a workgroup reads line by
line before its first load of tensor data, so a tensor of a few MB feels every line more: the blocks hold what the
kernel reads and no more, and the data pointers behind them start in the line of the last Mbar entries."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include <cstddef>
#include <cstdio>
#include "hip_layer.h"
int main() {
  std::printf("%zu %zu\\n", offsetof(cuttHipTiledArgs, mbar) + sizeof(cuttHipMbar), sizeof(cuttHipTiledArgs));
  std::printf("%zu %zu\\n", offsetof(cuttHipCopyTiles, mbar) + sizeof(cuttHipMbar), sizeof(cuttHipCopyTiles));
}
"""


def test_data_pointers_share_the_line_of_the_last_mbar_entries(tmp_path):
    src = tmp_path / "blocks.cpp"
    src.write_text(PROGRAM)
    exe = str(tmp_path / "blocks")
    subprocess.check_call(["g++", "-std=c++17", "-I" + os.path.join(ROOT, "cutt_amd", "csrc"),
                           "-I" + os.path.join(ROOT, "include"), str(src), "-o", exe])
    for line in subprocess.check_output([exe], text=True).splitlines():
        mbar_end, pointers = map(int, line.split())
        # (both pointers: with the second one in the next line launches of 8-10 us take 2-3 % longer)
        first = (pointers + 7) // 8 * 8
        assert (mbar_end - 1) // 128 == first // 128 == (first + 15) // 128, line


def test_copy_tiles_carry_no_row_table(tmp_path):
    # scalars, the digit list of a free tile order and the Mbar table: 1736 bytes; the 552 bytes of cuttHipRowArgs go to the
    # kernel that reads them
    src = tmp_path / "copy.cpp"
    src.write_text('#include "hip_layer.h"\nstatic_assert(sizeof(cuttHipCopyTiles) == 13 * 4 + sizeof(cuttHipTileDigits) + sizeof(cuttHipMbar), "");\n')
    subprocess.check_call(["g++", "-std=c++17", "-fsyntax-only", "-I" + os.path.join(ROOT, "cutt_amd", "csrc"),
                           "-I" + os.path.join(ROOT, "include"), str(src)])
