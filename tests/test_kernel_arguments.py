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
        assert (mbar_end - 1) // 128 == pointers // 128, line
