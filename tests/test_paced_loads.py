"""The instance of the Tiled kernel that paces its loads, in the machine code of the library built here: the four row groups wait
for each other, the four loads of a group go out back to back.  A test per row instead of one per group leaves a branch before every
load (large 8-byte tensors with ordinary stores took 1-2.5 % longer)."""
import os
import re
import struct
import subprocess

import cutt_amd

LLVM = "/opt/rocm/llvm/bin/"


def code_objects(path):
    data = open(path, "rb").read()
    at = data.find(b"\x7fELF", 1)
    while at >= 0:
        table, = struct.unpack_from("<Q", data, at + 40)
        size, count = struct.unpack_from("<HH", data, at + 58)
        if struct.unpack_from("<H", data, at + 18)[0] == 224:  # EM_AMDGPU
            yield data[at:at + table + size * count]
        at = data.find(b"\x7fELF", at + 1)


def test_loads_of_a_row_group_go_out_back_to_back(tmp_path):
    checked = 0
    for i, obj in enumerate(code_objects(cutt_amd.lib_path())):
        path = os.path.join(str(tmp_path), "%d.co" % i)
        with open(path, "wb") as f:
            f.write(obj)
        names = subprocess.check_output([LLVM + "llvm-readelf", "-sW", path], text=True)
        # 8-byte elements, ordinary stores, rows not in groups, a single rank per axis
        for name in sorted(set(re.findall(r"FUNC .* (\S+11tiledKernelImLi[01]ELb0ELb0EE\w+)\n", names))):
            code = subprocess.check_output([LLVM + "llvm-objdump", "-d", "--disassemble-symbols=" + name, path], text=True)
            straight = re.split(r"\n\s+s_c?branch\S*", code)
            loads = [len(re.findall(r"global_load_dwordx2", piece)) for piece in straight]
            assert [n for n in loads if n] == [4, 4, 4, 4], (name, loads)
            checked += 1
    assert checked == 2
