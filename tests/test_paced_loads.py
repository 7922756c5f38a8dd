"""The Tiled kernel for large tensors with ordinary stores, in the machine code of the library built here: a lane's sixteen loads go out in
four groups, and nothing waits for a load before the last one is out.  (Where the compiler keeps the rows in one register tuple, the tests between
the groups merge it with copies that wait for the loads: 1-2.5 % on such tensors.)"""
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


def kernels(tmp_path, pattern):
    """(name, disassembly) of the library's kernels whose mangled name matches."""
    for i, obj in enumerate(code_objects(cutt_amd.lib_path())):
        path = os.path.join(str(tmp_path), "%d.co" % i)
        with open(path, "wb") as f:
            f.write(obj)
        names = subprocess.check_output([LLVM + "llvm-readelf", "-sW", path], text=True)
        for name in sorted(set(re.findall(r"FUNC .* (\S+%s\w+)\n" % pattern, names))):
            yield name, subprocess.check_output([LLVM + "llvm-objdump", "-d", "--disassemble-symbols=" + name, path], text=True)


# (8-byte elements, whose loads nothing else in the kernel looks like; a single rank per axis)
def test_no_load_is_waited_for_before_all_are_out(tmp_path):
    found = list(kernels(tmp_path, "11tiledKernelImLi[0-3]ELi0ELb0EE"))
    assert len(found) == 4
    for name, code in found:
        at = [m.start() for m in re.finditer("global_load_dwordx2", code)]
        assert len(at) == 16 and "vmcnt" not in code[at[0]:at[-1]], name


def test_rows_in_groups_are_one_piece_of_code(tmp_path):
    # (a piece per number of row groups: 3.5-5.5 % on large 4-byte tensors)
    found = list(kernels(tmp_path, "11tiledKernelImLi[0-3]ELi1ELb0EE"))
    assert len(found) == 4
    for name, code in found:
        at = [m.start() for m in re.finditer("global_load_dwordx2", code)]
        assert len(at) == 16 and all("vmcnt(0)" in code[at[k]:at[k + 1]] for k in (3, 7, 11)), name
