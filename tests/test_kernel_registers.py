"""Registers of kernels whose resident waves hang on a few of them, read from the notes of the library built here.  CPU
only."""
import os
import re
import struct
import subprocess

import mstcfd as M

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def kernels(tmp_path):
    """{mangled name: (vector registers, spilled ones)} of the library's gfx950 code objects"""
    data = open(M.LIB_PATH, "rb").read()
    out, pos, magic = {}, 0, b"__CLANG_OFFLOAD_BUNDLE__"
    while (i := data.find(magic, pos)) >= 0:
        p = i + 32
        for _ in range(struct.unpack_from("<Q", data, i + 24)[0]):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + n]
            p += 24 + n
            if b"gfx950" not in target or not size:
                continue
            f = tmp_path / "code.elf"
            f.write_bytes(data[i + off:i + off + size])
            notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
            for entry in re.split(r"\n\s*- \.", notes):
                field = {k: re.search(rf"\.{k}:\s+(\S+)", entry) for k in ("name", "vgpr_count", "vgpr_spill_count")}
                if all(field.values()):
                    out[field["name"][1]] = (int(field["vgpr_count"][1]), int(field["vgpr_spill_count"][1]))
        pos = i + len(magic)
    return out


def test_cell_kernel_of_3d_ausm_keeps_four_waves(tmp_path):
    regs = {k: v for k, v in kernels(tmp_path).items() if re.search(r"k_cellILi3ELi1ELb1EdLi\d+E", k)}
    assert len(regs) == 3, sorted(regs)
    for name, (vgpr, spilled) in regs.items():
        assert vgpr <= 128 and spilled == 0, (name, vgpr, spilled)  # 512 registers per lane and SIMD
