"""Registers of the slot-form kernels, read from the metadata of the built library.

The last pass keeps its values in registers: at most 16 spilled vector registers
per lane, a tenth of the 168 that 3 waves per SIMD leave each lane.  (FP64 kernels
without a signature that loaded a cell's values before the row transform spilled
up to 149 and took up to 1.3 times the time.)

Without demag the FP64 kernels of single systems and batches fit 3 waves per SIMD,
168 registers.  (With the stages' k held over the field RK4's final took 173 and
1.25 times the time.)"""
import os
import re
import shutil
import struct
import subprocess

import mmx
import pytest

READELF = os.environ.get("MMX_READELF", "/opt/rocm/llvm/bin/llvm-readelf")


def _code_objects(path):
    data = open(path, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        (n,), p = struct.unpack_from("<Q", data, at + 24), at + 32
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + ln]
            p += 24 + ln
            if b"gfx950" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(magic, at + 24)


def _kernels(path, tmp, name_re, key):
    """mangled name -> the metadata's value of key, for the kernels that match name_re"""
    out = {}
    for q, obj in enumerate(_code_objects(path)):
        f = tmp / f"{q}.co"
        f.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
        name = None
        for line in notes.splitlines():
            m = re.match(r"\s+\.name:\s+(\S+)", line)
            if m and m.group(1).startswith("_Z"):
                name = re.match(name_re, m.group(1))
            m = re.match(rf"\s+\.{key}:\s+(\d+)", line)
            if m and name:
                out[name.string] = (name.groups(), int(m.group(1)))
                name = None
    return out


needs_readelf = pytest.mark.skipif(not shutil.which(READELF), reason="llvm-readelf not found")


@needs_readelf
def test_last_pass_slot_form_keeps_its_registers(tmp_path):
    # k_p5<T, H, V, ...> and k_p5_batch<T, H, V, E>: V = 1..4 and 7 are the slot form
    slot = _kernels(mmx._lib.LIB_PATH, tmp_path, r"_ZN3mmx(?:4k_p5|10k_p5_batch)I([df])Li(\d+)ELi([12347])E",
                    "vgpr_spill_count")
    assert len(slot) > 200
    bad = {k: v for k, v in slot.items() if v[1] > 16}
    assert not bad, bad


@needs_readelf
def test_local_slot_form_fits_three_waves(tmp_path):
    # k_local<T, V, SIG> and k_batch_local<T, V, CPT, BS, SIG, ...>: V = 1..4 and 6
    slot = _kernels(mmx._lib.LIB_PATH, tmp_path, r"_ZN3mmx(?:7k_local|13k_batch_local)IdLi([12346])E", "vgpr_count")
    assert len(slot) > 50
    bad = {k: v for k, v in slot.items() if v[1] > 168}
    assert not bad, bad
