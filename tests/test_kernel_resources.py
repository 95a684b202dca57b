"""Registers of the last pass, read from the metadata of the built library: the
slot-form kernels keep their values in registers.  (FP64 kernels without a
signature that loaded a cell's values before the row transform spilled up to 149
registers per lane and took up to 1.3 times the time.)

Bound: 16 spilled vector registers per lane, a tenth of the 168 that 3 waves per
SIMD leave each lane."""
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


def _kernels(path, tmp):
    """mangled name -> spilled vector registers per lane"""
    out = {}
    for q, obj in enumerate(_code_objects(path)):
        f = tmp / f"{q}.co"
        f.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
        name = None
        for line in notes.splitlines():
            m = re.match(r"\s+\.name:\s+(_Z\S*k_p5\S*)", line)
            if m:
                name = m.group(1)
            m = re.match(r"\s+\.vgpr_spill_count:\s+(\d+)", line)
            if m and name:
                out[name] = int(m.group(1))
                name = None
    return out


def test_last_pass_slot_form_keeps_its_registers(tmp_path):
    if not shutil.which(READELF):
        pytest.skip("llvm-readelf not found")
    spills = _kernels(mmx._lib.LIB_PATH, tmp_path)
    slot = {}
    for name, n in spills.items():
        # k_p5<T, H, V, ...> and k_p5_batch<T, H, V, E>: V = 1..4 and 7 are the slot form
        m = re.match(r"_ZN3mmx(?:4k_p5|10k_p5_batch)I([df])Li(\d+)ELi(\d)E", name)
        assert m, name
        if m.group(3) in "12347":
            slot[name] = n
    assert len(slot) > 200
    bad = {k: v for k, v in slot.items() if v > 16}
    assert not bad, bad
