"""The batch-1 GEMV keeps everything in registers: no form of it that the library holds uses scratch memory."""
import os
import re
import struct
import subprocess

import pytest

from conftest import ROOT

LIB = os.path.join(ROOT, "my-nn-engine_amd", "lib", "libmynn_hip.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def device_code(data):
    """the gfx950 code objects of a library: one bundle per translation unit (magic, count, then offset, size and name of each part)"""
    at = data.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, chars = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24 : pos + 24 + chars]
            pos += 24 + chars
            if b"gfx950" in name and size:
                yield data[at + offset : at + offset + size]
        at = data.find(MAGIC, at + len(MAGIC))


def test_gemv_forms_use_no_scratch_memory(tmp_path):
    if not (os.path.exists(READELF) and os.path.exists(LIB)):
        pytest.skip("needs the built library and llvm-readelf")
    forms = {}
    for code in device_code(open(LIB, "rb").read()):
        if b"dequant_gemv1_kernel" not in code:
            continue
        (tmp_path / "code").write_bytes(code)
        notes = subprocess.check_output([READELF, "--notes", str(tmp_path / "code")], text=True)
        # (the keys of a kernel are in the order of the alphabet: .name before .private_segment_fixed_size)
        for name, scratch in re.findall(r"\.name:\s+(\S*dequant_gemv1_kernel\S*)\n(?:(?!\.name:).)*?\.private_segment_fixed_size:\s+(\d+)", notes, re.S):
            forms[name] = int(scratch)
    assert len(forms) >= 40  # (both types, row lengths of up to 14 chunks, with the norm inside and without)
    assert not {k: v for k, v in forms.items() if v}


def test_tile_products_use_no_scratch_memory(tmp_path):
    """(with the K ranges of a tile one after the other, for captured calls, the loop over the steps was called in two places and no longer
    inlined: fragments and sums in memory, ten times as long)"""
    if not (os.path.exists(READELF) and os.path.exists(LIB)):
        pytest.skip("needs the built library and llvm-readelf")
    forms = {}
    for code in device_code(open(LIB, "rb").read()):
        if b"tile_gemm_kernel" not in code:
            continue
        (tmp_path / "code").write_bytes(code)
        notes = subprocess.check_output([READELF, "--notes", str(tmp_path / "code")], text=True)
        for name, scratch in re.findall(r"\.name:\s+(\S*tile_gemm_kernel\S*)\n(?:(?!\.name:).)*?\.private_segment_fixed_size:\s+(\d+)", notes, re.S):
            forms[name] = int(scratch)
    assert len(forms) >= 200  # (every tile, store and row tail of three kinds, with and without ranges in sequence)
    assert not {k: v for k, v in forms.items() if v}
