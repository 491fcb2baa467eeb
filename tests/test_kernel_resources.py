"""Register use of the built kernels, read from the metadata of the library's own code objects (no GPU)."""

from __future__ import annotations

import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tts-inference_amd", "qtts_amd", "libqtts_amd.so")
READELF = next((p for p in ("/opt/rocm/llvm/bin/llvm-readelf", shutil.which("llvm-readelf")) if p and os.path.exists(p)), None)
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _spills(tmp_path) -> dict[str, int]:
    """Vector registers that each kernel spills to scratch."""
    with open(LIB, "rb") as f:
        data = f.read()
    out = {}
    at = data.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            target = data[entry + 24:entry + 24 + length]
            entry += 24 + length
            if b"gfx950" not in target:
                continue
            obj = tmp_path / "code_object"
            obj.write_bytes(data[at + offset:at + offset + size])
            notes = subprocess.run([READELF, "--notes", str(obj)], check=True, capture_output=True, text=True).stdout
            for kernel in notes.split("- .agpr_count")[1:]:
                name = re.search(r"\.name:\s+(\S+)", kernel).group(1)
                out[name] = int(re.search(r"\.vgpr_spill_count:\s+(\d+)", kernel).group(1))
        at = data.find(MAGIC, at + len(MAGIC))
    return out


def test_kernels_keep_their_registers(tmp_path):
    """No kernel spills more than the few registers that the largest W8A8 tile with read-ahead is left with (its two
    operand sets and accumulators fill the file): a spill in a K loop is memory traffic on every stage."""
    if not READELF or not os.path.exists(LIB):
        pytest.skip("no built library or no llvm-readelf")
    spills = _spills(tmp_path)
    assert len(spills) > 1000
    assert not {name: n for name, n in spills.items() if n > 4}
