"""What the compiler gave the RMSNorm kernels (CPU; read from the metadata of the
library built here): none keeps a row's worth of registers in scratch memory,
which its row loop would then read and write beside the rows."""

from __future__ import annotations

import re
import shutil
import struct
import subprocess
from pathlib import Path

import pytest

from thundersync_amd import _build

READELF = next((p for p in ("/opt/rocm/llvm/bin/llvm-readelf", shutil.which("llvm-readelf") or "") if p and Path(p).exists()), None)
LIBRARY = _build.HERE / _build.LIB_NAME
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data: bytes):
    """The gfx950 code objects of the offload bundles in a shared library."""
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", data, entry)
            if b"gfx950" in data[entry + 24 : entry + 24 + name] and size:
                yield data[at + offset : at + offset + size]
            entry += 24 + name
        at = data.find(MAGIC, entry)


@pytest.mark.skipif(READELF is None or not LIBRARY.exists(), reason="no llvm-readelf or library")
def test_scratch_memory(tmp_path):
    scratch = {}
    for i, obj in enumerate(code_objects(LIBRARY.read_bytes())):
        if b"rmsnorm" not in obj:
            continue
        path = tmp_path / f"{i}.co"
        path.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"\n\s*- \.a", notes)[1:]:
            name, size = re.search(r"\.name:\s+(\S+)", kernel), re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel)
            if name and size and "rmsnorm" in name[1]:
                scratch[name[1]] = int(size[1])
    assert len(scratch) > 50
    # the fp32 backward of 10 full vectors keeps 27 registers there and is faster for its eight waves a
    # block; 12 kept 284 (512 bytes) and took 1.7 times the time of 16 vectors without
    assert {k: v for k, v in scratch.items() if v > 128} == {}
