"""Registers of the built kernels, as the compiler reports them in the code
objects' metadata: the quantised matrix-core kernels keep everything their K loop
touches in registers (a spill reload waits for every load in flight)."""

import struct
import subprocess
from pathlib import Path

import pytest

from quantaweave_amd import _lib

READELF = Path("/opt/rocm/llvm/bin/llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(blob: bytes):
    """The gfx950 ELF images of the offload bundles in a host library."""
    at = blob.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", blob, at + 24)
        entry = at + 32
        for _ in range(count if count < 16 else 0):  # the magic also occurs as a string of its own
            offset, size, length = struct.unpack_from("<QQQ", blob, entry)
            if length < 256 and b"gfx950" in blob[entry + 24:entry + 24 + length]:
                yield blob[at + offset:at + offset + size]
            entry += 24 + length
        at = blob.find(MAGIC, at + 24)


def test_quantised_kernels_do_not_spill(tmp_path):
    if not READELF.exists() or not _lib.available():
        pytest.skip("needs the built library and llvm-readelf")
    spills = {}
    for i, image in enumerate(code_objects(_lib.LIB_PATH.read_bytes())):
        path = tmp_path / f"{i}.co"
        path.write_bytes(image)
        notes = subprocess.run([str(READELF), "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        name = None
        for line in notes.splitlines():
            key, _, value = line.strip().lstrip("- ").partition(":")
            if key == ".name" and value.strip().startswith("_Z"):
                name = value.strip()
            elif key == ".vgpr_spill_count" and name is not None:
                spills[name] = int(value)
    checked = {n: v for n, v in spills.items() if "ffn_quant_kernel" in n or "quant_split_kernel" in n}
    assert len(checked) >= 48
    assert not {n: v for n, v in checked.items() if v}
