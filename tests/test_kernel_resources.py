"""No kernel of the row library spills registers or uses scratch memory, read from the
metadata of the code objects built here."""
import shutil
import subprocess
from pathlib import Path

import pytest

from origami_amd.build_native import LIB_PATH

ROCM = Path("/opt/rocm/llvm/bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _tool(name):
    return shutil.which(name) or (str(ROCM / name) if (ROCM / name).exists() else None)


def _code_objects(data):
    """The device ELFs of the offload bundles in a linked library."""
    at = data.find(MAGIC)
    while at >= 0:
        cursor = at + len(MAGIC) + 8
        for _ in range(int.from_bytes(data[at + len(MAGIC):cursor], "little")):
            offset, size, name = (int.from_bytes(data[cursor + 8 * i:cursor + 8 * i + 8], "little")
                                  for i in range(3))
            cursor += 24 + name
            if size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 1)


def test_no_scratch(tmp_path):
    readelf = _tool("llvm-readelf")
    if readelf is None or not LIB_PATH.exists():
        pytest.skip("no llvm-readelf or library")
    kernels = {}
    for i, elf in enumerate(_code_objects(LIB_PATH.read_bytes())):
        path = tmp_path / f"{i}.elf"
        path.write_bytes(elf)
        notes = subprocess.run([readelf, "--notes", str(path)], check=True, capture_output=True,
                               text=True).stdout
        scratch = 0
        for line in notes.splitlines():
            key, _, value = line.strip().lstrip("- ").partition(":")
            if key == ".private_segment_fixed_size":
                scratch = int(value)
            elif key == ".symbol":
                name = value.strip()
            elif key == ".vgpr_spill_count":
                kernels[name] = (scratch, int(value))
    assert any("rows_unpack" in k for k in kernels) and any("rows_pack" in k for k in kernels)
    assert {k: v for k, v in kernels.items() if v != (0, 0)} == {}
