"""What the compiled device code asks of the card, read from the built library
(no GPU): the decode tile kernels keep their operands in registers."""
import os
import re
import struct
import subprocess

import pytest

from ramvamp_amd import _lib as L

READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")


def code_objects():
    """The gfx950 code objects of the library's offload bundles."""
    data = open(L.LIB_PATH, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    for m in re.finditer(magic, data):
        at = m.start() + len(magic)
        (n,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(n):
            off, size, name = struct.unpack_from("<QQQ", data, at)
            triple = data[at + 24:at + 24 + name]
            at += 24 + name
            if b"gfx950" in triple and size:
                yield data[m.start() + off:m.start() + off + size]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Kernel name -> its metadata's integers."""
    if not os.path.exists(L.LIB_PATH):
        pytest.fail(f"{L.LIB_PATH} not built (run __graft_entry__.build())")
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    path = tmp_path_factory.mktemp("code") / "object"
    found = {}
    for obj in code_objects():
        path.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for entry in notes.split("\n  - ")[1:]:
            name = re.findall(r"^\s*\.name:\s+(_Z\S+)", entry, re.M)
            if name:
                found[name[-1]] = {k: int(v) for k, v in re.findall(r"^\s*\.(\w+):\s+(\d+)$", entry, re.M)}
    return found


def test_the_decode_tile_kernels_do_not_spill(kernels):
    tiles = {k: v for k, v in kernels.items() if "decode_tile_kernel" in k}
    assert len(tiles) >= 40
    for name, v in tiles.items():
        assert v["vgpr_spill_count"] == 0 and v["private_segment_fixed_size"] == 0, name
