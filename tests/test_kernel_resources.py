"""No kernel of the built library keeps registers in memory: the grouped GEMMs and the quantisers are laid out to the
register file, and what does not fit is written and read back by every thread."""
import os
import re
import struct
import subprocess

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(path):
    """The gfx950 code objects inside a library: a bundle per source file, each a table of (offset, size, target)."""
    data = open(path, "rb").read()
    for start in (m.start() for m in re.finditer(MAGIC, data)):
        at = start + len(MAGIC)
        (count,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            target = data[at + 24 : at + 24 + length]
            at += 24 + length
            if target.endswith(b"gfx950") and size:
                yield data[start + offset : start + offset + size]


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_no_kernel_keeps_registers_in_memory(tmp_path):
    from atorch_amd._lib import LIB_PATH

    kernels, scratch = 0, []
    for i, obj in enumerate(_code_objects(LIB_PATH)):
        file = tmp_path / f"{i}.co"
        file.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(file)], capture_output=True, text=True, check=True).stdout
        for block in notes.split("\n  - ")[1:]:
            field = lambda f: re.search(rf"\.{f}: +(\S+)", block)  # noqa: E731
            if field("private_segment_fixed_size") is None:
                continue
            kernels += 1
            if int(field("vgpr_spill_count").group(1)):
                scratch.append((field("symbol").group(1), field("private_segment_fixed_size").group(1)))
    assert kernels > 10
    assert not scratch, f"spilled registers, bytes per thread: {scratch}"
