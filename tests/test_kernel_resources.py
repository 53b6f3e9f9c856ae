"""No kernel of the built library keeps registers in memory: the grouped GEMMs and the quantisers are laid out to the
register file, and what does not fit is written and read back by every thread."""
import os
import re
import struct
import subprocess

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
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


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_loops_of_higher_row_tiles_begin_a_cache_line(tmp_path):
    """row_tiles_kernel<.., EITHER = true>: the place of a step's first instruction is worth 2 % of it and must not hang on the code in front."""
    from atorch_amd._lib import LIB_PATH

    loops = {}
    for i, obj in enumerate(_code_objects(LIB_PATH)):
        file = tmp_path / f"{i}.co"
        file.write_bytes(obj)
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(file)], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"\n(?=[0-9a-f]+ <)", listing):
            name = re.match(r"[0-9a-f]+ <(\S*row_tiles_kernel\S*Lb1EEEv\S*)>:", kernel)
            if not name:
                continue
            code = [(int(m[3], 16), m[1], m[2]) for m in re.finditer(r"^\t(\S+)(.*?)//\s*([0-9A-F]+):", kernel, re.M)]
            products = [at for at, op, _ in code if "mfma" in op]
            steps = []  # backward branches over the products of a step or two
            for at, op, args in code:
                if op.startswith(("s_cbranch", "s_branch")) and int(args.split()[0]) >= 1 << 15:
                    to = at + 4 + 4 * (int(args.split()[0]) - (1 << 16))
                    if at - to < 6300 and sum(to <= x <= at for x in products) in (16, 18, 32):
                        steps.append((to, at))
            loops[name[1]] = {to for to, _ in steps if not any(t < to < at for t, at in steps)}
    assert len(loops) == 8 and all(len(of) == 3 for of in loops.values())  # with more rows, without, and the form of 256 rows
    assert all(to % 64 == 0 for of in loops.values() for to in of), loops
