"""The compiler does not look into inline assembly, so the wait states that gfx950 asks for around it are checked in the built
library: five between a scalar register's write by the vector unit (v_readlane, v_readfirstlane, a compare) and a memory
instruction that reads it, and one between a store of more than eight bytes and the next write of its data registers."""
import os
import re
import subprocess

import pytest

from test_kernel_resources import _code_objects

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def _registers(text, kind):
    found = set()
    for m in re.finditer(rf"\b{kind}\[(\d+):(\d+)\]|\b{kind}(\d+)\b", text):
        found |= {int(m[3])} if m[3] else set(range(int(m[1]), int(m[2]) + 1))
    return found


def _violations(listing):
    """(memory instructions seen, what is too close to one) of a disassembly."""
    seen, bad, name, before = 0, [], "", []  # before: (mnemonic, operands, wait states, scalar registers the vector unit wrote)
    for line in listing.splitlines():
        head = re.match(r"^[0-9a-f]+ <(.+)>:", line)
        text = line.split("//")[0].strip()
        if head:
            name, before = head[1], []
            continue
        if not text or not re.match(r"[a-z]", text):
            continue
        op, _, args = text.partition(" ")
        if re.match(r"(buffer|global|scratch|flat)_", op):
            seen += 1
            distance = 0
            for _, _, states, wrote in reversed(before):
                if distance >= 5:
                    break
                if wrote & _registers(args, "s"):
                    bad.append((name, text, f"scalar register written {distance} wait states earlier"))
                distance += states
        if before and re.match(r"(buffer|global)_store_dwordx[34]", before[-1][0]) and op.startswith("v_"):
            operands = before[-1][1].split(",")
            data = _registers(operands[0] if before[-1][0].startswith("buffer") else operands[1], "v")
            written = args.split(",")[: 2 if "swap" in op else 1]
            if not re.match(r"v_(cmp|read)", op) and data & _registers(",".join(written), "v"):
                bad.append((name, text, "data of the store in front"))
        scalar = op in ("v_readlane_b32", "v_readfirstlane_b32") or (op.startswith("v_cmp") and args.strip().startswith("s["))
        before = before[-11:] + [(op, args, int(args) + 1 if op == "s_nop" else 1, _registers(args.split(",")[0], "s") if scalar else set())]
    return seen, bad


def test_the_check_finds_what_it_looks_for():
    near = "0000 <k>:\n v_readlane_b32 s4, v1, 3\n s_nop 3\n buffer_load_dword v0, s[4:7], 0 offen lds\n"
    assert len(_violations(near)[1]) == 1 and not _violations(near.replace("s_nop 3", "s_nop 4"))[1]
    store = "0000 <k>:\n buffer_store_dwordx4 v[2:5], v0, s[4:7], 0 offen\n v_mov_b32_e32 v3, v9\n"
    assert len(_violations(store)[1]) == 1 and not _violations(store.replace("\n v_mov", "\n s_nop 1\n v_mov"))[1]


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_wait_states_around_inline_assembly(tmp_path):
    from atorch_amd._lib import LIB_PATH

    seen, bad = 0, []
    for i, obj in enumerate(_code_objects(LIB_PATH)):
        file = tmp_path / f"{i}.co"
        file.write_bytes(obj)
        n, b = _violations(subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(file)], capture_output=True, text=True, check=True).stdout)
        seen, bad = seen + n, bad + b
    assert seen > 1000 and not bad, bad[:5]
