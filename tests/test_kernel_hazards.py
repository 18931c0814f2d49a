"""Wait states that the hardware does not insert: two between a vector write of a register and its read through another
lane (a DPP operand, a lane-group swap).  The compiler keeps them between its own instructions, but it does not see what
an inline asm block writes, so the built library's machine code is read back."""

from __future__ import annotations

import re
import struct
import subprocess
from collections import deque
from pathlib import Path

import pytest

from orbitquant_amd import _lib

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
WAIT_STATES = 2
REGISTERS = re.compile(r"v\[(\d+):(\d+)\]|\bv(\d+)\b")


def registers(operand: str) -> set[int]:
    found = set()
    for first, last, single in REGISTERS.findall(operand):
        found |= set(range(int(first), int(last) + 1)) if first else {int(single)}
    return found


def too_close(lines):
    """(write, read) for every read through another lane that follows its operand's write within the wait states."""
    recent = deque(maxlen=WAIT_STATES)   # (an instruction is one wait state or more)
    for line in lines:
        text = line.split("//")[0].strip()
        if line[:1] != "\t" or not text:
            recent.clear()               # another function
            continue
        op, _, rest = text.partition(" ")
        swap = op.startswith("v_permlane")
        if swap or "_dpp" in op:
            operands = rest.split(",")
            need = registers(operands[0]) | registers(operands[1]) if swap else registers(operands[1])
            waited = 0
            for before in reversed(recent):
                before_op, _, before_rest = before.partition(" ")
                if before_op.startswith("v_"):
                    written = before_rest.split(",")[: 2 if before_op.startswith("v_permlane") else 1]
                    if need & set().union(*map(registers, written)):
                        yield before, text
                waited += int(before_rest, 0) + 1 if before_op == "s_nop" else 1
                if waited >= WAIT_STATES:
                    break
        recent.append(text)


def code_objects(library: bytes):
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = library.find(magic)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", library, at + 24)
        entry = at + 32
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", library, entry)
            if b"gfx950" in library[entry + 24 : entry + 24 + name] and size:
                yield library[at + offset : at + offset + size]
            entry += 24 + name
        at = library.find(magic, at + 24)


def test_the_search_finds_what_it_is_for():
    write, swap, dpp = "\tv_add_f32_e32 v3, v1, v2", "\tv_permlane16_swap_b32_e32 v7, v3", "\tv_mov_b32_dpp v9, v3 row_ror:8 row_mask:0xf"
    for read in (swap, dpp):
        assert list(too_close([write, read])) and list(too_close([write, "\ts_mov_b32 s0, s1", read])) and list(too_close([write, "\ts_nop 0", read]))
        assert not list(too_close([write, "\ts_nop 1", read])) and not list(too_close([write, "\ts_nop 0", "\ts_nop 0", read]))
        assert not list(too_close(["\tv_add_f32_e32 v4, v3, v2", read]))
    assert list(too_close([swap, "\tv_permlane32_swap_b32_e32 v7, v8"]))


def test_no_lane_exchange_reads_what_was_written_too_recently(tmp_path):
    if not OBJDUMP.exists():
        pytest.skip("needs llvm-objdump")
    seen = 0
    for i, elf in enumerate(code_objects(_lib.LIB_PATH.read_bytes())):
        if b"rotate_quantize" not in elf and b"token_linear" not in elf:   # (the kernels with asm in front of lane exchanges)
            continue
        path = tmp_path / f"{i}.elf"
        path.write_bytes(elf)
        with subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(path)], stdout=subprocess.PIPE, text=True) as dump:
            assert list(too_close(dump.stdout))[:4] == []
        seen += dump.returncode == 0
    assert seen >= 5
