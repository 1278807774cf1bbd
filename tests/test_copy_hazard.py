"""The tile copies are inline assembly, which the compiler's hazard recognizer does not look into: a memory instruction must not
read a scalar register within five wait states of the vector instruction that wrote it (the reload of a spilled scalar register
is one).  Looks at every memory instruction of the built library."""

import os
import re
import shutil
import struct
import subprocess

import pytest

from cornstarch_amd import build

LLVM = "/opt/rocm/llvm/bin"
WAIT_STATES = 5


def _code_objects(path, tmp):
    """The gfx950 code objects of a shared library (uncompressed offload bundles, one per source file)."""
    fat = os.path.join(tmp, "fat.bin")
    subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", path, os.path.join(tmp, "copy.so")], check=True)
    data = open(fat, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(magic))
        p = at + len(magic) + 8
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24 : p + 24 + length]
            p += 24 + length
            if b"gfx950" in name and size:
                yield data[at + offset : at + offset + size]
        at = data.find(magic, p)


def _scalars(operand):
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.fullmatch(r"s(\d+)", operand)
    return {int(m[1])} if m else set()


def hazards(lines):
    """(function, instruction) of memory instructions that read a scalar register too soon.  Along the text: a branch only adds
    wait states, a label keeps what lies before it."""
    function, written, copies, found = None, [], 0, []  # written: (wait states since, registers)
    for line in lines:
        if line.endswith(">:\n"):
            function, written = line.split("<")[1][:-3], []
            continue
        words = re.split(r"[ ,\t]+", line.split("//")[0].strip())
        op, operands = words[0], words[1:]
        if not op:
            continue
        if op == "s_nop":
            written = [(w + int(operands[0], 0) + 1, r) for w, r in written]
            continue
        if op.startswith(("buffer_", "global_", "flat_", "scratch_")):
            copies += op.startswith("buffer_load") and "lds" in operands
            read = set().union(*(_scalars(o) for o in operands)) if operands else set()
            found += [(function, line.strip()) for w, r in written if w < WAIT_STATES and r & read]
        written = [(w + 1, r) for w, r in written if w + 1 < WAIT_STATES]
        if op.startswith(("v_readlane", "v_readfirstlane", "v_cmp")):
            written.append((0, _scalars(operands[0])))
        elif op.startswith(("v_add_co", "v_sub_co", "v_subrev_co", "v_addc_co", "v_subb_co", "v_div_scale")):
            written.append((0, _scalars(operands[1])))
    return copies, found


def test_the_scan_finds_a_register_read_too_soon():
    text = ["0 <k>:\n", "\tv_readlane_b32 s6, v1, 3 // x\n", "\ts_nop 0\n", "\tbuffer_load_dwordx4 v1, s[8:11], {} offen lds\n"]
    assert hazards([x.format("s6") for x in text]) == (1, [("k", "buffer_load_dwordx4 v1, s[8:11], s6 offen lds")])
    assert hazards([x.format("s7") for x in text]) == (1, [])
    assert hazards([x.format("s6").replace("s_nop 0", "s_nop 4") for x in text]) == (1, [])


def test_no_copy_reads_a_scalar_register_too_soon(tmp_path):
    if shutil.which("llvm-objdump", path=LLVM) is None or not os.path.exists(build.LIB_PATH):
        pytest.skip("needs the built library and the LLVM tools it is built with")
    total, found = 0, []
    for i, code in enumerate(_code_objects(build.LIB_PATH, str(tmp_path))):
        path = tmp_path / f"{i}.co"
        path.write_bytes(code)
        out = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", str(path)], capture_output=True, text=True, check=True)
        copies, bad = hazards(out.stdout.splitlines(keepends=True))
        total, found = total + copies, found + bad
    assert total > 1000  # the copies are there and the text is understood
    assert found == []
