"""An MFMA may not read a vector register sooner than two wait states after a vector instruction wrote it (hardware does not
wait; the compiler puts the distance in, for instructions that it chose itself).  The bf16 conversions of the large-tile
contraction feed MFMAs directly: their distance in the built library is checked here, from its disassembly."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin:" + os.environ.get("PATH", ""))
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(path):
    """The gfx950 code objects of a library: every offload bundle lists (offset, size, target) of its parts."""
    data = open(path, "rb").read()
    for at in (m.start() for m in re.finditer(MAGIC, data)):
        pos = at + len(MAGIC)
        count, = struct.unpack_from("<Q", data, pos)
        pos += 8
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", data, pos)
            target = data[pos + 24:pos + 24 + name]
            pos += 24 + name
            if b"gfx950" in target and size:
                yield data[at + offset:at + offset + size]


def _registers(operand):
    found = re.fullmatch(r"v\[(\d+):(\d+)\]|v(\d+)", operand)
    if not found:
        return ()
    first, last, single = found.groups()
    return (int(single),) if single else range(int(first), int(last) + 1)


def short_waits(lines):
    """Lines of MFMAs that read a register fewer than two wait states after a bf16 conversion wrote it, in program order, and
    the number of conversions."""
    since, bad, conversions = {}, [], 0
    for line in lines:
        text = line.split("//")[0].strip()
        if not text or text.endswith(":"):
            continue
        op, _, rest = text.partition(" ")
        operands = [part.strip() for part in rest.split(", ")]
        if op.startswith("v_mfma"):
            if any(since.get(r, 2) < 2 for operand in operands[1:3] for r in _registers(operand)):
                bad.append(text)
        states = int(operands[0], 0) + 1 if op == "s_nop" else 1
        since = {r: n + states for r, n in since.items() if n + states < 2}
        if op.startswith("v_cvt_pk_bf16"):
            conversions += 1
            since[_registers(operands[0])[0]] = 0
    return bad, conversions


def test_the_check_sees_a_missing_wait():
    program = ["v_cvt_pk_bf16_f32 v5, v1, v2", "v_add_f32_e32 v9, v9, v9", "v_mfma_f32_32x32x16_bf16 v[16:31], v[4:7], v[8:11], v[16:31]"]
    assert len(short_waits(program)[0]) == 1
    assert not short_waits(program[:2] + ["s_nop 0"] + program[2:])[0]


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
def test_conversions_of_the_built_library_keep_their_distance(tmp_path):
    total = 0
    for k, code in enumerate(_code_objects(os.path.join(ROOT, "aihwkit_amd", "lib", "librpu_amd.so"))):
        if b"k_mvm_big" not in code:
            continue
        path = tmp_path / f"{k}.co"
        path.write_bytes(code)
        run = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(path)], capture_output=True,
                             text=True, check=True, timeout=300)
        bad, conversions = short_waits(run.stdout.splitlines())
        assert not bad, bad[:5]
        total += conversions
    assert total > 100
