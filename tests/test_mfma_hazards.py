"""The MFMAs that the row-adaptive GEMM kernel writes in assembly (mma_vgpr in csrc/gmm_rows_kernel.h): the compiler knows neither
how long their operands have to have been written nor how long their results take, and inserts no wait states.  The built
kernels are read back and each of these instructions is checked: two wait states before it in which no vector
instruction writes what it reads, and none that touches its result before that is there."""
import os
import re
import shutil
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hetu-galvatron_amd", "_lib",
                   "libgalvatron_moe.so")
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
BEFORE = 2   # wait states between a vector instruction's result and an MFMA that reads it
AFTER = 18   # between an MFMA's result (up to 16 passes) and an instruction that reads or overwrites it
LINE = re.compile(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-F]+): ([0-9A-F]{8})")
FUNCTION = re.compile(r"^[0-9a-f]+ <(\S+)>:")


def code_objects():
    """The gfx950 code objects in the library that hold the kernel."""
    data, at = open(LIB, "rb").read(), 0
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        pos = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            pos += 24 + length
            code = data[at + offset:at + offset + size]
            if b"gfx950" in data[pos - length:pos] and b"gmm_rows_kernel" in code:
                yield code
        at += 32


def registers(operand):
    """Vector registers named by an operand, accumulation registers not among them."""
    m = re.match(r"^-?\|?v(?:\[(\d+):(\d+)\]|(\d+))", operand)
    if not m:
        return frozenset()
    low, high = (int(m[1]), int(m[2])) if m[1] else (int(m[3]), int(m[3]))
    return frozenset(range(low, high + 1))


def functions(text):
    """name -> instructions: (mnemonic, operands, address, branch target or None)"""
    found, now = {}, None
    for line in text.splitlines():
        if m := FUNCTION.match(line):
            now = found.setdefault(m[1], [])
        elif now is not None and (m := LINE.match(line)):
            address, target = int(m[3], 16), None
            if m[1].startswith(("s_cbranch", "s_branch")):
                offset = int(m[4], 16) & 0xffff
                target = address + 4 + 4 * (offset - 0x10000 if offset & 0x8000 else offset)
            now.append((m[1], [o.strip() for o in m[2].split(",")], address, target))
    return found


def states(op):
    return int(op[1][0], 0) + 1 if op[0] == "s_nop" else 1


def paths(ops, index, i, left):
    """Instructions that may follow ops[i] within `left` wait states, branches taken and not."""
    while i + 1 < len(ops) and left > 0:
        name, _, _, target = ops[i]
        if target in index and name.startswith("s_cbranch"):
            yield from paths(ops, index, index[target] - 1, left)
        i = index[target] - 1 if name == "s_branch" and target in index else i
        i += 1
        yield ops[i]
        left -= states(ops[i])
        if ops[i][0].startswith(("s_endpgm", "s_setpc")):
            return


def faults(ops):
    index = {op[2]: i for i, op in enumerate(ops)}
    targets = {op[3] for op in ops}
    for i, (name, operands, address, _) in enumerate(ops):
        if not name.startswith("v_mfma") or not registers(operands[0]):
            continue
        result, read = registers(operands[0]), frozenset().union(*map(registers, operands[1:4]))
        left, j = BEFORE, i - 1
        while left > 0 and j >= 0:
            before = ops[j]
            if before[3] is not None or not before[0].startswith(("s_nop", "v_", "s_", "ds_", "buffer_", "global_", "scratch_")):
                yield "0x%x: reached by a branch %d wait states before" % (address, BEFORE - left)
            if before[0].startswith("v_") and not before[0].startswith("v_mfma") and registers(before[1][0]) & read:
                yield "0x%x: %s writes an operand right before" % (address, before[0])
            left -= states(before)
            j -= 1
        if targets & set(range(address - 4, address + 1)):
            yield "0x%x: a branch leads right to it" % address
        for after in paths(ops, index, i, AFTER):
            if after[0].startswith("v_mfma"):
                same = registers(after[1][0]) == result and registers(after[1][3]) == result
                used = registers(after[1][1]) | registers(after[1][2])
                bad = used & result or (not same and (registers(after[1][0]) | registers(after[1][3])) & result)
            else:
                bad = any(registers(o) & result for o in after[1])
            if bad:
                yield "0x%x: %s touches its result within %d wait states" % (address, after[0], AFTER)


@pytest.fixture(scope="module")
def kernels():
    if not (os.path.exists(LIB) and os.path.exists(OBJDUMP)):
        pytest.skip("needs the built library and llvm-objdump")
    found = {}
    for code in code_objects():
        text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", "-"], input=code, capture_output=True, check=True).stdout
        found.update({k: v for k, v in functions(text.decode()).items() if "gmm_rows_kernel" in k})
    return found


def test_assembly_mfmas_keep_their_wait_states(kernels):
    assert len(kernels) == 16  # two types, eight forms
    for name, ops in kernels.items():
        mine = [o for o in ops if o[0].startswith("v_mfma") and registers(o[1][0])]
        assert len(mine) >= 48, name  # four K steps of 4 (320 rows) and 8 (384 rows) of them
        found = list(faults(ops))
        assert not found, (name, len(found), found[:4])


def test_the_check_finds_what_it_is_for():
    ops = [("v_mov_b32_e32", ["v2", "0"], 0, None), ("v_mfma_f32_32x32x16_bf16", ["v[16:31]", "v[0:3]", "v[4:7]", "v[16:31]"], 4, None),
           ("s_nop", ["7"], 12, None), ("ds_write_b64", ["v40", "v[30:31]"], 16, None), ("s_endpgm", [""], 24, None)]
    found = list(faults(ops))
    assert len(found) == 2 and "v_mov_b32_e32 writes" in found[0] and "ds_write_b64 touches" in found[1], found
