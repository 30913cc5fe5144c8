"""The FP6 prefill kernels spell one matrix instruction out (the row sums of gemm_e2m3.hip), where the compiler inserts no wait states: in the
built code nothing may touch its result, and no vector instruction may write its operands, closer than the hardware allows."""
import pathlib
import re
import shutil
import struct
import subprocess

import pytest

from quarot_amd import _lib

TOOLS = pathlib.Path("/opt/rocm/llvm/bin")
INLINE = "v_mfma_f32_16x16x128_f8f6f4"
RESULT = 11          # wait states from this instruction (4 passes of 4 cycles) to a read or write of its result by another kind of instruction; 8 are needed
SAME = 2             # ... to the next one that accumulates into the same registers
OPERAND = 2          # ... from a vector instruction that writes an operand


def _code_object(kernel, tmp):
    """The gfx950 code object in the library that holds a kernel of this name."""
    fat = tmp / "fat.bin"
    subprocess.run([TOOLS / "llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", _lib.LIB_PATH, tmp / "copy.so"], check=True)
    data = fat.read_bytes()
    for bundle in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at, (count,) = bundle.start() + 32, struct.unpack_from("<Q", data, bundle.start() + 24)
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            name, at = data[at + 24:at + 24 + length], at + 24 + length
            code = data[bundle.start() + offset:bundle.start() + offset + size]
            if b"gfx950" in name and kernel in code:
                out = tmp / "kernels.elf"
                out.write_bytes(code)
                return out
    raise AssertionError(f"no {kernel} in {_lib.LIB_PATH}")


def _registers(text):
    """Vector registers in an operand text."""
    found = set()
    for one, low, high in re.findall(r"\bv(?:(\d+)|\[(\d+):(\d+)\])", text):
        found |= {int(one)} if one else set(range(int(low), int(high) + 1))
    return found


def _functions(listing):
    """{name: [(address, mnemonic, operands, branch target or None)]}"""
    functions, starts = {}, {}
    for line in listing.splitlines():
        head = re.match(r"([0-9a-f]+) <(.+)>:", line)
        if head:
            current = functions.setdefault(head[2], [])
            starts[head[2]] = int(head[1], 16)
            continue
        code = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):[^<]*(?:<(.+?)(?:\+0x([0-9a-f]+))?>)?", line)
        if code:
            target = starts[code[4]] + int(code[5] or "0", 16) if code[4] in starts and code[1].startswith(("s_branch", "s_cbranch")) else None
            current.append((int(code[3], 16), code[1], code[2], target))
    return functions


def _within(function, places, index, states):
    """Instructions that can follow `index` with fewer than so many wait states between, over branches: (index, wait states between)."""
    todo, seen = [(index, 0)], {}
    while todo:
        at, passed = todo.pop()
        _, name, operands, target = function[at]
        if (at, passed) != (index, 0):
            passed += 1 + int(operands, 0) if name == "s_nop" else 1
        if passed >= states or seen.get(at, states) <= passed:
            continue
        seen[at] = passed
        follow = [] if name in ("s_branch", "s_endpgm") or at + 1 == len(function) else [at + 1]
        for following in follow + ([] if target is None else [places[target]]):
            yield following, passed
            todo.append((following, passed))


@pytest.mark.skipif(not shutil.which("llvm-objdump", path=str(TOOLS)), reason="needs the ROCm LLVM tools")
def test_spelled_out_matrix_instruction_keeps_its_distance(tmp_path):
    elf = _code_object(b"gemm_sp256_kernel", tmp_path)
    listing = subprocess.run([TOOLS / "llvm-objdump", "-d", "--mcpu=gfx950", elf], check=True, capture_output=True, text=True).stdout
    seen = 0
    for name, function in _functions(listing).items():
        if "gemm_sp" not in name:
            continue
        places = {entry[0]: i for i, entry in enumerate(function)}
        inline = 0
        for i, (_, op, operands, _) in enumerate(function):
            if op == INLINE:
                inline += 1
                result = _registers(operands.split(", ")[0])
                assert result == _registers(operands.split(", ")[3].split(" ")[0]) and len(result) == 4, operands
                for j, passed in _within(function, places, i, RESULT):
                    other = function[j]
                    if other[1] == INLINE and _registers(other[2].split(", ")[0]) == result:
                        assert passed >= SAME and not result & _registers(", ".join(other[2].split(", ")[1:3])), (name, i, j)
                    else:
                        assert not result & _registers(other[2]), (name, hex(function[i][0]), other)
            elif op.startswith("v_") and not op.startswith(("v_mfma", "v_cmp", "v_readfirstlane", "v_readlane")):
                written = _registers(", ".join(operands.split(", ")[:2]) if "swap" in op else operands.split(", ")[0])
                for j, _ in _within(function, places, i, OPERAND):
                    if function[j][1] == INLINE:
                        assert not written & _registers(", ".join(function[j][2].split(", ")[1:3])), (name, function[i], function[j])
        assert inline > 0, name
        seen += 1
    assert seen == 12
