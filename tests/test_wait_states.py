"""Wait states that gfx950 leaves to the program, in the built library's own kernels.

A vector ALU instruction that writes a scalar register needs five wait states before a vector
memory instruction reads it; the hardware does not check. The compiler keeps the distance for the
instructions it knows, not for those of inline assembly (the direct loads into LDS), so the
disassembly of the kernels is checked here, along every path.
"""
import os
import re
import shutil
import subprocess

import pytest

from cachepotato_amd.build import ARCH, LIB

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
pytestmark = pytest.mark.skipif(not (os.path.exists(OBJDUMP) and os.path.exists(LIB)),
                                reason="llvm-objdump or the built library is absent")
NEEDED = 5
LINE = re.compile(r"^\s+(\S+)(?:\s+(.*?))?\s*// ([0-9A-F]+): (.*)$")


def sgprs(text):
    out = {1000, 1001} if "vcc" in text else set()
    for one, lo, hi in re.findall(r"(?<![a-z0-9_])s(?:(\d+)\b|\[(\d+):(\d+)\])", text):
        out.update(range(int(one or lo), int(one or hi) + 1))
    return out


def kernels(path):
    """(name, [(op, operands, address, branch target or None)])"""
    text = subprocess.run([OBJDUMP, "-d", path], capture_output=True, text=True, check=True).stdout
    out = []
    for line in text.splitlines():
        m = re.match(r"^[0-9a-f]+ <(.+)>:$", line)
        if m:
            out.append((m.group(1), []))
            continue
        m = LINE.match(line)
        if m and out:
            op, args, addr, rest = m.group(1), m.group(2) or "", int(m.group(3), 16), m.group(4)
            b = re.search(r"<(.+?)(?:\+0x([0-9a-f]+))?>", rest) if op.startswith(("s_cbranch", "s_branch")) else None
            out[-1][1].append((op, args, addr, (b.group(1), int(b.group(2) or "0", 16)) if b else None))
    return out


def scalar_written(op, args):
    """the scalar registers that a vector ALU instruction writes"""
    ops = re.split(r",\s*(?![^\[]*\])", args)
    if re.match(r"v_(readfirstlane|readlane|cmp)", op):
        return sgprs(ops[0])
    if op.startswith("v_") and re.search(r"_co_|div_scale", op):
        return sgprs(ops[1])
    return set()


def close_reads(name, ins):
    """reads by a vector memory instruction fewer than NEEDED wait states after the write"""
    start = ins[0][2] if ins else 0
    at = {i[2]: k for k, i in enumerate(ins)}
    for k, (op, args, addr, _) in enumerate(ins):
        written = scalar_written(op, args)
        if not written:
            continue
        todo, seen = [(k + 1, 0)], set()
        while todo:
            j, waited = todo.pop()
            while j < len(ins) and waited < NEEDED and (j, waited) not in seen:
                seen.add((j, waited))
                o, a, to, branch = ins[j]
                if re.match(r"(global|buffer|flat|scratch)_", o) and written & sgprs(a):
                    yield f"{name}: {op} {args} at {addr:#x}, {o} {a} at {to:#x}: {waited} wait states"
                if branch and branch[0] == name and start + branch[1] in at:
                    todo.append((at[start + branch[1]], waited + 1))
                if o in ("s_branch", "s_endpgm", "s_setpc_b64"):
                    break
                waited += int(a, 0) + 1 if o == "s_nop" else 1
                j += 1


def test_scalar_written_by_vector_alu_then_read_by_vector_memory(tmp_path):
    lib = shutil.copy(LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", lib], capture_output=True, check=True, cwd=tmp_path)
    objs = sorted(p for p in os.listdir(tmp_path) if p.endswith(ARCH))
    assert objs
    direct, found = 0, []
    for o in objs:
        for name, ins in kernels(str(tmp_path / o)):
            direct += sum(op.startswith("global_load_lds") for op, *_ in ins)
            found += close_reads(name, ins)
    assert direct > 100                          # the direct loads are among what was read
    assert not found, "\n".join(found)
