"""Wait states of the direct global -> LDS loads in the built library.

The assembly blocks of csrc/fa_pipe.h take the address from two
v_readfirstlane_b32. gfx9 wants five wait states between a vector
instruction's write of a scalar register and a memory instruction's read of
it, and one between the write of m0 and the load; the compiler inserts
neither for instructions inside an assembly block. This reads the
disassembly of the kernels that were built here."""
import os
import re
import shutil
import subprocess

import pytest

from tests.conftest import REPO

LIB = os.path.join(REPO, "flash-attention-npu_amd", "fa_mi355x", "lib", "libfa_mi355x.so")
OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
NEED, NEED_M0 = 5, 1
# vector instructions whose second operand is a scalar result (carry, scale flag)
CARRY = re.compile(r"v_(add|sub|subrev|addc|subb|subbrev)_co_|v_div_scale_|v_mad_[ui]64_")


def scalar_regs(operand):
    m = re.fullmatch(r"s(\d+)", operand)
    if m:
        return {int(m.group(1))}
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    return set(range(int(m.group(1)), int(m.group(2)) + 1)) if m else set()


def split(line):
    """(mnemonic, operands) of a disassembly or assembly line, or None."""
    text = line.split("//")[0].strip()
    if not text or text.endswith(":") or not re.match(r"[a-z]+_", text):
        return None
    name, _, rest = text.partition(" ")
    return name, [x.strip() for x in rest.split(",")]


def vector_writes(name, ops):
    if not name.startswith("v_"):
        return set()
    out = scalar_regs(ops[0])
    return out | (scalar_regs(ops[1]) if len(ops) > 1 and CARRY.match(name) else set())


def hazards(lines):
    """(loads seen, [text of each load that comes too early])."""
    code, bad, loads = [], [], 0
    for line in lines:
        ins = split(line)
        if ins is None:
            continue
        name, ops = ins
        if name.startswith("global_load_lds_"):
            loads += 1
            base = set().union(*(scalar_regs(o.split()[0]) for o in ops if o))
            waited = 0
            for pname, pops in reversed(code):
                if waited < NEED and vector_writes(pname, pops) & base:
                    bad.append(f"{line.strip()}: {waited} wait states after {pname} {', '.join(pops)}")
                    break
                if waited < NEED_M0 and pops[0] == "m0":
                    bad.append(f"{line.strip()}: right after m0")
                    break
                waited += int(pops[0], 0) + 1 if pname == "s_nop" else 1
                if waited >= NEED:
                    break
        code.append(ins)
        del code[:-NEED]
    return loads, bad


@pytest.mark.parametrize("between,early", [
    ([], True),
    (["s_mov_b32 m0, s9", "s_nop 0"], True),
    (["s_mov_b32 m0, s9", "s_mov_b64 s[4:5], exec", "s_mov_b64 exec, s[12:13]"], True),
    (["s_mov_b32 m0, s9", "s_mov_b64 s[4:5], exec", "s_mov_b64 exec, s[12:13]", "s_nop 1"], False),
    (["s_nop 3", "s_mov_b32 m0, s9"], True),
    (["s_nop 4"], False),
])
def test_scan_finds_early_loads(between, early):
    lines = ["v_readfirstlane_b32 s7, v1", *between, "global_load_lds_dwordx4 v2, s[6:7] offset:1024 // 0:"]
    loads, bad = hazards(lines)
    assert loads == 1 and len(bad) == early
    other = ["v_readfirstlane_b32 s8, v1", "s_nop 0", "global_load_lds_dwordx4 v2, s[6:7]"]
    assert hazards(other) == (1, [])


def test_built_library(tmp_path):
    if not os.path.exists(LIB) or not os.path.exists(OBJDUMP):
        pytest.skip("needs the built library and ROCm's llvm-objdump")
    lib = shutil.copy(LIB, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    loads, bad = 0, []
    for f in sorted(os.listdir(tmp_path)):
        if "amdgcn" in f:
            asm = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", os.path.join(tmp_path, f)], check=True,
                                 capture_output=True, text=True).stdout
            n, b = hazards(asm.splitlines())
            loads, bad = loads + n, bad + b
    assert loads > 100
    assert not bad, f"{len(bad)} of {loads} loads:\n" + "\n".join(bad[:10])
