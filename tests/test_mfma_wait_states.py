"""The compiled kernels keep the matrix instructions' wait states on every path.

Hardware does not hold back an instruction that reads the result of a matrix instruction too early: it gets the old value.
The compiler puts wait states in between (s_nop, or other instructions), but where a branch follows a matrix instruction and the
result is first read at the branch's target, it has been seen to count the way that falls through and to leave a single one on
the way that branches.  These checks walk every path through the disassembly of the library that was built here."""
import os
import re
import shutil
import subprocess

import pytest

import innova_amd as ia

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
# wait states, as the compiler itself leaves them in straight code on gfx950: from a matrix instruction to a reader or writer of its
# result; to a writer of the registers that it adds to; from a vector instruction to a matrix instruction that reads its result
RESULT = {"16x16x32_f16": 8, "16x16x64_i8": 8, "32x32x16_bf16": 12}
ADDEND = {"16x16x32_f16": 3, "16x16x64_i8": 3, "32x32x16_bf16": 7}
VECTOR_TO_MATRIX = 2

_REG = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")
_NO_RESULT = re.compile(r"v_cmp|v_readlane|v_readfirstlane|v_nop|s_|ds_write|ds_add|(global|buffer|flat|scratch)_(store|atomic)")


def _regs(text):
    out = set()
    for kind, first, last, only in _REG.findall(text):
        out.update((kind, i) for i in range(int(first or only), int(last or only) + 1))
    return out


class Instr:
    def __init__(self, text, target):
        self.name, _, rest = text.partition(" ")
        ops = rest.split(",")
        self.matrix = self.name.startswith("v_mfma")
        self.target = target                       # of a branch: index in the function
        self.ops = [_regs(o) for o in ops]
        self.all = set().union(*self.ops)
        self.written = set() if _NO_RESULT.match(self.name) else self.ops[0] | (self.ops[1] if "swap" in self.name else set())
        self.states = int(ops[0], 0) + 1 if self.name == "s_nop" else 1


def reachable(code, start, limit):
    """(index, wait states passed) of everything that can run within `limit` wait states behind `start`."""
    seen, todo = {}, [(start + 1, 0)]
    while todo:
        i, passed = todo.pop()
        while i is not None and i < len(code) and passed < seen.get(i, limit):
            seen[i] = passed
            c = code[i]
            passed += c.states
            if c.name == "s_endpgm" or c.name.startswith(("s_setpc", "s_swappc")):
                break
            if c.name.startswith("s_cbranch"):
                todo.append((c.target, passed))
            i = c.target if c.name == "s_branch" else i + 1
    return seen.items()


def violations(code):
    """(index of the earlier instruction, index of the later one, wait states between them) wherever these are too few."""
    out = []
    for i, c in enumerate(code):
        if c.matrix:
            shape = next(k for k in RESULT if k in c.name)
            result, addend, wait, hold = c.ops[0], c.ops[3], RESULT[shape], ADDEND[shape]
            for j, passed in reachable(code, i, max(wait, hold)):
                d = code[j]
                if d.matrix:                       # sums may be handed on from one matrix instruction to the next
                    early = (d.ops[1] | d.ops[2]) & result and passed < wait
                else:
                    early = (d.all & result and passed < wait) or (d.written & addend and passed < hold)
                if early:
                    out.append((i, j, passed))
        elif c.name.startswith("v_") and c.written:
            for j, passed in reachable(code, i, VECTOR_TO_MATRIX):
                if code[j].matrix and c.written & (code[j].ops[1] | code[j].ops[2] | code[j].ops[3]):
                    out.append((i, j, passed))
    return out


def parse_listing(text):
    """{function: [Instr]} of a disassembly with addresses."""
    rows, base, cur = {}, {}, None
    for line in text.splitlines():
        head = re.match(r"([0-9a-f]{16}) <(\S+)>:", line)
        if head:
            cur = head.group(2)
            base[cur], rows[cur] = int(head.group(1), 16), []
        elif cur:
            m = re.match(r"\s+(\S.*?)\s*// ([0-9A-F]{12}):(?:.*<(\S+?)(?:\+0x([0-9a-f]+))?>)?", line)
            if m:
                rows[cur].append(m.groups())
    funcs = {}
    for f, lines in rows.items():
        index = {int(addr, 16): n for n, (_, addr, _, _) in enumerate(lines)}
        funcs[f] = [Instr(t, index.get(base[sym] + int(off or "0", 16)) if sym in base and "branch" in t else None) for t, _, sym, off in lines]
    return funcs


LISTING = """0000000000001000 <k>:
\tv_mfma_f32_16x16x32_f16 v[110:113], v[30:33], v[134:137], v[110:113] // 000000001000: 00000000 00000000
{wait}\ts_cbranch_scc1 8                                     // 000000001008: BF850008 <k+0x2c>
\ts_add_i32 s65, s65, 1                                 // 00000000100C: 00000000
\ts_nop 5                                               // 000000001010: 00000000
\tv_mul_f32_e32 v110, v110, v34                         // 00000000102C: 00000000
\ts_endpgm                                              // 000000001030: 00000000
"""


def test_the_walk_finds_a_read_at_a_branch_target():
    """8 wait states along the code that falls through, 1 along the branch: the pattern of a kernel whose sums lacked the products of
    their last matrix instruction."""
    assert violations(parse_listing(LISTING.format(wait=""))["k"]) == [(0, 4, 1)]
    assert violations(parse_listing(LISTING.format(wait="\ts_nop 6 // 000000001004: 00000000\n"))["k"]) == []


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_every_path_of_the_library_waits_for_matrix_results(tmp_path):
    lib = shutil.copy(ia._lib.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    matrix, bad = 0, []
    for name in sorted(os.listdir(tmp_path)):
        if "gfx950" not in name:
            continue
        text = subprocess.run([OBJDUMP, "-d", name], cwd=tmp_path, check=True, capture_output=True, text=True).stdout
        if "v_mfma" not in text:
            continue
        for f, code in parse_listing(text).items():
            matrix += sum(c.matrix for c in code)
            bad += [(f, code[i].name, code[j].name, n) for i, j, n in violations(code)]
    assert matrix > 1000
    assert not bad, bad[:20]
