"""Wait states before FP64 DPP operands.  A lane broadcast reads a register no sooner than two
wait states after a vector instruction wrote it and five after one wrote EXEC; the compiler's
hazard pass does not look into inline assembly, so the sources place the waits.  Checked in
the sources (no wait that names no register outside dpp_wait) and in the built library's
gfx950 code (this repository's own kernels), along branches too."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "shtnskit.jl_amd", "csrc")
LIB = os.path.join(ROOT, "shtnskit.jl_amd", "libshtk_mi355x.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def _without_comments(text):
    return re.sub(r"//[^\n]*|/\*.*?\*/", "", text, flags=re.S)


def test_no_wait_without_its_registers():
    """A free-standing wait is tied to nothing: the scheduler may move the writers past it."""
    for name in sorted(os.listdir(CSRC)):
        text = _without_comments(open(os.path.join(CSRC, name)).read())
        if name == "shtk_internal.h":
            body = re.search(r"void dpp_wait\(.*?\n}", text, flags=re.S).group(0)
            assert "dpp_written(v)" in body
            text = text.replace(body, "")
        assert not re.search(r'asm volatile\(\s*"s_nop \d+"\s*\)', text), name


def _regs(operand):
    """VGPR numbers of an operand text."""
    m = re.fullmatch(r"-?\|?v\[(\d+):(\d+)\]\|?", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.fullmatch(r"-?\|?v(\d+)\|?", operand)
    return {int(m[1])} if m else set()


class _Code:
    """Instructions of one function: (address, mnemonic, operands), and who jumps where."""

    def __init__(self):
        self.ins, self.at, self.jumps = [], {}, {}

    def add(self, addr, op, args, target):
        self.at[addr] = len(self.ins)
        self.ins.append((op, args))
        if target is not None:
            self.jumps.setdefault(target, []).append(len(self.ins) - 1)

    def index(self):
        self.sources = {self.at[t]: s for t, s in self.jumps.items() if t in self.at}


def _functions(disassembly):
    code, base = None, 0
    for line in disassembly.splitlines():
        m = re.match(r"([0-9a-f]+) <(.+)>:$", line)
        if m:
            if code is not None:
                yield code
            code, base = _Code(), int(m[1], 16)
            continue
        m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):[ 0-9A-F]*(<.*\+0x([0-9a-f]+)>)?", line)
        if m and code is not None:
            args = [a.strip() for a in m[2].split(",")] if m[2] else []
            target = base + int(m[5], 16) if m[5] and m[1].startswith(("s_cbranch", "s_branch")) else None
            code.add(int(m[3], 16), m[1], args, target)
    if code is not None:
        yield code


def _too_close(code, i, regs, waits, states, seen):
    """Whether a vector write of regs lies fewer than `waits` (EXEC: 5) states before instruction i."""
    if states >= 5 or (i, states) in seen:
        return False
    seen.add((i, states))
    before = list(code.sources.get(i, []))
    if i > 0 and code.ins[i - 1][0] not in ("s_branch", "s_endpgm", "s_setpc_b64"):
        before.append(i - 1)
    for p in before:
        op, args = code.ins[p]
        if op.startswith("v_cmpx"):
            return True
        if op.startswith("v_") and args and states < waits and regs & _regs(args[0].split(" ")[0]):
            return True
        step = int(args[0], 0) + 1 if op == "s_nop" else 1
        if _too_close(code, p, regs, waits, states + step, seen):
            return True
    return False


def _broadcasts(code):
    for i, (op, args) in enumerate(code.ins):
        if op.startswith("v_fmac_f64") and any("row_newbcast" in a for a in args):
            yield i, _regs(args[1].split(" ")[0])


@pytest.mark.skipif(not (os.path.exists(LIB) and os.path.exists(OBJDUMP)), reason="needs the built library and llvm-objdump")
def test_built_code_keeps_the_wait_states(tmp_path):
    lib = shutil.copy(LIB, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True)
    total = 0
    for name in sorted(os.listdir(tmp_path)):
        if not name.endswith("gfx950"):
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(tmp_path / name)], check=True,
                              capture_output=True, text=True).stdout
        for code in _functions(text):
            code.index()
            for i, regs in _broadcasts(code):
                assert regs, code.ins[i]
                assert not _too_close(code, i, regs, 2, 0, set()), (name, code.ins[max(0, i - 6):i + 1])
                total += 1
    assert total > 1000


def test_the_check_sees_a_close_write():
    """The check itself, on code written here: straight, past a wait, and around a loop."""
    head = "0000000000001000 <k>:\n"
    fma = "\tv_fmac_f64_dpp v[0:1], v[4:5], v[2:3] row_newbcast:0 row_mask:0xf bank_mask:0xf // %012X: 00\n"
    cases = [
        (["\tv_mov_b32_e32 v5, v9 // %012X: 00\n", "\ts_nop 0 // %012X: 00\n", fma], True),
        (["\tv_mov_b32_e32 v5, v9 // %012X: 00\n", "\ts_nop 1 // %012X: 00\n", fma], False),
        (["\tv_mov_b32_e32 v6, v9 // %012X: 00\n", fma], False),
        ([fma, "\tv_mul_f64 v[4:5], v[6:7], v[8:9] // %012X: 00\n", "\ts_cbranch_scc1 65532 // %012X: 00 <k+0x0>\n"], True),
        (["\tv_cmpx_lt_u32_e32 1, v9 // %012X: 00\n", "\ts_nop 3 // %012X: 00\n", fma], True),
        (["\tv_cmpx_lt_u32_e32 1, v9 // %012X: 00\n", "\ts_nop 4 // %012X: 00\n", fma], False),
    ]
    for lines, close in cases:
        text = head + "".join(l % (0x1000 + 8 * k) for k, l in enumerate(lines))
        (code,) = list(_functions(text))
        code.index()
        found = [_too_close(code, i, r, 2, 0, set()) for i, r in _broadcasts(code)]
        assert len(found) == 1 and found[0] == close, lines
