"""Memory-to-LDS transfers of the built kernels (no GPU needed): the compiler does not add the wait states of gfx950
around an instruction written in inline asm, so the disassembly of the library is checked for them.  One state is
needed between a scalar write of m0 and a transfer, five between a vector write of a scalar register and a memory
instruction that reads it."""
import os
import re
import shutil
import subprocess

import pytest

import xqbind as xb

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")


def scalar_regs(text):
    for a, b, c in re.findall(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b", text):
        yield from range(int(a), int(b) + 1) if a else [int(c)]


def findings(lines):
    """(transfers, those without a state behind the write of m0, those that read a register a vector instruction wrote
    less than five states before, other uses of m0 in a function with transfers), in program order."""
    transfers, close, early, other = 0, [], [], []
    fn, since, m0, uses, here = "", {}, 99, [], 0
    for raw in list(lines) + ["<end>:"]:
        line = raw.split("//")[0].split(";")[0].strip()
        if m := re.match(r"(?:[0-9a-f]+ )?<?([\w$.]+)>?:$", line):
            if not m.group(1).startswith(("L", ".L")):  # a function, not a branch target within one
                if here:
                    other += uses
                fn, since, m0, uses, here = m.group(1), {}, 99, [], 0
            continue
        op, _, args = line.partition(" ")
        if not re.match(r"[a-z]\w+$", op):
            continue
        to_lds = op.startswith("buffer_load") and re.search(r"\blds\b", args)
        if to_lds:
            transfers, here = transfers + 1, here + 1
            if m0 < 1:
                close.append((fn, line))
            if min((since.get(r, 99) for r in scalar_regs(args)), default=99) < 5:
                early.append((fn, line))
        elif re.search(r"\bm0\b", args) and not (op == "s_mov_b32" and re.match(r"m0,", args.strip())):
            uses.append((fn, line))
        states = int(args, 0) + 1 if op == "s_nop" else 1
        m0 += states
        since = {r: n + states for r, n in since.items() if n + states < 20}
        if re.match(r"m0\b", args.strip()) and op.startswith("s_"):
            m0 = 0
        if op.startswith("v_"):
            first = args.split(",")[0] if not re.match(r"\s*v", args) else ""
            second = args.split(",")[1] if re.search(r"_co_|div_scale|mad_[ui]64", op) and "," in args else ""
            since.update((r, 0) for r in scalar_regs(first + " " + second))
    return transfers, close, early, other


def test_the_checker_sees_each_hazard():
    good = ["<k>:", "s_mov_b32 m0, s3", "s_nop 0", "buffer_load_dwordx4 v1, s[4:7], 0 offen lds"]
    assert findings(good) == (1, [], [], [])
    assert len(findings([x for x in good if "nop" not in x])[1]) == 1
    vector = good[:1] + ["v_readfirstlane_b32 s5, v0"] + good[1:]
    assert len(findings(vector)[2]) == 1 and not findings(vector[:2] + ["s_nop 4"] + vector[2:])[2]
    assert len(findings(good + ["v_movrels_b32 v0, v1, m0"])[3]) == 1


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_built_transfers_have_their_wait_states(tmp_path):
    lib = shutil.copy(xb.hip_path(), tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    total = 0
    for name in sorted(os.listdir(tmp_path)):
        if not name.endswith("gfx950"):
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", name], cwd=tmp_path, check=True, capture_output=True,
                              text=True).stdout
        if " lds" not in text:
            continue
        transfers, close, early, other = findings(text.splitlines())
        total += transfers
        assert not close and not early and not other, (close[:3], early[:3], other[:3])
    assert total, "no transfer found"
