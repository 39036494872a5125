"""Where the hot loops of the built library start modulo 32 bytes, against the
offsets they were measured at (csrc/wave.h, loop_offset): the same loops at
other offsets take up to 3% (leaf kernel) and 7% (fused adjoint) longer.  A
change of a kernel that fails this has moved a loop and needs the offsets
measured again."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "hacc-coral_amd", "libhaccsr.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"

FORCE = "k_forceILi0ELi5ELb0ELi2ELi2ELi%dE"
# kernel, loops by their reciprocal square roots and DPP adds, start mod 32
CASES = [(FORCE % 128, 4, 0, {16, 0}), (FORCE % 256, 4, 0, {16, 0}),
         ("k_adj_fused5", 2, 18, {20}), ("k_adj_fused6", 2, 18, {20})]


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("lib")
    shutil.copy(LIB, d / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    text = ""
    for f in sorted(os.listdir(d)):
        if "gfx950" in f:
            r = subprocess.run([OBJDUMP, "-d", f], cwd=d, check=True, capture_output=True, text=True).stdout
            if "k_force" in r or "k_adj_fused" in r:
                text += r
    return text


def loops(text, kernel):
    """(start, rsq, DPP instructions) of the loops without an inner loop."""
    m = re.search(r"^([0-9a-f]+) <\S*" + kernel + r"\S*>:\n(.*?)(?=^[0-9a-f]+ <|\Z)", text, re.S | re.M)
    assert m, kernel
    base, ins = int(m.group(1), 16), []
    for line in m.group(2).split("\n"):
        x = re.match(r"\s+(\S+)(.*?)//\s*([0-9A-F]+):(.*)", line)
        if x:
            ins.append((int(x.group(3), 16), x.group(1), x.group(2) + x.group(4)))
    at = {a: i for i, (a, _, _) in enumerate(ins)}
    back = {}  # start -> the first branch back to it
    for i, (a, op, rest) in enumerate(ins):
        y = re.search(r"<\S+\+0x([0-9a-f]+)>", rest) if op.startswith(("s_branch", "s_cbranch")) else None
        t = base + int(y.group(1), 16) if y else None
        if t is not None and t in at and t < a:
            back.setdefault(t, i)
    out = []
    for t, i in back.items():
        if any(u != t and t < u < ins[i][0] and back[u] < i for u in back):
            continue
        body = [op for _, op, _ in ins[at[t]:i + 1]]
        out.append((t, sum(op.startswith("v_rsq") for op in body), sum("dpp" in op for op in body)))
    return out


@pytest.mark.parametrize("kernel,rsq,dpp,starts", CASES)
def test_hot_loops_start_where_measured(assembly, kernel, rsq, dpp, starts):
    found = [(t % 32, r, n) for t, r, n in loops(assembly, kernel) if r == rsq]
    assert {t for t, _, n in found if n >= dpp} == starts, found
