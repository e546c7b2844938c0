"""No kernel of the built library reaches a workgroup barrier with an LDS
operation of its wavefront outstanding: what it wrote before the barrier is what
the other wavefronts read after it.  (The compiler drops the wait that a barrier
stands for at the head of some loops; the library's barriers write it out.)

The library's own code objects are disassembled, and the number of outstanding
LDS operations is followed over the blocks of every kernel, each loop's back edge
included."""
import glob
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "2degas_amd", "lib2degas_hip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MANY = 64


def _functions(text):
    """(name, [(label or None, instruction)]) of every function."""
    name, body = None, []
    for line in text.splitlines():
        m = re.match(r"^[0-9a-f]+ <(\w+)>:$", line)
        if m and re.fullmatch(r"L\d+", m.group(1)):
            body.append((m.group(1), None))
        elif m:
            if name:
                yield name, body
            name, body = m.group(1), []
        elif line.startswith("\t"):
            body.append((None, line.split("//")[0].strip()))
    if name:
        yield name, body


def _blocks(body):
    """Instruction lists and successor indices."""
    blocks, starts = [[]], {}
    for label, ins in body:
        if label is not None:
            if blocks[-1]:
                blocks.append([])
            starts[label] = len(blocks) - 1
        else:
            blocks[-1].append(ins)
            if re.match(r"s_(c?branch|endpgm|setpc)", ins):
                blocks.append([])
    succ = []
    for k, b in enumerate(blocks):
        last = b[-1] if b else ""
        m = re.match(r"s_(c?)branch\w*\s+(\S+)", last)
        out = [starts[m.group(2)]] if m else []
        if not (m and not m.group(1)) and not re.match(r"s_(endpgm|setpc)", last) and k + 1 < len(blocks):
            out.append(k + 1)
        succ.append(out)
    return blocks, succ


def _outstanding_at_barriers(body):
    """(barriers, those reached with LDS operations outstanding)."""
    blocks, succ = _blocks(body)
    state, work, bad = {0: 0}, [0], set()
    while work:
        k = work.pop()
        n = state[k]
        for at, ins in enumerate(blocks[k]):
            if ins.startswith("ds_"):
                n = min(MANY, n + 1)
            elif ins.startswith("s_waitcnt"):
                m = re.search(r"lgkmcnt\((\d+)\)", ins)
                n = min(n, int(m.group(1))) if m else n
            elif ins.startswith("s_barrier") and n:
                bad.add((k, at))
        for q in succ[k]:
            if n > state.get(q, -1):
                state[q] = n
                work.append(q)
    return sum(i.startswith("s_barrier") for b in blocks for i in b), len(bad)


def test_the_check_sees_a_back_edge():
    """The check itself, on a loop whose entry waits and whose back edge does
    not, and on the same loop with the wait at the barrier."""
    loop = [(None, "ds_write_b32 v0, v1"), (None, "s_waitcnt lgkmcnt(0)"), ("L0", None), (None, "s_barrier"),
            (None, "ds_write_b32 v0, v1"), (None, "s_cbranch_scc0 L0"), (None, "s_endpgm")]
    assert _outstanding_at_barriers(loop) == (1, 1)
    assert _outstanding_at_barriers(loop[:3] + [(None, "s_waitcnt lgkmcnt(0)")] + loop[3:]) == (1, 0)


def test_barriers_wait_for_lds(tmp_path):
    if not os.path.exists(LIB) or not os.path.exists(OBJDUMP):
        pytest.skip("needs the built library and llvm-objdump")
    shutil.copy(LIB, tmp_path / "l.so")
    subprocess.run([OBJDUMP, "--offloading", "l.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    kernels, barriers, bad = 0, 0, []
    for f in sorted(glob.glob(str(tmp_path / "l.so.*gfx950"))):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--symbolize-operands", f], check=True,
                              stdout=subprocess.PIPE).stdout.decode()
        for name, body in _functions(text):
            n, b = _outstanding_at_barriers(body)
            kernels, barriers = kernels + 1, barriers + n
            if b:
                bad.append((name, n, b))
    assert kernels > 40 and barriers > 300
    assert not bad, bad
