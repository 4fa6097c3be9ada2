"""Wait states in the built gfx950 code (CPU): a vector read or write of an
MFMA's result, and an MFMA that takes it as A or B, come 8 wait states after
one of 4 passes (16x16) and 12 after one of 8 (32x32); an LDS copy comes one
after the scalar write of its M0.  The compiler keeps these within a block, but
has lost the MFMA behind a branch, and it does not look into inline assembly."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.environ.get("MXFA_LIB", os.path.join(REPO, "acestep.cpp_amd", "lib", "libmxfa.so"))
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
VECTOR = ("v_", "ds_", "global_", "buffer_", "flat_", "scratch_")


def _regs(op):
    m = re.fullmatch(r"-?\|?v(?:\[(\d+):(\d+)\]|(\d+))\|?", op)
    if not m:
        return frozenset()
    lo = int(m.group(1) or m.group(3))
    return frozenset(range(lo, int(m.group(2) or lo) + 1))


def _functions(text):
    """{name: [(opcode, operand registers, first operand, branch target index)]}"""
    for body in re.split(r"\n(?=[0-9a-f]{16} <)", text):
        head = re.match(r"([0-9a-f]{16}) <(\S+)>:", body)
        if not head:
            continue
        base, rows, at = int(head.group(1), 16), [], {}
        for line in body.splitlines()[1:]:
            m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+): \S+.*?(?:<[^>+]+(?:\+0x([0-9a-f]+))?>)?$", line)
            if not m:
                continue
            ops = [o.split()[0] if o else "" for o in re.split(r",\s*(?![^\[]*\])", m.group(2))]
            at[int(m.group(3), 16)] = len(rows)
            rows.append((m.group(1), [_regs(o) for o in ops], ops[0] if ops else "", base + int(m.group(4) or "0", 16)))
        yield head.group(2), [(o, r, f, at.get(t) if "branch" in o else None) for o, r, f, t in rows]


def _states(op, first):
    return int(first, 0) + 1 if op == "s_nop" else 1


def _short_mfma(code):
    """(index of the early reader, wait states it had, needed) of a function."""
    out = {}
    for i, (op, regs, _, _) in enumerate(code):
        if not op.startswith("v_mfma"):
            continue
        need = 12 if "32x32" in op else 8
        todo, seen = [(i + 1, 0, regs[0])], set()
        while todo:
            j, w, live = todo.pop()
            while j < len(code) and w < need and live and (j, w, live) not in seen:
                seen.add((j, w, live))
                o, r, first, target = code[j]
                if target is not None:
                    if o != "s_branch":
                        todo.append((j + 1, w + 1, live))
                    j, w = target, w + 1
                    continue
                if o == "s_endpgm":
                    break
                if o.startswith("v_mfma"):
                    if (r[1] | r[2]) & live:
                        out[j] = (w, need)
                    live -= r[0]
                elif o.startswith(VECTOR) and any(x & live for x in r):
                    out[j] = (w, need)
                    live = live.difference(*r)
                w += _states(o, first)
                j += 1
    return out


@pytest.fixture(scope="module")
def functions(tmp_path_factory):
    if not (os.path.exists(OBJDUMP) and os.path.exists(LIB)):
        pytest.skip("no llvm-objdump or no built library")
    d = tmp_path_factory.mktemp("code")
    lib = shutil.copy(LIB, d)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=d, check=True, capture_output=True)
    out = {}
    for f in sorted(os.listdir(d)):
        if "gfx950" in f:
            text = subprocess.run([OBJDUMP, "-d", os.path.join(d, f)], check=True, capture_output=True, text=True).stdout
            out.update(_functions(text))
    assert sum(o.startswith("v_mfma") for c in out.values() for o, *_ in c) > 1000
    return out


def test_mfma_results(functions):
    bad = [(name, code[j][0], w, need) for name, code in functions.items()
           for j, (w, need) in _short_mfma(code).items()]
    assert not bad, bad


def test_lds_copies_after_m0(functions):
    after = [(name, code[j + 1][0]) for name, code in functions.items()
             for j, (op, _, first, _) in enumerate(code) if first == "m0" and op.startswith("s_")]
    bad = [x for x in after if x[1].startswith(("buffer_load", "global_load"))]
    assert len(after) > 100 and not bad, bad[:5]
