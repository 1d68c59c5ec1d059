"""Wait states that gfx950 leaves to software, checked in device assembly.

The compiler inserts them around its own instructions, but not around those
written in inline asm (the MFMAs and the LDS copies of the LM head kernels).
``hazards`` walks each kernel's control-flow graph (isa_dataflow) with the wait
states that have passed since each write and reports every instruction that
comes too early (instructions count one wait state, ``s_nop n`` n + 1):

  * an MFMA's A, B or C operand after a VALU write of it: 2;
  * a vector-memory instruction's SGPR after a VALU write of it
    (v_readlane of a spilled one, v_readfirstlane, a compare): 5;
  * a copy to LDS after a write of m0: 1;
  * anything but an MFMA reading or writing an MFMA's result, or an MFMA
    reading it as A or B: 11 (an MFMA of 8 passes); an MFMA adding to it: 2.
"""
from __future__ import annotations

import re

from isa_dataflow import _blocks, _operands, kernels

VALU_TO_MFMA = 2
VALU_TO_VMEM_SGPR = 5
M0_TO_COPY = 1
MFMA_RESULT = 11
MFMA_CHAIN = 2
_WINDOW = 12

_REGS = re.compile(r"\b([vas])\[(\d+):(\d+)\]|\b([vas])(\d+)\b")
_VMEM = ("buffer_", "global_", "flat_", "scratch_")
_TWO_RESULTS = re.compile(r"v_(permlane\d+_swap|swap_b32)")
_SECOND_SGPR = re.compile(r"v_\w*_co_|v_mad_[ui]64|v_div_scale")


def _registers(text: str) -> set:
    out = set()
    for m in _REGS.finditer(text):
        if m.group(1):
            out |= {(m.group(1), r) for r in range(int(m.group(2)), int(m.group(3)) + 1)}
        else:
            out.add((m.group(4), int(m.group(5))))
    out |= {("s", n) for n in ("vcc", "m0") if re.search(rf"\b{n}\b", text)}
    return out


def _vector(regs: set) -> set:
    return {r for r in regs if r[0] != "s"}


def _step(ins: str, age: dict, found: list | None) -> dict:
    """`age`: (kind, register) -> wait states since the write."""
    op, _, rest = ins.partition(" ")
    ops = _operands(rest)
    first = _registers(ops[0]) if ops else set()
    others = set().union(*(_registers(o) for o in ops[1:])) if len(ops) > 1 else set()

    def need(kind: str, regs: set, states: int) -> None:
        for r in regs:
            if age.get((kind, r), _WINDOW) < states and found is not None:
                found.append((ins, kind, r, age[kind, r]))

    wrote = []
    if op.startswith("v_mfma"):
        a_b = set().union(*(_registers(o) for o in ops[1:3]))
        c = _registers(ops[3]) if len(ops) > 3 else set()
        need("valu", a_b | c, VALU_TO_MFMA)
        need("mfma", a_b, MFMA_RESULT)
        need("mfma", c | first, MFMA_CHAIN)
        wrote = [("mfma", r) for r in first]
    else:
        if not op.startswith("s_"):
            need("mfma", _vector(first | others), MFMA_RESULT)
        if op.startswith(_VMEM):
            need("valu", {r for r in first | others if r[0] == "s"}, VALU_TO_VMEM_SGPR)
            if re.search(r"\blds\b", rest) or "_lds_" in op:
                need("m0", {("s", "m0")}, M0_TO_COPY)
        elif op.startswith("v_"):
            dst = set(first)
            if _TWO_RESULTS.match(op) or _SECOND_SGPR.match(op):
                dst |= _registers(ops[1])
            wrote = [("valu", r) for r in dst]
        if ("s", "m0") in first and not op.startswith(_VMEM):
            wrote.append(("m0", ("s", "m0")))
    states = int(rest, 0) + 1 if op == "s_nop" else 1
    age = {k: n + states for k, n in age.items() if n + states < _WINDOW}
    for kind, r in wrote:
        age[kind, r] = 0
    if op.startswith("s_"):  # a scalar write ends the vector one's hazard
        for r in first:
            age.pop(("valu", r), None)
    return age


def hazards_of_kernel(lines: list[str]):
    blocks, succ = _blocks(lines)
    code = [[s.split(";")[0].strip() for s in b] for b in blocks]
    code = [[s.replace("\t", " ") for s in b if s and not s.startswith(".")] for b in code]
    entry: list = [None] * len(code)
    if not code:
        return []
    entry[0] = {}
    work = [0]
    while work:
        i = work.pop()
        age = entry[i]
        for s in code[i]:
            age = _step(s, age, None)
        for j in succ[i]:
            if entry[j] is None:
                entry[j] = dict(age)
                work.append(j)
                continue
            new = dict(entry[j])
            for k, n in age.items():
                new[k] = min(n, new.get(k, n))
            if new != entry[j]:
                entry[j] = new
                work.append(j)
    found: list = []
    for i, age in enumerate(entry):
        for s in code[i] if age is not None else ():
            age = _step(s, age, found)
    return found


def hazards(listing: str):
    """{kernel: [(instruction, kind of write, register, wait states)]}"""
    found = {name: hazards_of_kernel(body) for name, body in kernels(listing).items()}
    return {name: f for name, f in found.items() if f}
