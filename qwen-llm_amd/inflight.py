"""Checks generated gfx950 assembly for registers that are touched while a load still fills them.

Some kernels ask for loads in inline asm and wait for them with hand-counted ``s_waitcnt``; the compiler takes such a load's
output as written at once and may copy or reuse the register ahead of the wait.  This follows every path through a kernel: a
load's destination is in flight until a wait says that it has arrived, and an instruction that reads or writes a register in
flight is a complaint.  The compiler's own loads pass the same check, so that the model is tried on all of them.

Reads from LDS are followed in every kernel, loads from memory in those that ``check_assembly`` is given for it: where a
kernel picks one of several waits by a number it knows at run time, paths are followed that are never taken.

Arrival.  ``s_waitcnt vmcnt(n)`` / ``lgkmcnt(n)``: at most n of the counter's operations are still under way, and reads
return in the order of issue, so a load with n or more later reads of its counter behind it has arrived.  Only reads
count as later ones: stores (vmcnt) and scalar loads (lgkmcnt) may return out of that order."""
from __future__ import annotations

import re

_REG = re.compile(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])")
_WAIT = re.compile(r"\b(vmcnt|lgkmcnt)\((\d+)\)")
_LABEL = re.compile(r"^([.\w$]+):")
_FAR = 64  # more operations behind a load than any wait can leave under way


def _registers(text):
    """Vector registers named in an operand text, accumulation registers numbered from 1000."""
    out = set()
    for kind, one, lo, hi in _REG.findall(text):
        base = 1000 if kind == "a" else 0
        out.update(range(base + int(one), base + int(one) + 1) if one else range(base + int(lo), base + int(hi) + 1))
    return out


def _decode(text):
    """One instruction -> (kind, payload, registers it names); kinds: load (counter, destination), wait, branch, jump, end, other."""
    op, _, rest = text.partition(" ")
    if op == "s_waitcnt":
        waits = {("vm" if c == "vmcnt" else "lgkm"): int(n) for c, n in _WAIT.findall(rest)}
        return "wait", waits, frozenset()
    if op.startswith("s_cbranch"):
        return "branch", rest.strip(), frozenset()
    if op == "s_branch":
        return "jump", rest.strip(), frozenset()
    if op in ("s_endpgm", "s_setpc_b64", "s_trap"):
        return "end", None, frozenset()
    if op.startswith("s_"):
        return "other", None, frozenset()
    regs = frozenset(_registers(rest))
    if op.startswith(("global_load_lds", "buffer_load")) and "lds" in text:
        return "load", ("vm", frozenset()), regs
    if op.startswith(("global_load", "buffer_load", "scratch_load")):
        return "load", ("vm", frozenset(_registers(rest.split(",")[0]))), regs
    if op.startswith("flat_load"):
        return "load", ("flat", frozenset(_registers(rest.split(",")[0]))), regs
    if op.startswith(("ds_read", "ds_bpermute", "ds_permute", "ds_swizzle")):
        return "load", ("lgkm", frozenset(_registers(rest.split(",")[0]))), regs
    return "other", None, regs


def _blocks(lines):
    """Basic blocks of one kernel: [(instructions, successors)], instruction = (line number, text, decoded)."""
    blocks, names, cur = [], {}, []
    ends = []  # how each block ends: (kind, label)

    def close(kind="fall", label=None):
        nonlocal cur
        blocks.append(cur)
        ends.append((kind, label))
        cur = []

    for number, raw in lines:
        text = raw.split(";")[0].strip()
        label = _LABEL.match(text)
        if label:
            close()
            names[label.group(1)] = len(blocks)
            continue
        if not text or text.startswith((".", "//")):
            continue
        text = re.sub(r"\s+", " ", text)
        what = _decode(text)
        cur.append((number, text, what))
        if what[0] in ("branch", "jump", "end"):
            close(what[0], what[1] if what[0] != "end" else None)
    close("end")
    succ = []
    for i, (kind, label) in enumerate(ends):
        to = [] if kind in ("jump", "end") else [i + 1]
        if label is not None:
            to.append(names[label])
        succ.append(to)
    return blocks, succ


def _step(state, what):
    """State after an instruction: register -> (counter, later reads of that counter, at least)."""
    kind, payload, _ = what
    if kind == "wait":
        for counter, n in payload.items():
            # (a flat load is on both counters, and may return out of order on either: a wait for all of one is enough)
            state = {r: a for r, a in state.items() if not ((a[0] == counter and a[1] >= n) or (a[0] == "flat" and n == 0))}
    elif kind == "load":
        counter, dest = payload
        state = {r: (c, min(_FAR, n + (c == counter))) for r, (c, n) in state.items()}
        for r in dest:
            state[r] = (counter, 0)
    return state


def _join(a, b):
    if a is None:
        return dict(b)
    out = dict(a)
    for r, (c, n) in b.items():
        if r not in out:
            out[r] = (c, n)
        elif out[r][0] != c:
            out[r] = ("flat", 0)
        elif n < out[r][1]:
            out[r] = (c, n)
    return out


def check_kernel(lines, memory=True) -> list:
    """Complaints about one kernel, lines = [(number, text)] from its label to its last instruction.  memory: loads from
    memory too, not only reads from LDS."""
    blocks, succ = _blocks(lines)
    if not memory:
        blocks = [[(n, t, (k, (p[0], frozenset()), r) if k == "load" and p[0] != "lgkm" else (k, p, r)) for n, t, (k, p, r) in b]
                  for b in blocks]
    at_entry = [None] * len(blocks)
    at_entry[0] = {}
    work = [0]
    while work:
        i = work.pop()
        state = at_entry[i]
        for _, _, what in blocks[i]:
            if what[0] in ("wait", "load"):
                state = _step(state, what)
        for j in succ[i]:
            if j < len(blocks):
                joined = _join(at_entry[j], state)
                if joined != at_entry[j]:
                    at_entry[j] = joined
                    work.append(j)
    bad = []
    for i, block in enumerate(blocks):
        state = at_entry[i]
        if state is None:
            continue
        for number, text, what in block:
            touched = [r for r in what[2] if r in state]
            if touched:
                bad.append(f"line {number}: {text}: {', '.join(('v%d' % r) if r < 1000 else ('a%d' % (r - 1000)) for r in sorted(touched))} in flight")
            if what[0] in ("wait", "load"):
                state = _step(state, what)
    return bad


def check_assembly(text: str, memory=()) -> list:
    """Complaints about all kernels in an assembly file.  ``memory``: name fragments of the kernels whose loads from memory are
    followed too; a fragment that no kernel's name holds is a complaint, so that the check cannot pass for want of one."""
    lines = text.splitlines()
    kernels = set(re.findall(r"^\s*\.amdhsa_kernel\s+(\S+)", text, re.M))
    bad, seen = [], set()
    i = 0
    while i < len(lines):
        m = _LABEL.match(lines[i])
        if m and m.group(1) in kernels:
            name, start = m.group(1), i + 1
            while i < len(lines) and not lines[i].startswith(".Lfunc_end") and ".section" not in lines[i]:
                i += 1
            seen.add(name)
            bad += [f"{name}: {c}" for c in check_kernel(list(enumerate(lines[start:i], start + 1)), any(k in name for k in memory))]
        i += 1
    bad += [f"{k}: no such kernel in the assembly" for k in memory if not any(k in name for name in seen)]
    bad += [f"{k}: its code was not found" for k in kernels - seen]
    return bad
