"""Checks the compiler's listing of a kernel whose vector loads are written as inline assembly.

The compiler takes the output registers of such a load as written at once.  Between the load and the hand-placed
``s_waitcnt vmcnt`` that covers it, an instruction of the compiler's own that reads those registers (a copy, a spill) gets
what they held before, and one that writes them is overwritten when the data arrive; neither draws a diagnostic.  Whether
one is there depends on the register allocation of the build at hand, so the listing of that build is checked: along every
path of every kernel, no instruction may name a register that a load of an inline-assembly block has not yet filled.

gfx9 rules used: every vector-memory instruction counts in ``vmcnt``, they retire in the order of issue, and
``s_waitcnt vmcnt(n)`` returns when at most the ``n`` last ones are outstanding."""

from __future__ import annotations

import re
from typing import Dict, FrozenSet, List, Tuple

_VMEM = ("global_", "buffer_load", "buffer_store", "buffer_atomic", "flat_", "scratch_")
_REG = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")
_LABEL = re.compile(r"^(\.?[A-Za-z_$][\w.$]*):")

Outstanding = Tuple[FrozenSet[str], ...]  # oldest first: the registers an inline-assembly load will still write


def _registers(text: str) -> FrozenSet[str]:
    out = set()
    for kind, lo, hi, one in _REG.findall(text):
        out.update(f"{kind}{i}" for i in range(int(lo or one), int(hi or one) + 1))
    return frozenset(out)


def _vmcnt(line: str):
    """n of ``s_waitcnt vmcnt(n)``; None where the instruction does not wait for vector memory."""
    m = re.search(r"vmcnt\((\d+)\)", line)
    if m:
        return int(m[1])
    m = re.match(r"s_waitcnt\s+(0x[0-9a-fA-F]+|\d+)$", line)
    if m:  # raw encoding: bits 3:0 and 15:14
        v = int(m[1], 0)
        return (v & 15) | ((v >> 14 & 3) << 4)
    return None


def kernels(listing: str) -> Dict[str, List[Tuple[str, bool]]]:
    """Instructions and labels of each function in the listing, each with whether it stands in an inline-assembly block."""
    out: Dict[str, List[Tuple[str, bool]]] = {}
    body, in_asm = None, False
    for raw in listing.splitlines():
        if "#ASMSTART" in raw:
            in_asm = True
            continue
        if "#ASMEND" in raw:
            in_asm = False
            continue
        line = raw.split(";")[0].split("//")[0].strip()
        m = _LABEL.match(line)
        if m:
            if m[1].startswith(".Lfunc_end"):
                body = None
            elif not m[1].startswith(".L"):
                body = out.setdefault(m[1], [])
                continue
            if body is not None:
                body.append((m[1] + ":", False))
            continue
        if body is not None and line and not line.startswith("."):
            body.append((line, in_asm))
    return {name: b for name, b in out.items() if b}


def hazards(body: List[Tuple[str, bool]]) -> List[str]:
    """The instructions of one kernel that touch a register still to be filled, one message each."""
    at = {line[:-1]: i for i, (line, _) in enumerate(body) if line.endswith(":")}
    found: Dict[int, str] = {}
    seen = set()
    work: List[Tuple[int, Outstanding]] = [(0, ())]
    while work:
        i, out = work.pop()
        while i < len(body):
            if (i, out) in seen:
                break
            # states are compared at labels and branches only: the rest follows from them
            line, in_asm = body[i]
            if line.endswith(":") or line.startswith(("s_branch", "s_cbranch")):
                seen.add((i, out))
            if line.endswith(":"):
                i += 1
                continue
            op = line.split()[0]
            regs = _registers(line)
            late = regs & frozenset().union(*out)
            if late:
                found.setdefault(i, f"{line}  <- {', '.join(sorted(late))} not loaded yet")
                break  # what follows on this path follows from it (and a loop without a wait ends here)
            if op == "s_endpgm":
                if any(out):
                    found.setdefault(i, "s_endpgm with a load in flight")
                break
            if op == "s_waitcnt":
                n = _vmcnt(line)
                if n is not None:
                    out = out[len(out) - n:] if n < len(out) else out
            elif op.startswith(_VMEM) and not op.startswith("global_wb") and not op.startswith("global_inv"):
                dest = frozenset()
                if in_asm and "_load_" in op and "_lds_" not in op:
                    dest = _registers(line.split(None, 1)[1].split(",")[0])
                out = out + (dest,)
            while out and not out[0]:  # what is older than the first load in flight does not matter
                out = out[1:]
            if op == "s_branch":
                i = at[line.split()[1]]
                continue
            if op.startswith("s_cbranch"):
                work.append((at[line.split()[1]], out))
            i += 1
    return [found[i] for i in sorted(found)]


def check(listing: str) -> Dict[str, List[str]]:
    """Hazards by kernel, for the kernels that have any."""
    out = {}
    for name, body in kernels(listing).items():
        if any(in_asm and "_load_" in line for line, in_asm in body):
            h = hazards(body)
            if h:
                out[name] = h
    return out
