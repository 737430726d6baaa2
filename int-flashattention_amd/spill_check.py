"""Checks the compiler's assembly of the HIP kernels for register spills that lose lanes.

The kernels of this package are allowed to spill a few vector registers in their tightest instances.  A spill store
writes the lanes that are active when it executes; the compiler places spill code per basic block and does not ask which
lanes are active there.  Two placements lose data silently:

* at the top of the block where divergent lanes rejoin, BEFORE the instruction that restores the exec mask
  (``s_or_b64 exec, exec, ...``): the store (or the reload) runs with the mask of the branch that was just left;
* a spill STORE anywhere between an instruction that narrows exec and the one that widens it again.

Both were seen with this compiler (the per-block, per-channel V scale instances at head_dim 256 wrote a wrong LSE for
the waves whose lanes had been masked off around a scale fetch).  The kernels avoid per-thread branches around their
global loads for that reason (they branch on the wave index, a scalar); this scan runs at build time over every kernel
and fails the build if such a placement appears again.
"""
from __future__ import annotations

import re
from typing import Iterator, List, Tuple

_LABEL = re.compile(r"^\.LBB\d+_\d+:")
_KERNEL = re.compile(r"^(_Z\w+):")
_BLOCK_END = re.compile(r"^\s+(s_cbranch\w*|s_branch|s_endpgm|s_setpc_b64)\b")
_EXEC_RESTORE = re.compile(r"^\s+(s_or_b64 exec, exec,|s_mov_b64 exec, -1)")
_EXEC_NARROW = re.compile(r"^\s+(s_and_saveexec_b64|s_or_saveexec_b64|s_and_b64 exec, exec,|s_andn2_b64 exec, exec,|s_xor_b64 exec, exec,)")
_SPILL = re.compile(r"^\s+(scratch_|buffer_)\w+.*Folded (Spill|Reload)")


_BRANCH = re.compile(r"^\s+s_c?branch\w*\s+(\.LBB\d+_\d+)")
_NO_FALLTHROUGH = ("s_branch", "s_endpgm", "s_setpc_b64")


def kernels(asm: str) -> Iterator[Tuple[str, List[dict]]]:
    """The kernels of one translation unit's assembly text: name and basic blocks, each its label and its [(line number, text)]."""
    name, blocks = "?", []
    for n, line in enumerate(asm.split("\n"), 1):
        m = _KERNEL.match(line)
        if m:
            if blocks:
                yield name, blocks
            name, blocks = m.group(1), []
            continue
        if _LABEL.match(line) or not blocks or blocks[-1]["done"]:
            blocks.append({"label": line.split(":")[0] if _LABEL.match(line) else None, "lines": [], "done": False})
        blocks[-1]["lines"].append((n, line))
        if _BLOCK_END.match(line):
            blocks[-1]["done"] = True
    if blocks:
        yield name, blocks


def successors(blocks: List[dict]) -> List[List[int]]:
    """Where control goes from the end of each block, by the branches and not by the order of the text."""
    by_label = {b["label"]: k for k, b in enumerate(blocks) if b["label"]}
    ways = []
    for k, b in enumerate(blocks):
        last = b["lines"][-1][1] if b["lines"] else ""
        nxt = [by_label[m.group(1)] for m in [_BRANCH.match(last)] if m and m.group(1) in by_label]
        if not (last.split() and last.split()[0] in _NO_FALLTHROUGH) and k + 1 < len(blocks):
            nxt.append(k + 1)
        ways.append(nxt)
    return ways


def scan(asm: str) -> List[str]:
    """Returns one line per suspicious spill / reload in the assembly text of one translation unit.

    Which blocks are entered with a narrowed mask follows the branches, not the order of the text: a block that stands behind an
    unconditional branch, inside or after a masked region, is entered from wherever its label is named."""
    findings: List[str] = []
    for kernel, blocks in kernels(asm):
        ways = successors(blocks)
        entry = [0] * len(blocks)      # line of an exec-narrowing instruction that may be in force on entry, 0: none
        work = list(range(len(blocks)))
        while work:
            k = work.pop(0)
            state = entry[k]
            for n, t in blocks[k]["lines"]:
                if _EXEC_NARROW.match(t):
                    state = n
                elif _EXEC_RESTORE.match(t):
                    state = 0
            for j in ways[k]:
                if state and not entry[j]:
                    entry[j] = state
                    if j not in work:
                        work.append(j)
        for k, b in enumerate(blocks):
            restore = next((i for i, (_, t) in enumerate(b["lines"]) if _EXEC_RESTORE.match(t)), None)
            state = entry[k]
            for i, (n, t) in enumerate(b["lines"]):
                if _SPILL.match(t):
                    if restore is not None and i < restore:
                        findings.append(f"{kernel}: line {n}: `{t.strip()}` runs before exec is restored at line {b['lines'][restore][0]}")
                    if state and "Folded Spill" in t:
                        findings.append(f"{kernel}: line {n}: `{t.strip()}` stores while exec is narrowed (since line {state})")
                if _EXEC_NARROW.match(t):
                    state = n
                elif _EXEC_RESTORE.match(t):
                    state = 0
    return findings
