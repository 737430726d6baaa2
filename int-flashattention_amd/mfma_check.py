"""Checks the compiler's assembly of the HIP kernels for reads of a matrix product ahead of its wait states.

A matrix instruction (MFMA) writes its result some time after it was issued, and the hardware does not hold back an
instruction that reads it sooner: on gfx950 a product of P passes (four clocks each) needs P + 4 wait states (two passes: P + 3) between itself and
any other instruction that reads or overwrites one of its registers, or a matrix instruction that multiplies them.
The next product of a chain, which takes the whole result as its addend, needs none.  The compiler puts ``s_nop`` in place where
other instructions do not fill the time, but not for hand-written instructions, and across branches it can count along the longer of
two ways into a block: a decode kernel's first product was then read too early, and its rows came out wrong, once the
compiler had moved the read behind the branch that closes the loop.  This scan follows every product along all ways through
the kernel to its readers and runs at build time over every kernel.
"""
from __future__ import annotations

import re
from typing import Dict, List, Tuple

import spill_check

_INSTRUCTION = re.compile(r"^\s+([a-z]\w*)\s*([^;]*)")
_REGISTERS = re.compile(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])")
_VECTOR = ("v_", "ds_", "buffer_", "global_", "flat_", "scratch_")
# Passes of the instructions that the kernels use.
_PASSES = {"i32_16x16x64_i8": 4, "f32_16x16x32_f16": 4, "f32_16x16x32_bf16": 4,
           "i32_32x32x32_i8": 8, "f32_32x32x16_f16": 8, "f32_32x32x16_bf16": 8}


def _registers(text: str) -> List[Tuple[str, int]]:
    return [(f, r) for f, one, lo, hi in _REGISTERS.findall(text) for r in (range(int(lo), int(hi) + 1) if lo else (int(one),))]


def scan(asm: str) -> List[str]:
    """Returns one line per early access in the assembly text of one translation unit."""
    findings: List[str] = []
    for kernel, blocks in spill_check.kernels(asm):
        if not any("v_mfma" in t for b in blocks for _, t in b["lines"]):
            continue
        code = [[(n, *m.groups()) for n, t in b["lines"] for m in [_INSTRUCTION.match(t)] if m] for b in blocks]
        ways = spill_check.successors(blocks)
        # register -> (wait states that its product still needs, line of the product) on entry; the larger need of all ways in
        entry: List[Dict[Tuple[str, int], Tuple[int, int]]] = [{} for _ in blocks]
        found: Dict[int, str] = {}
        work = list(range(len(blocks)))
        while work:
            k = work.pop(0)
            pending = dict(entry[k])
            for n, op, operands in code[k]:
                is_mfma = op.startswith("v_mfma_")
                if pending and op.startswith(_VECTOR):
                    args = re.split(r",\s*(?![^\[]*\])", operands.strip())
                    used = _registers(", ".join(args[1:3]) if is_mfma else operands)
                    if is_mfma:                # an addend that is not exactly a product's registers (a chain's next instruction starts when they are there)
                        addend = _registers(args[3].split()[0])
                        lines = {pending[r][1] for r in addend if r in pending}
                        if lines and (len(lines) > 1 or any(r not in pending for r in addend) or
                                      any(p[1] in lines and r not in addend for r, p in pending.items())):
                            used += addend
                    early = [pending[r] for r in used if r in pending]
                    if early:
                        need, line = max(early)
                        found[n] = f"{kernel}: line {n}: `{op} {operands.strip()}` comes {need} wait states too early for the product of line {line}"
                states = int(operands, 0) + 1 if op == "s_nop" else 1
                pending = {r: (need - states, line) for r, (need, line) in pending.items() if need > states}
                if is_mfma:
                    passes = _PASSES.get(op[len("v_mfma_"):])
                    if passes is None:
                        findings.append(f"{kernel}: line {n}: the passes of {op} are not in this scan's table")
                        continue
                    for r in _registers(operands.split(",")[0]):
                        pending[r] = (passes + 4, n)
            for j in ways[k]:
                grown = False
                for r, p in pending.items():
                    if p[0] > entry[j].get(r, (0, 0))[0]:
                        entry[j][r] = p
                        grown = True
                if grown and j not in work:
                    work.append(j)
        findings += [found[n] for n in sorted(found)]
    return findings


_DPP = re.compile(r"_dpp\b|\b(quad_perm|row_newbcast|row_shl|row_shr|row_ror|row_mirror|row_half_mirror|row_bcast|wave_)")


def scan_lanes(asm: str) -> List[str]:
    """Returns one line per instruction that takes another lane's register (DPP, its first source) less than two wait states after a vector instruction wrote
    it, or less than five after one wrote the exec mask, along all ways through the kernel.  The hardware does not hold it back; the compiler
    keeps the distance for its own instructions only, and the kernels' hand-written ones read registers that it may copy or fetch back from an
    accumulation register just ahead."""
    findings: List[str] = []
    for kernel, blocks in spill_check.kernels(asm):
        code = [[(n, t, *m.groups()) for n, t in b["lines"] for m in [_INSTRUCTION.match(t)] if m] for b in blocks]
        if not any(_DPP.search(t) for c in code for _, t, _, _ in c):
            continue
        ways = spill_check.successors(blocks)
        entry: List[Dict[object, Tuple[int, int]]] = [{} for _ in blocks]      # register, or "exec" -> (wait states still needed, line of the write)
        found: Dict[int, str] = {}
        work = list(range(len(blocks)))
        while work:
            k = work.pop(0)
            pending = dict(entry[k])
            for n, text, op, operands in code[k]:
                args = re.split(r",\s*(?![^\[]*\])", operands.strip())
                if pending and op.startswith("v_") and _DPP.search(text):
                    early = [pending[r] for r in ["exec", *_registers(args[1].split()[0] if len(args) > 1 else "")] if r in pending]
                    if early:
                        need, line = max(early)
                        found[n] = f"{kernel}: line {n}: `{op} {operands.strip()}` comes {need} wait states too early for the write of line {line}"
                states = int(operands, 0) + 1 if op == "s_nop" else 1
                pending = {r: (need - states, line) for r, (need, line) in pending.items() if need > states}
                if op.startswith("v_"):
                    for r in _registers(args[0]):
                        pending[r] = (2, n)
                    if op.startswith("v_cmpx"):
                        pending["exec"] = (5, n)
            for j in ways[k]:
                grown = False
                for r, p in pending.items():
                    if p[0] > entry[j].get(r, (0, 0))[0]:
                        entry[j][r] = p
                        grown = True
                if grown and j not in work:
                    work.append(j)
        findings += [found[n] for n in sorted(found)]
    return findings


_LOAD_WAIT = re.compile(r"^\s+s_waitcnt\b.*\bvmcnt\(")


def _in_loops(ways: List[List[int]]) -> List[bool]:
    """Which blocks can be reached from their own end."""
    def reach(k):
        seen, work = set(), list(ways[k])
        while work:
            j = work.pop()
            if j not in seen:
                seen.add(j)
                work += ways[j]
        return seen
    return [k in reach(k) for k in range(len(ways))]


def scan_waits(asm: str) -> List[str]:
    """Returns one line per wait for loads that the compiler put directly ahead of a product inside a loop.

    Tiles come through LDS, by hand-written copies and waits that the compiler does not know.  A wait of its own ahead of a product in the loop is
    for Q, which arrived long ago, and holds the products back until the next tiles, requested just before, are there as well: no copy runs under
    the work of a step (decoding steps lost up to a third).  Kernels that fetch a spilled fragment back from scratch in the loop have to wait there."""
    findings: List[str] = []
    for kernel, blocks in spill_check.kernels(asm):
        found, by_hand, wait, reload = [], False, 0, False
        if not any("v_mfma" in t for b in blocks for _, t in b["lines"]):
            continue
        for b, loop in zip(blocks, _in_loops(spill_check.successors(blocks))):
            for n, t in b["lines"]:
                if "#ASMSTART" in t or "#ASMEND" in t:
                    by_hand = "#ASMSTART" in t
                m = _INSTRUCTION.match(t)
                if not m or not loop:
                    continue
                reload = reload or "Folded Reload" in t
                if wait and m.group(1).startswith("v_mfma"):
                    found.append(f"{kernel}: line {wait}: a wait for loads ahead of the product of line {n}, inside a loop")
                wait = n if _LOAD_WAIT.match(t) and not by_hand else 0
        findings += [] if reload else found
    return findings
