"""Build-time checks of the prefill kernels' inline-asm MFMAs.

`prefill_mfma_kernel` issues its PV MFMAs as inline asm (so that the O^T
accumulators stay in AGPRs), `prefill_wide_kernel` all of its MFMAs.  The
compiler cannot see an MFMA inside asm, so it neither inserts the wait states
the MFMA needs around it nor avoids placing a register copy right behind it.
The build therefore scans the kernels' gfx950 assembly and fails on

* any read of an inline-asm MFMA's destination registers, or (vector registers)
  any write to them, within the MFMA's result latency: a copy of an accumulator
  placed there once computed wrong prefill outputs;
* any vector instruction that writes an operand of an inline-asm MFMA, its
  accumulator among them, within the two wait states before it;
* in kernels that address the accumulation registers by number (`owned_agprs`),
  any use of one outside asm: it would overwrite an accumulator.
"""
from __future__ import annotations

import re

# Wait states a v_mfma_f32_32x32x16_bf16 result (16 passes) needs before a
# VALU or v_accvgpr read of it; the kernels' drains give 20 (s_nop 7, s_nop 7,
# s_nop 3).
RESULT_WAIT_STATES = 19
# Wait states between a VALU write of a register and an MFMA that reads it.
OPERAND_WAIT_STATES = 2

_INDEX = r"(0x[0-9a-f]+|\d+)"
_REGISTER = re.compile(rf"\b([av])\[{_INDEX}:{_INDEX}\]|\b([av])\[?{_INDEX}\b")
_NOP = re.compile(r"^s_nop\s+(\d+)")


def _registers(operand: str):
    """(file, first, last) of every vector / accumulation register named."""
    found = []
    for m in _REGISTER.finditer(operand):
        if m.group(1):
            found.append((m.group(1), int(m.group(2), 0), int(m.group(3), 0)))
        else:
            found.append((m.group(4), int(m.group(5), 0), int(m.group(5), 0)))
    return found


def _vector_writes(opcode: str, operands):
    """The registers that a vector instruction writes: its first operand, both of a swap."""
    if not opcode.startswith("v_"):
        return []
    return operands[0] + (operands[1] if "swap" in opcode else [])


def _overlap(x, y) -> bool:
    return x[0] == y[0] and x[1] <= y[2] and y[1] <= x[2]


def asm_mfma_hazards(assembly: str, owned_agprs: bool = False) -> list[str]:
    """The violations of the rules above (s_nop n counts n + 1 wait states, any
    other instruction 1).  Code is followed in listing order, labels included,
    so a fall-through is checked like straight-line code; a taken branch is not
    followed (prefill_mfma_kernel drains its asm MFMAs before each loop
    back-edge, prefill_wide_kernel has the next tile's first operand reads and
    the max of its scores there).  Reads by other MFMAs are not checked: an
    accumulator feeds only the next MFMA of its own chain, which the hardware's
    dependency check covers."""
    hazards: list[str] = []
    pending: list[list] = []  # [destination, wait states left, line] of asm MFMAs
    written: list[list] = []  # [register, wait states left, line] of VALU writes
    in_asm = False
    for number, raw in enumerate(assembly.splitlines(), 1):
        text = raw.strip()
        if text.startswith(";;#ASMSTART"):
            in_asm = True
            continue
        if text.startswith(";;#ASMEND"):
            in_asm = False
            continue
        text = text.split(";")[0].strip()
        if not text or text.startswith(".") or text.endswith(":"):
            continue
        issued = None  # the destination of an asm MFMA on this line
        opcode = text.split()[0]
        operands = [_registers(x) for x in text[len(opcode):].split(",")]
        nop = _NOP.match(text)
        if opcode.startswith("v_mfma"):
            if in_asm and operands[0]:
                for source in operands[1] + operands[2] + operands[3]:
                    for register, left, line in written:
                        if left > 0 and _overlap(register, source):
                            hazards.append(f"line {number}: '{text}' reads a register written at line {line}, "
                                           f"{OPERAND_WAIT_STATES - left} wait states before")
                issued = operands[0][0]
        elif nop is None:
            stores = opcode.startswith("ds_write") or "store" in opcode
            reads = [r for x in (operands if stores else operands[1:]) for r in x]
            writes = [r for r in _vector_writes(opcode, operands) if r[0] == "v" and r not in reads]
            for verb, registers in (("reads", reads), ("writes", writes)):
                for register in registers:
                    for dest, left, line in pending:
                        if left > 0 and _overlap(dest, register):
                            hazards.append(f"line {number}: '{text}' {verb} {dest[0]}[{dest[1]}:{dest[2]}], written by "
                                           f"the inline-asm MFMA at line {line}, after "
                                           f"{RESULT_WAIT_STATES - left} wait states")
            if owned_agprs and not in_asm and any(r[0] == "a" for x in operands for r in x):
                hazards.append(f"line {number}: '{text}' uses an accumulation register outside asm")
        step = int(nop.group(1)) + 1 if nop else 1
        for entry in pending + written:
            entry[1] -= step
        pending = [e for e in pending if e[1] > 0]
        if issued is not None:
            pending.append([issued, RESULT_WAIT_STATES, number])
        written = [e for e in written if e[1] > 0]
        if not opcode.startswith("v_mfma"):
            written += [[r, OPERAND_WAIT_STATES, number] for r in _vector_writes(opcode, operands)]
    return hazards
