"""CPU: inline assembly in the sources that use the matrix cores.

An MFMA reads its C operand and writes its result over several cycles.  The
compiler keeps the wait states that another instruction needs before it may
write those registers, but only around instructions that it generates; the
text of an asm statement is opaque to it.  So the asm statements of these
sources are empty (they hide a value's origin) or set up a constant before
the first matrix instruction.
"""
from __future__ import annotations

import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "cogito_amd" / "csrc"
CONSTANT = re.compile(r"[sv]_mov_b32 %0, 0x[0-9a-f]+")


def asm_texts(src: str) -> list[str]:
    return re.findall(r'\basm\s*(?:volatile)?\s*\(\s*"([^"]*)"', src)


def test_no_instruction_in_asm_beside_the_matrix_cores():
    files = [p for p in sorted(CSRC.rglob("*")) if p.suffix in (".hip", ".hpp", ".h")
             and "mfma" in p.read_text()]
    assert files
    for p in files:
        for text in asm_texts(p.read_text()):
            assert text == "" or CONSTANT.fullmatch(text), f"{p.name}: asm {text!r}"
