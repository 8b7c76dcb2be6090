"""Inline assembly in the kernels declares what it writes besides its operands."""
from __future__ import annotations

import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "neurogrid_amd" / "csrc"


def asm_statements():
    for f in sorted(CSRC.glob("*.h*")):
        for m in re.finditer(r"\b_*asm_*(?:\s+volatile)?\s*\((.*?)\)\s*;", f.read_text(), re.S):
            yield f.name, m.group(1)


def test_m0_is_declared_where_it_is_written():
    writers = [(f, s) for f, s in asm_statements() if re.search(r"\bs_\w+ m0\b", s)]
    assert writers
    for f, s in writers:
        assert '"m0"' in s.rsplit(":", 1)[1], f"{f}: {s}"
