"""Inline asm of the HIP sources names what it writes: a statement that moves to m0
lists m0 among its clobbers, so that the compiler sets it anew for any use of its own."""

from __future__ import annotations

import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "leanmoe-quant_amd", "csrc")


def _asm_statements(text: str) -> list[str]:
    text = re.sub(r"//[^\n]*", "", text)
    return [m.group(0) for m in re.finditer(r"\b(?:__)?asm(?:__)?\b[^;]*?\((?:[^;\"]|\"(?:[^\"\\]|\\.)*\")*?\)\s*;", text)]


def test_asm_that_writes_m0_clobbers_it():
    found = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip"))):
        with open(path, encoding="utf-8") as f:
            text = f.read()
        writes = re.findall(r"s_mov_b32 m0\b", re.sub(r"//[^\n]*", "", text))
        statements = [s for s in _asm_statements(text) if re.search(r"s_mov_b32 m0\b", s)]
        assert len(statements) == len(writes), path
        for s in statements:
            assert re.search(r'"m0"', s), "%s: m0 is written but not clobbered: %s" % (os.path.basename(path), s)
        found += len(statements)
    assert found
