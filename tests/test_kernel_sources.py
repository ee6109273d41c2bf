"""Assumptions of the kernels' inline assembly that no result would show (no
GPU): a block that writes m0 must say so, or the compiler may keep a value of
its own there across it."""

from __future__ import annotations

import re
from pathlib import Path

SOURCES = Path(__file__).resolve().parents[1] / "tensorforge_amd" / "csrc"


def test_assembly_that_writes_m0_declares_it():
    blocks = [(path.name, block) for path in sorted(SOURCES.glob("*.h*"))
              for block in re.findall(r"\basm\b.*?\)\s*;", path.read_text(), re.DOTALL)]
    writers = [(name, block) for name, block in blocks if re.search(r"\bm0,", block)]
    assert writers
    undeclared = [name for name, block in writers if '"m0"' not in block]
    assert not undeclared
