"""Assumptions of the kernels' inline assembly that no result would show (no
GPU): a direct-to-LDS load reads m0, so m0 must be an operand of its block, and
no block may write m0 behind the compiler's back."""

from __future__ import annotations

import re
from pathlib import Path

SOURCES = Path(__file__).resolve().parents[1] / "tensorforge_amd" / "csrc"


def test_assembly_binds_m0_as_an_operand():
    blocks = [block for path in sorted(SOURCES.glob("*.h*"))
              for block in re.findall(r"\basm\b.*?\)\s*;", path.read_text(), re.DOTALL)]
    loads = [block for block in blocks if "global_load_lds" in block]
    assert loads and all('"{m0}"' in block for block in loads)
    assert not [block for block in blocks if re.search(r"\bm0,", block)]
