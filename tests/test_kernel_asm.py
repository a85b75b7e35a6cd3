"""Every load written in inline asm waits for its data in the same statement.

The compiler takes an asm statement's outputs as written when it ends.  A load
whose wait stands in a later statement may be copied, or its register given to
something else, while the data is still on its way: wrong values, with nothing
to show it in a test that happens to be compiled well.
"""

from __future__ import annotations

import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "stream-attn_amd" / "csrc"
LOAD = re.compile(r"\b(ds_read|ds_load|global_load|buffer_load|flat_load|scratch_load|s_load|s_buffer_load)")


def asm_statements(text):
    """The text of each asm statement's template: its string literals up to the operands."""
    for match in re.finditer(r"\basm\s+volatile\s*\(\s*((?:\"(?:[^\"\\]|\\.)*\"\s*)+)", text):
        yield "".join(re.findall(r"\"((?:[^\"\\]|\\.)*)\"", match.group(1)))


@pytest.mark.parametrize("path", sorted(p.name for p in CSRC.iterdir() if p.suffix in (".h", ".hip", ".cpp")))
def test_asm_loads_wait_in_their_own_statement(path):
    for template in asm_statements((CSRC / path).read_text()):
        lines = [line.strip() for line in re.split(r"\\n(?:\\t)?", template) if line.strip()]
        if any(LOAD.match(line) for line in lines):
            assert re.match(r"s_waitcnt\b.*\b(lgkmcnt|vmcnt)\(0\)", lines[-1]), template


def test_the_kernels_reads_are_found():
    templates = list(asm_statements((CSRC / "sa_update_kernel.h").read_text()))
    assert sum("ds_read_b64_tr_b16" in t for t in templates) == 3
