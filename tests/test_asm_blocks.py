"""Inline asm of the kernels: a scalar operand may have reached its register by a vector instruction (a reloaded
spill), which needs two wait states before a vector instruction reads it, and the compiler adds none inside a block."""

import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "aleph_amd" / "csrc"


def _blocks(text):
    """Source of every asm statement, macros' line ends joined."""
    text = text.replace("\\\n", "\n")
    for m in re.finditer(r"\basm volatile\(", text):
        depth, i, quoted = 1, m.end(), False
        while depth:
            if text[i] == '"' and text[i - 1] != "\\":
                quoted = not quoted
            depth += 0 if quoted else {"(": 1, ")": -1}.get(text[i], 0)
            i += 1
        yield text[m.end():i - 1]


@pytest.mark.parametrize("name", ["inplace.hpp", "op_loop.hpp", "k_noise.hip", "k_pauli.hip"])
def test_blocks_with_scalar_operands_start_with_wait_states(name):
    text = (CSRC / name).read_text()
    found = 0
    for block in _blocks(text):
        code, _, operands = block.partition(":")
        scalar = '"s"(' in operands or "ALEPH_ROWS_IN" in operands
        if scalar and re.search(r"\bv_|MUL|FMA|MOV", code):
            found += 1
            assert code.lstrip().startswith('"s_nop 1\\n'), block
    assert found or name != "inplace.hpp"
