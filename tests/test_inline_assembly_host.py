"""Inline assembly does not write m0 by itself, which the compiler does not take as a
clobber and may hold a value of its own in: it asks for what it needs there."""

import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "numba_mlir_amd", "csrc")


def _statements():
    for folder, _, files in os.walk(CSRC):
        for name in files:
            if name.endswith((".h", ".hip", ".cpp")):
                with open(os.path.join(folder, name)) as f:
                    text = f.read()
                for found in re.finditer(r"\basm\s+volatile\s*\(.*?\);", text, re.S):
                    yield name, found.group()


def test_m0_is_an_operand():
    loads = 0
    for name, text in _statements():
        code, *operands = text.split(":")
        assert not re.search(r"\bm0\b", code), (name, text)
        if "_lds_" in code:
            loads += 1
            assert '"{m0}"' in operands[1], (name, text)
    assert loads
