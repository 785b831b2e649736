"""Inline assembly leaves m0, which the compiler does not take as a clobber and may hold a
value of its own in, as it was."""

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


def test_m0_is_put_back():
    writes = [(name, text) for name, text in _statements() if re.search(r"\bm0\b", text)]
    assert writes
    for name, text in writes:
        code = "".join(re.findall(r'"([^"]*)"', text.split(":")[0])).replace(r"\t", "")
        first, *_, last = code.split(r"\n")
        saved = re.fullmatch(r"s_mov_b32 (%\d), m0", first)
        assert saved and last == f"s_mov_b32 m0, {saved.group(1)}", (name, code)
