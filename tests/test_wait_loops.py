"""Every loop in which device code waits for another workgroup (it sleeps
between its reads) polls by atomic loads: a buffer load is neither atomic nor
volatile, so the compiler may take one out of the loop, and the grid would wait
for ever."""

import os
import re

import pytest

import oqupy_amd

CSRC = os.path.join(os.path.dirname(oqupy_amd.__file__), "csrc")
FILES = sorted(f for f in os.listdir(CSRC) if f.endswith((".hip", ".h")))
POLLS = ("__hip_atomic_load", "ld_agent(")
PLAIN = ("ld_agent16(", "raw_buffer_load")


def _matching(text, at, opening, closing):
    """End of the bracket pair that starts at text[at]."""
    depth = 0
    for i in range(at, len(text)):
        depth += (text[i] == opening) - (text[i] == closing)
        if depth == 0:
            return i + 1
    raise AssertionError("unbalanced source")


def _loops(text):
    """Text of every for / while loop, head and body."""
    for m in re.finditer(r"\b(for|while)\s*\(", text):
        end = _matching(text, m.end() - 1, "(", ")")
        rest = text[end:]
        if rest.lstrip().startswith("{"):
            end = _matching(text, end + rest.index("{"), "{", "}")
        else:
            end += rest.index(";") + 1
        yield text[m.start():end]


def _waits(name):
    with open(os.path.join(CSRC, name)) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    waits = [loop for loop in _loops(text) if "s_sleep" in loop]
    # the innermost one of nested loops
    return [w for w in waits if not any(o != w and o in w for o in waits)]


@pytest.mark.parametrize("name", FILES)
def test_waits_poll_atomics(name):
    for loop in _waits(name):
        assert any(p in loop for p in POLLS), loop
        assert not any(p in loop for p in PLAIN), loop


def test_waits_are_found():
    assert sum(len(_waits(name)) for name in FILES) >= 3
