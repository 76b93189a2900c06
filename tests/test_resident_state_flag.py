"""A resident grid that has lost a block is given up, and the launched kernels
carry on from the state it began with, unless a block has raised GS_WRITTEN:
whatever stores the solver state or vectors at the end of such a kernel raises
that flag too (csrc/isph_resident.hip, csrc/isph_streamed.hip)."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "beach_slope_confined_amd", "csrc")


def functions(text):
    """Bodies of the top-level functions, by the braces."""
    depth, start = 0, 0
    for m in re.finditer(r"[{}]", text):
        if m.group() == "{":
            if depth == 0:
                start = m.end()
            depth += 1
        else:
            depth -= 1
            if depth == 0:
                yield text[start:m.start()]


@pytest.mark.parametrize("name,stores", [("isph_resident.hip", 2), ("isph_streamed.hip", 1)])
def test_state_stores_raise_the_flag(name, stores):
    text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, name)).read())
    text = re.sub(r"namespace (isph|host) \{", "", text)
    found = 0
    for body in functions(text):
        for m in re.finditer(r"\*sc = ", body):
            found += 1
            # in the same thread, before the state
            assert "atomicOr(gs.state, GS_WRITTEN)" in body[:m.start()]
    assert found == stores
