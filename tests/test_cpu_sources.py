"""Properties of the device sources that no run on a GPU shows."""
import os
import re

from conftest import ROOT


def test_dpp_statements_bring_their_wait_states():
    """Two wait states have to lie between a VALU write and a DPP read, and the
    compiler does not count them for a DPP inside an asm string: every statement
    that holds one begins with them (the read before any operand's own write
    included), whatever the compiler puts in front of it."""
    text = open(os.path.join(ROOT, "caps_amd", "csrc", "waves.hip")).read()
    macros = dict(re.findall(r"^#define (\w+)(?:\([^)]*\))? (.*)$", text, flags=re.M))
    dpp = {k for k, v in macros.items() if "row_newbcast" in v}
    while True:   # macros made of such macros
        more = {k for k, v in macros.items() if any(re.search(r"\b%s\b" % d, v) for d in dpp)} - dpp
        if not more:
            break
        dpp |= more
    found = 0
    for template in re.findall(r"\basm volatile\(([^:]*):", text):
        words = re.findall(r'"(?:[^"\\]|\\.)*"|\w+', template)
        if "row_newbcast" not in template and not any(w in dpp for w in words):
            continue
        found += 1
        first = macros.get(words[0], words[0])
        assert first.startswith('"s_nop 1\\n"'), template
    assert found > 2
