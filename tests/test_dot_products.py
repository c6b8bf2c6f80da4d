"""A dot product's result is read by an instruction of another opcode too early unless wait states stand between the two, and only the compiler
places them: it knows nothing of an instruction inside inline assembly. Dot products are therefore left to its builtins everywhere."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tim-vx_amd", "csrc")


def test_no_dot_product_in_inline_assembly():
    sources = sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h")))
    assert len(sources) > 20
    found = []
    for path in sources:
        text = open(path).read()
        for m in re.finditer(r"\basm\b[^;]*;", text):
            if "v_dot" in m.group(0):
                found.append((os.path.basename(path), text[:m.start()].count("\n") + 1))
    assert not found, found
