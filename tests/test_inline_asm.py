"""Inline assembly in the kernels declares what it writes behind its operands:
a statement that sets m0 names it as clobbered, and one that fills LDS by DMA
names memory too, so that the compiler neither keeps a value of its own in m0
nor moves an LDS read across the fill."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "light-rocm-runtime_amd", "csrc")


def statements():
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        with open(path) as f:
            text = f.read()
        for m in re.finditer(r"\basm\s+volatile\s*\((.*?)\);", text, re.S):
            yield f"{os.path.basename(path)}:{text.count(chr(10), 0, m.start()) + 1}", m.group(1)


def test_clobbers_are_declared():
    seen = 0
    for where, body in statements():
        code = re.split(r'"\s*:', body, maxsplit=1)[0]
        clobbers = body.rsplit(":", 1)[-1] if body.count(":") >= 3 else ""
        if re.search(r"\b[sv]_\w+ m0\b", code):
            seen += 1
            assert '"m0"' in clobbers, where
        if "global_load_lds" in code or "s_waitcnt" in code or "s_barrier" in code:
            seen += 1
            assert '"memory"' in clobbers, where
    assert seen >= 8
