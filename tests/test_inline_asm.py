"""Inline assembly in the kernels: the compiler puts the waits that the hardware does not make by itself only in front of (and
behind) instructions that it knows, so what stands in an asm statement brings its own."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "customize-block-sparse-attention-with-triton_amd", "csrc")


def statements():
    """(file, instructions) of every asm statement that holds any."""
    out = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip"))):
        text = re.sub(r"//[^\n]*", "", open(path).read())
        for m in re.finditer(r"\basm\s*(?:volatile)?\s*\(\s*((?:\"(?:[^\"\\]|\\.)*\"\s*)+)", text):
            code = "".join(re.findall(r"\"((?:[^\"\\]|\\.)*)\"", m.group(1)))
            lines = [x.strip() for x in code.replace("\\t", " ").split("\\n") if x.strip()]
            if lines:
                out.append((os.path.basename(path), lines))
    return out


def test_no_vector_arithmetic():
    """A vector instruction in an asm statement may read what a matrix instruction has not finished, which needs up to 18 wait states."""
    found = statements()
    assert len(found) >= 5
    assert not [(f, x) for f, s in found for x in s if x.startswith("v_")]
