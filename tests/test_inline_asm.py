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


def test_copies_into_lds():
    """m0 is written at least one instruction in front of the copy that uses it, and the base address is in a register that a
    scalar instruction of the same statement wrote (after a vector instruction, a spilled value's way back, five states are needed)."""
    copies = [(f, s) for f, s in statements() if any(x.startswith("global_load_lds") for x in s)]
    assert copies
    for f, s in copies:
        first = next(i for i, x in enumerate(s) if x.startswith("global_load_lds"))
        m0 = [i for i, x in enumerate(s) if re.match(r"s_mov_b32 m0,", x)]
        assert m0 and m0[-1] + 1 < first, (f, s)
        written = {x.split()[1].rstrip(",") for x in s[:first] if x.startswith("s_mov_b64")}
        assert all(x.split(",")[1].split()[0] in written for x in s[first:]), (f, s)


def test_wide_stores():
    """The data of a store of more than 8 bytes may be overwritten two states later: the statement ends with them."""
    stores = [(f, s) for f, s in statements() if any(re.match(r"global_store_dwordx[34]", x) for x in s)]
    assert stores
    for f, s in stores:
        m = re.match(r"s_nop (\d+)$", s[-1])
        assert m and int(m.group(1)) >= 1, (f, s)
