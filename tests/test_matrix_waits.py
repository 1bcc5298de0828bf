"""Kernels with matrix instructions hold no instruction written in inline asm.

After a matrix instruction a vector instruction that reads or overwrites its
registers must come a number of cycles later; the hardware does not hold it
back, the compiler puts the waits in, and only for instructions it knows.  An
asm statement with instructions in it may land in such a place without a wait.
Empty templates (they only hide a value from the compiler) are allowed."""
import glob
import os
import re

import pytest

ROOT = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pico_amd")


def test_no_asm_instruction_in_sources_with_matrix_instructions():
    seen = 0
    for path in glob.glob(os.path.join(ROOT, "csrc", "*")):
        text = open(path).read()
        if "__builtin_amdgcn_mfma" not in text:
            continue
        seen += 1
        for m in re.finditer(r"\basm\s*(?:volatile)?\s*\(\s*\"([^\"]*)\"", text):
            assert m.group(1).strip() == "", (os.path.basename(path), m.group(1))
    assert seen


def test_no_asm_instruction_in_built_matrix_kernels():
    path = os.path.join(ROOT, "_build", "merkle_gfx950.s")
    if not os.path.exists(path):
        pytest.skip("no device assembly beside the library (the build writes it)")
    kernels = re.split(r"\n(?=_ZN\w+:)", open(path).read())
    checked = 0
    for k in kernels:
        body = k.split(".Lfunc_end")[0]
        if "v_mfma_" not in body:
            continue
        checked += 1
        for block in re.findall(r"#ASMSTART(.*?);;?#ASMEND", body, re.S):
            code = [x for x in block.splitlines() if x.strip() and not x.strip().startswith(";")]
            assert not code, (k.split(":")[0], code)
    assert checked
