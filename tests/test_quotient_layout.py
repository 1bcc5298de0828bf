"""The windowed quotient kernel's interpreter loop starts where its dispatch was
measured to run fastest: at byte 8 of a 32-byte line of instructions, whatever
code stands in front of it (other places cost up to 5%)."""
import os
import re
import struct
import subprocess

import pytest

OBJ = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pico_amd", "_build", "quotient.o")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def _device_code(blob, triple_end):
    """The gfx950 code object in a host object's offload bundle."""
    at = blob.index(b"__CLANG_OFFLOAD_BUNDLE__")
    n, p = struct.unpack_from("<Q", blob, at + 24)[0], at + 32
    for _ in range(n):
        off, size, length = struct.unpack_from("<QQQ", blob, p)
        name = blob[p + 24:p + 24 + length].decode()
        p += 24 + length
        if name.endswith(triple_end):
            return blob[at + off:at + off + size]
    raise AssertionError("no gfx950 code in the object")


@pytest.mark.parametrize("prime", [2130706433, 2013265921])
def test_interpreter_loop_placement(tmp_path, prime):
    if not (os.path.exists(OBJ) and os.path.exists(OBJDUMP)):
        pytest.skip("no object file beside the library, or no disassembler (the build has both)")
    elf = tmp_path / "quotient.co"
    elf.write_bytes(_device_code(open(OBJ, "rb").read(), "gfx950"))
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(elf)], check=True, capture_output=True, text=True).stdout
    m = re.search(rf"^(\w+) <_ZN2pg15quotient_kernelINS_10MontyFieldILj{prime}E\w+>:\n(.*?)(?:\n\n|\Z)", text, re.M | re.S)
    start, body = int(m.group(1), 16), m.group(2)
    backward = []  # (target, branch) of the loops of more than 4 KiB
    for at, to in re.findall(r"s_c?branch\w* \d+\s+// (\w+):.*?<\S+\+0x(\w+)>", body):
        at, to = int(at, 16) - start, int(to, 16)
        if at - to > 4096:
            backward.append(to)
    assert start % 32 == 0 and min(backward) % 32 == 8, (hex(start), [hex(x) for x in backward])
