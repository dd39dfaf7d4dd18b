"""The built SHA-256 kernels keep the ISA's distance between a VALU write of a VGPR and a DPP instruction with it.

CDNA wants two wait states between a VALU instruction that writes a VGPR and a DPP instruction that reads it.  The
compiler keeps them in its own code, not inside inline assembly, where the rounds are: every DPP instruction's
VGPRs, the permuted source, the other one and the destination that masked lanes keep, are looked up in the
disassembly of the library built here.
"""
import re
import shutil
import struct
import subprocess
from pathlib import Path

import pytest

from kvsnap_amd.build import HIP_LIBRARY

OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin:/opt/rocm/lib/llvm/bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
WAIT_STATES = 2


def device_code(library):
    """The gfx950 code object in a HIP library's offload bundle."""
    data = Path(library).read_bytes()
    at = data.index(MAGIC)
    count, = struct.unpack_from("<Q", data, at + len(MAGIC))
    entry = at + len(MAGIC) + 8
    for _ in range(count):
        offset, size, length = struct.unpack_from("<QQQ", data, entry)
        if data[entry + 24:entry + 24 + length].endswith(b"gfx950"):
            return data[at + offset:at + offset + size]
        entry += 24 + length
    raise AssertionError("no gfx950 code in the library")


def vgprs(operand):
    found = re.fullmatch(r"v\[(\d+):(\d+)\]|v(\d+)", operand)
    if not found:
        return set()
    low, high, one = found.groups()
    return {int(one)} if one else set(range(int(low), int(high) + 1))


def too_close(lines):
    """(writer, DPP instruction) pairs with fewer than WAIT_STATES between them, in instruction order."""
    pairs, before = [], []                     # before: (text, VGPRs written, wait states), the latest last
    for line in lines:
        text = line.split("//")[0].strip()
        if not text or text.endswith(":"):
            continue
        name, _, rest = text.partition(" ")
        operands = [operand.strip().split(" ")[0] for operand in rest.split(",")]
        if name.endswith("_dpp"):
            uses, waited = set().union(*map(vgprs, operands)), 0
            for writer, written, states in reversed(before):
                if waited >= WAIT_STATES:
                    break
                if written & uses:
                    pairs.append((writer, text))
                waited += states
        written = vgprs(operands[0]) if name.startswith("v_") and not name.startswith("v_cmp") else set()
        before = before[-8:] + [(text, written, int(operands[0], 0) + 1 if name == "s_nop" else 1)]
    return pairs


def test_the_checker():
    add = "v_add_u32_dpp v1, v2, v1 row_half_mirror row_mask:0xf bank_mask:0x5"
    assert too_close(["v_mov_b32_e32 v2, v9", "v_mov_b32_e32 v3, v9", add])
    assert too_close(["v_mov_b32_e32 v1, v9", add]) and too_close([add, "s_nop 0", add])
    assert not too_close(["v_mov_b32_e32 v2, v9", "s_nop 1", add])
    assert not too_close(["v_add3_u32 v2, v1, v1, v1", "s_nop 0", "v_mov_b32_e32 v3, v9", add])
    assert not too_close(["v_mov_b32_e32 v4, v1", add])


@pytest.mark.skipif(OBJDUMP is None or not HIP_LIBRARY.exists(), reason="needs llvm-objdump and the built library")
def test_dpp_instructions_keep_two_wait_states_from_their_operands_writes(tmp_path):
    (tmp_path / "device.co").write_bytes(device_code(HIP_LIBRARY))
    listing = subprocess.run([OBJDUMP, "-d", str(tmp_path / "device.co")], check=True, capture_output=True,
                             text=True).stdout
    kernels = {}
    for part in re.split(r"^[0-9a-f]+ <", listing, flags=re.M)[1:]:
        name, _, body = part.partition(">:")
        if "sha256" in name or "sha_round_probe" in name:
            kernels[name] = body.splitlines()
    assert len(kernels) >= 8 and all(any("_dpp" in line for line in lines) for lines in kernels.values())
    assert {name: pairs for name, lines in kernels.items() if (pairs := too_close(lines))} == {}
