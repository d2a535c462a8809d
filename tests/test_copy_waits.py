"""The wait states between a global -> LDS copy and the writes of the scalar
registers it reads, in the compiled device code. The copies are inline assembly
(hy3x_dma.h), so the compiler inserts none of these waits. CPU only (hipcc)."""
import os
import re
import subprocess

import pytest

from hy3_amd import build

M0_STATES, BASE_STATES = 1, 5  # after a scalar write of m0; after a vector write of the base


def wait_states(instruction):
    m = re.match(r"s_nop (\w+)", instruction)
    return int(m.group(1), 0) + 1 if m else 1


def scalar_pair(operand):
    m = re.search(r"s\[(\d+):(\d+)\]", operand)
    return set(range(int(m.group(1)), int(m.group(2)) + 1)) if m else set()


def short_waits(asm):
    """(number of copies, descriptions of those that follow a write too closely),
    in program order: a distance over a branch counts as the lines between."""
    code = [line.split(";")[0].strip() for line in asm.splitlines()]
    code = [c for c in code if c and not c.startswith(".") and not c.endswith(":")]
    copies, bad = 0, []
    for i, c in enumerate(code):
        if not c.startswith("global_load_lds"):
            continue
        copies += 1
        base, states, j = scalar_pair(c), 0, i - 1
        while j >= 0 and states < BASE_STATES:
            w = code[j]
            if states < M0_STATES and re.match(r"s_\w+ m0,", w):
                bad.append(f"{w} | {c}")
            m = re.match(r"v_\w+ (s\d+|s\[\d+:\d+\]|m0),", w)
            if m and (m.group(1) == "m0" or base & (
                    scalar_pair(m.group(1)) or {int(m.group(1)[1:])})):
                bad.append(f"{w} | {states} | {c}")
            states += wait_states(w)
            j -= 1
    return copies, bad


def test_short_waits_finds_them():
    copy = "global_load_lds_dwordx4 v1, s[4:5]\n"
    assert short_waits("s_mov_b32 m0, s3\n" + copy) == (1, ["s_mov_b32 m0, s3 | " + copy.strip()])
    assert short_waits("s_mov_b32 m0, s3\ns_nop 0\n" + copy) == (1, [])
    near = "v_readfirstlane_b32 s5, v0\ns_mov_b32 m0, s3\ns_nop 0\n" + copy
    assert len(short_waits(near)[1]) == 1
    assert short_waits(near.replace("s_nop 0", "s_nop 3")) == (1, [])
    assert short_waits(near.replace(" s5", " s6")) == (1, [])


@pytest.mark.parametrize("src", [s for s in build.sources() if "mfma" in os.path.basename(s)],
                         ids=os.path.basename)
def test_copies_wait_for_their_scalar_registers(src):
    asm = subprocess.run([*build.compile_command(src), "-S", "--cuda-device-only", "-o", "-"],
                         check=True, capture_output=True, text=True).stdout
    copies, bad = short_waits(asm)
    assert not bad, bad[:5]
    assert copies or "mfma_few" in src  # the whole-row kernel uses none
