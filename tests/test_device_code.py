"""Checks on the gfx950 device code of the attention kernels (CPU only: hipcc cross-compiles).

M0.  The key-block DMA (``dma16`` in ``csrc/attn_common.h``) writes M0 in inline
assembly and declares it clobbered, which hipcc does not honour for a
reserved register.  That is only sound while no other instruction of these
kernels touches M0, so the assembly is checked: every write of M0 is the
DMA's own ``s_mov_b32 m0, <SGPR>`` / ``s_nop 0`` / ``global_load_lds_dwordx4``
sequence, and nothing else names M0.

Wait states.  The compiler keeps the distances that the hardware does not check
itself between instructions of its own, but does not look into inline assembly.
An SGPR that a vector instruction wrote (v_readfirstlane, v_readlane, a compare)
may be read by a vector memory instruction five wait states later, so the DMA's
address must not come from one directly, and by another vector instruction two
wait states later.
"""

import os
import re
import shutil
import subprocess

import pytest

from sol_attn_amd import _build

HIPCC = shutil.which("hipcc") or ("/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else None)


@pytest.fixture(scope="module")
def attention_asm(tmp_path_factory):
    """Lines of the attention kernels' device assembly."""
    if HIPCC is None:
        pytest.skip("hipcc not installed")
    src = os.path.join(_build.CSRC, "attention.hip")
    asm = tmp_path_factory.mktemp("asm") / "attention.s"
    cmd = [HIPCC, *_build.compile_flags(), "-Wno-inline-asm", "--cuda-device-only", "-S", src, "-o", str(asm)]
    res = subprocess.run(cmd, capture_output=True, text=True, timeout=900)
    assert res.returncode == 0, res.stderr[-2000:]
    return asm.read_text().splitlines()


def test_only_the_key_block_dma_uses_m0(attention_asm):
    lines = [l.split(";")[0].strip() for l in attention_asm]
    code = [l for l in lines if l and not l.startswith(".") and not l.endswith(":")]
    writes = 0
    for i, line in enumerate(code):
        if not re.search(r"\bm0\b", line):
            continue
        # The asm statement's scalar operand: any SGPR (vcc_lo/vcc_hi are SGPRs too).
        assert re.fullmatch(r"s_mov_b32 m0, (s\d+|vcc_lo|vcc_hi)", line), f"unexpected use of M0: {line!r}"
        assert code[i + 1] == "s_nop 0" and code[i + 2].startswith("global_load_lds_dwordx4"), \
            f"M0 write not followed by the DMA: {code[i:i + 3]!r}"
        writes += 1
    assert writes > 0  # the DMA helper is in the build at all


def _sgprs(operand):
    """The SGPRs an operand names."""
    name = operand.split()[0] if operand.split() else ""
    if name in ("vcc", "vcc_lo", "vcc_hi"):
        return {"vcc_lo", "vcc_hi"} if name == "vcc" else {name}
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", name) or re.fullmatch(r"s(\d+)()", name)
    return set(range(int(m[1]), int(m[2] or m[1]) + 1)) if m else set()


def _sgpr_distances(lines):
    """(line, in inline assembly, wait states since a vector instruction wrote one of its SGPRs) of every
    instruction that reads an SGPR whose last writer is a vector instruction."""
    written, state, inline = {}, 0, False
    for line in lines:
        if "#ASMSTART" in line or "#ASMEND" in line:
            inline = "#ASMSTART" in line
            continue
        text = line.split(";")[0].strip()
        if not text or text.startswith(".") or text.endswith(":"):
            continue
        op, _, rest = text.partition(" ")
        args = [a.strip() for a in rest.split(",")]
        if op == "s_nop":
            state += int(args[0], 0) + 1
            continue
        loads = op.startswith(("global_", "buffer_", "ds_", "flat_"))
        reads = set().union(*(_sgprs(a) for a in (args if loads else args[1:])))
        ages = [state - written[r] - 1 for r in reads if r in written]
        if ages:
            yield text, inline, min(ages)
        if op.startswith("v_"):
            for r in _sgprs(args[0]):
                written[r] = state
        elif op.startswith("s_"):
            for r in _sgprs(args[0]):
                written.pop(r, None)
        state += 1


def test_dma_addresses_keep_their_distance_from_vector_writes(attention_asm):
    close = [(text, age) for text, inline, age in _sgpr_distances(attention_asm)
             if inline and text.startswith("global_load_lds") and age < 5]
    assert not close, f"{len(close)} DMAs read an SGPR a vector instruction has just written: {close[:4]!r}"


def test_inline_vector_instructions_keep_their_distance_from_vector_writes(attention_asm):
    close = [(text, age) for text, inline, age in _sgpr_distances(attention_asm)
             if inline and text.startswith("v_") and age < 2]
    assert not close, f"{len(close)} vector instructions read an SGPR another has just written: {close[:4]!r}"
