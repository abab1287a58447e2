"""Wait states between a vector instruction and the matrix instruction that reads its result.

On gfx950 two instructions (or s_nop) have to lie between.  The compiler keeps that distance for its own instructions
and cannot for one written as inline asm, so the few-rows matmul, which dequantizes right before its matrix
instructions, is compiled to assembly and every pair is checked."""
import os
import re
import subprocess

import pytest

from lisa_amd import build

WAITS = 2


def _regs(op):
    m = re.fullmatch(r"v\[(\d+):(\d+)\]", op)
    if m:
        return range(int(m[1]), int(m[2]) + 1)
    m = re.fullmatch(r"v(\d+)", op)
    return [int(m[1])] if m else []


def short_waits(asm):
    """(matrix instructions, those that read a register fewer than WAITS wait states after a vector write)"""
    seen, short, now, wrote = 0, [], 0, {}
    for line in asm.splitlines():
        line = line.split(";")[0].strip()
        if re.match(r"[.\w$]+:", line):  # (a label: other ways lead here)
            wrote = {}
            continue
        if not line or line.startswith("."):
            continue
        op, _, rest = line.partition(" ")
        args = [a.strip() for a in re.split(r",\s*(?![^\[]*\])", rest)]
        if op.startswith("v_mfma"):
            seen += 1
            for a in args[1:3]:
                if any(now - wrote.get(r, now - WAITS - 1) - 1 < WAITS for r in _regs(a)):
                    short.append(line)
                    break
        for r in _regs(args[0]):
            wrote.pop(r, None)
            if op.startswith("v_") and not op.startswith("v_mfma"):
                wrote[r] = now
        now += 1 + (int(args[0], 0) if op == "s_nop" else 0)
    return seen, short


def test_scan_counts_wait_states():
    cvt, use = "v_cvt_pk_f16_f32 v4, v8, v9", "v_mfma_f32_32x32x16_f16 v[16:31], v[4:7], v[0:3], v[16:31]"
    for between, bad in ((["s_nop 1"], 0), (["s_nop 0"], 1), ([], 1), (["v_mov_b32_e32 v9, 0", "s_nop 0"], 0),
                         (["v_mov_b32_e32 v9, 0", "v_mov_b32_e32 v5, 0"], 1)):
        assert [len(x) if isinstance(x, list) else x for x in short_waits("\n".join([cvt, *between, use]))] == [1, bad]


@pytest.mark.parametrize("unit", ["qmm_rows_h4.hip", "qmm_rows_b4.hip"])
def test_few_rows_matmul_waits(tmp_path, unit):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path / "unit.s")
    subprocess.run([build.HIPCC, *build.FLAGS, "-x", "hip", "--cuda-device-only", "-S", os.path.join(build.CSRC, unit),
                    "-o", out], check=True, capture_output=True)
    seen, short = short_waits(open(out).read())
    assert seen > 0 and not short, f"{len(short)} of {seen}: {short[:3]}"
