"""Assembly of the fold-in kernels: a vector instruction that writes a scalar
register (a lane read, a comparison) is followed by at least two wait states
before a vector instruction reads that register.  The compiler places them for
its own instructions; it does not look into inline assembly."""
import os
import re
import subprocess

import pytest

from tests.helpers import ROOT

WAIT = 2


def _scalars(text):
    """Scalar registers named in an operand list."""
    out = set()
    for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        out.update(range(int(a), int(b) + 1))
    out.update(int(a) for a in re.findall(r"\bs(\d+)\b", text))
    if re.search(r"\bvcc\b", text):
        out.add("vcc")
    return out


def hazards(asm):
    bad, age = [], {}  # age: register -> wait states since its write
    for no, line in enumerate(asm.splitlines(), 1):
        ins = line.split(";")[0].strip()
        if not ins or ins.startswith("."):
            if re.match(r"\.L\S+:", ins):
                age = {}  # a branch target: nothing is known of what ran before
            continue
        if ins.endswith(":"):
            age = {}
            continue
        op, _, args = ins.partition(" ")
        if op == "s_nop":
            step = int(args) + 1
        else:
            step = 1
            if op.startswith("v_"):
                dst, _, src = args.partition(",")
                writes = _scalars(dst) if op.startswith(("v_readlane", "v_readfirstlane", "v_cmp")) else set()
                if any(age.get(r, WAIT) < WAIT for r in _scalars(src if writes else args)):
                    bad.append("%d: %s" % (no, ins))
        age = {r: a + step for r, a in age.items() if a + step < WAIT}
        if op.startswith("v_") and writes:
            age.update({r: 0 for r in writes})
    return bad


def test_the_check_finds_an_unwaited_read():
    seq = "v_readlane_b32 s4, v1, 3\n%s\tv_writelane_b32 v0, s4, 3\n"
    assert hazards(seq % "") and hazards(seq % "s_nop 0\n") and not hazards(seq % "s_nop 1\n")


def test_fold_kernels_wait_after_lane_reads(tmp_path):
    from cdmf_amd import _build as B
    if not os.path.exists(B.HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path / "fold.s")
    subprocess.run([B.HIPCC, *B.HIP_FLAGS, "-I" + B.INC, "-I" + B.CSRC, "-I" + os.path.join(B.CSRC, "kernels"), "-S",
                    "--cuda-device-only", os.path.join(B.CSRC, "kernels", "foldin_kernels.hip"), "-o", out], check=True,
                   stderr=subprocess.DEVNULL)
    asm = open(out).read()
    assert asm.count("v_readlane_b32") > 100
    bad = hazards(asm)
    assert not bad, "%d reads too early, the first: %s" % (len(bad), bad[0])
