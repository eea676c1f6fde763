"""CPU check of the pinned copies (cdmf_amd/csrc/host_pipe.h): its threads and
pieces over a restatement of the runtime's streams and events
(tests/native/pipe_check.cpp), with the thread and the address sanitizers."""
import os
import shutil
import subprocess

import pytest

from tests.helpers import ROOT


@pytest.mark.parametrize("sanitizer", ["thread", "address,undefined"])
def test_copies_through_pinned_pieces(tmp_path, sanitizer):
    inc = "/opt/rocm/include"
    if shutil.which("g++") is None or not os.path.exists(os.path.join(inc, "hip", "hip_runtime.h")):
        pytest.skip("no g++ or no HIP headers")
    out = str(tmp_path / "pipe_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-D__HIP_PLATFORM_AMD__", "-fsanitize=" + sanitizer,
                    "-I" + inc, "-I" + os.path.join(ROOT, "cdmf_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "pipe_check.cpp"), "-o", out], check=True)
    r = subprocess.run([out], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout[-2000:]
