"""The tile kernels read one matrix's arguments at once. A shared launch lets a workgroup's arguments be a later matrix's; where
the compiler then chooses between the two addresses of each argument and loads it where it is used, every launch, of one matrix
too, waits for one trip to memory after the other. This compiles the load-to-LDS instances to assembly (no GPU needed): no
scalar load goes through such a chosen address, that is, at offset 0 of a pointer other than the argument block's."""
import os
import re
import subprocess

import pytest

from tests.test_stream_loop_waits import CSRC, HIPCC

FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S"]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_arguments_are_loaded_from_the_argument_block(tmp_path):
    out = str(tmp_path / "b8.s")
    r = subprocess.run([HIPCC, *FLAGS, os.path.join(CSRC, "qmm_dma_b8.hip"), "-o", out], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    text = open(out).read()
    kernels = re.split(r"\n(?=_ZN3mtq14qmm_dma_kernel\w+:)", text)[1:]
    assert kernels
    for k in kernels:
        name, code = k.split(":", 1)
        code = code[:code.index("s_endpgm")]
        if re.search(r"kernelI(Li\d+E){5}Lb1E", name):   # grouped: one set of arguments, and the table of tiles behind a pointer
            continue
        loads = re.findall(r"s_load_dword\w* \S+, (s\[\d+:\d+\]), (\S+)", code)
        assert loads
        chosen = [l for l in loads if l[1] == "0x0" and l[0] != loads[0][0]]
        assert not chosen, (name, chosen)
