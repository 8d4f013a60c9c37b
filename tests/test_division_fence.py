"""The one-launch divisions publish a workgroup's flagged cells to the one that appends them: every wave
that flags a cell writes back to the device's coherence point, and waits, before its workgroup's barrier
(the barrier instruction itself waits for LDS only).  Read from the built library's own gfx950 code."""
import os
import re
import shutil
import subprocess

import pytest

from cil_cuda_amd import abi

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no AMD assembly tools")
def test_flags_are_written_back_before_the_barrier(tmp_path):
    lib = tmp_path / "lib.so"
    shutil.copy(abi.LIB_PATH, lib)
    subprocess.run([OBJDUMP, "--offloading", lib.name], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    code = next(p for p in tmp_path.iterdir() if p.name.endswith("gfx950"))
    names = set(re.findall(r"\s(_Z\w*k?b?_div_fused\w*?)\n", subprocess.run(
        [OBJDUMP, "-t", code], check=True, capture_output=True, text=True).stdout))
    assert len(names) >= 6  # three division models, alone and in a batch
    for name in names:
        out = subprocess.run([OBJDUMP, "-d", f"--disassemble-symbols={name}", code], check=True, capture_output=True,
                             text=True).stdout
        head = out.split("s_barrier")[0].splitlines()
        at = [i for i, line in enumerate(head) if "buffer_wbl2 sc1" in line]
        assert at and any("s_waitcnt vmcnt(0)" in line for line in head[at[-1]:at[-1] + 3]), name
