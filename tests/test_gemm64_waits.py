"""The FP64 complex tile (gemm64.hpp) reloads an LDS buffer right after the
barrier that ends the reads of it: each barrier has to wait for the wave's own
LDS reads.  Read in the assembly that the source compiles to."""
import os
import re
import subprocess

import pytest

from ecalj_amd import build


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
def test_every_stage_barrier_waits_for_the_lds_reads(tmp_path):
    src = os.path.join(build.HERE, "csrc", "gemm64.hip")
    out = str(tmp_path / "gemm64.s")
    flags = [f for f in build.FLAGS if f != "-shared"]
    subprocess.run([build.HIPCC, *flags, "-S", "--cuda-device-only", "-I", os.path.join(build.ROOT, "include"),
                    "-I", os.path.join(build.HERE, "csrc"), src, "-o", out], check=True, capture_output=True)
    code = [ln.split(";")[0].strip() for ln in open(out)]
    code = [ln for ln in code if re.match(r"[a-z]\w+ ?|\.LBB", ln)]
    barriers = [i for i, ln in enumerate(code) if ln.startswith("s_barrier")]
    assert len(barriers) >= 8  # a main loop and a tail in each of four kernels
    for i in barriers:
        wait = next(j for j in range(i, -1, -1) if code[j].startswith(("s_waitcnt", "ds_read", "ds_write", ".LBB")))
        assert code[wait].startswith("s_waitcnt") and "lgkmcnt(0)" in code[wait], code[wait:i + 1]
