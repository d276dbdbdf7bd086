"""The tiles that move their operands to LDS directly reload a buffer right after
the barrier that ends the reads of it: each barrier has to wait for the wave's
own LDS reads.  Read in the assembly that the sources compile to: in the FP64
tile (gemm64.hpp) the barrier's own wait covers them; in the bf16x3 ones
(sig3mtile.hpp, sigtile.hpp) an earlier wait, ahead of the products that use
them, has to."""
import os
import re
import subprocess

import pytest

from ecalj_amd import build


def assembly(source, tmp_path):
    src, out = os.path.join(build.HERE, "csrc", source), str(tmp_path / "a.s")
    flags = [f for f in build.FLAGS if f != "-shared"]
    subprocess.run([build.HIPCC, *flags, "-S", "--cuda-device-only", "-I", os.path.join(build.ROOT, "include"),
                    "-I", os.path.join(build.HERE, "csrc"), src, "-o", out], check=True, capture_output=True)
    code = [ln.split(";")[0].strip() for ln in open(out)]
    return [ln for ln in code if re.match(r"[a-z]\w+ ?|\.LBB|_Z\w+:", ln)]


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
def test_every_stage_barrier_waits_for_the_lds_reads(tmp_path):
    code = assembly("gemm64.hip", tmp_path)
    barriers = [i for i, ln in enumerate(code) if ln.startswith("s_barrier")]
    assert len(barriers) >= 8  # a main loop and a tail in each of four kernels
    for i in barriers:
        wait = next(j for j in range(i, -1, -1) if code[j].startswith(("s_waitcnt", "ds_read", "ds_write", ".LBB")))
        assert code[wait].startswith("s_waitcnt") and "lgkmcnt(0)" in code[wait], code[wait:i + 1]


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
@pytest.mark.parametrize("source", ["sigmodes.hip", "sig3m.hip", "zmelbf3.hip"])
def test_no_lds_read_is_in_flight_at_a_barrier(source, tmp_path):
    flight, barriers = 0, 0
    for ln in assembly(source, tmp_path):  # in program order; LDS reads return in order
        count = re.search(r"lgkmcnt\((\d+)\)", ln)
        if ln.startswith("_Z"):
            flight = 0
        elif ln.startswith("ds_read"):
            flight += 1
        elif count:
            flight = min(flight, int(count.group(1)))
        elif ln.startswith("s_barrier"):
            barriers += 1
            assert flight == 0
    assert barriers > 0
