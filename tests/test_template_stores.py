"""Results of any alignment: what the template tells the compiler about the addresses it stores results to (no GPU needed).  Instances
with epilogue 0, and the sum of split-K slices with any epilogue, may claim no more than an element's alignment."""
import os
import re
import subprocess

import pytest

from heron_amd import backend as B

DEFINES = dict(DTYPE=0, OP=0, BM=128, BN=128, BKB=128, WM=2, WN=2, MFMA=32, STAGES=2, SWZ=1, EPI=0, WPE=0, CONVWIN=0, PERSIST=0, SPLITK=0,
               SCHED=1, LSPREAD=2, COLSUM=0, NTSTORE=0, PART=0)
# staged and unstaged (strips of 16 columns) fp16, both store policies; int32; split-K with either epilogue; last: aligned results
CASES = [(dict(), 2), (dict(NTSTORE=1), 2), (dict(BN=64, WN=4, MFMA=16), 2), (dict(DTYPE=1), 4), (dict(SPLITK=1), 2), (dict(SPLITK=1, DTYPE=1, EPI=1), 4),
         (dict(EPI=1), 16)]


@pytest.mark.parametrize("change,align", CASES)
def test_alignment_of_result_stores(change, align, tmp_path):
    out = tmp_path / "template.ll"
    subprocess.run([os.environ.get("HRN_HIPCC", "/opt/rocm/bin/hipcc"), "-x", "hip", "--offload-device-only", "--offload-arch=gfx950", "-O3", "-std=c++17",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-S", "-emit-llvm", os.path.join(B.CSRC, "mfma_gemm_template.hip"),
                    "-o", str(out)] + ["-DHRN_%s=%d" % kv for kv in dict(DEFINES, **change).items()], check=True, capture_output=True)
    found = re.findall(r"store (<4 x \w+>|i64) [^,]*, ptr addrspace\(1\) [^,]*, align (\d+)", out.read_text())
    assert found
    assert {int(a) for _, a in found} <= {align, min(align, 8)}, set(found)
