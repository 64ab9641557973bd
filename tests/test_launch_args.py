"""The argument block of a launch: kernels take as many bytes as the library hands over, products only their own."""
import os
import re
import subprocess

import pytest

from heron_amd import backend as B
from launch_args import library
from test_template_stores import DEFINES


@pytest.mark.parametrize("op", [0, 1])
def test_kernels_take_what_a_launch_hands_over(op, tmp_path):
    out = tmp_path / "template.s"
    subprocess.run([os.environ.get("HRN_HIPCC", "/opt/rocm/bin/hipcc"), "-x", "hip", "--offload-device-only", "--offload-arch=gfx950", "-O3", "-std=c++17",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-S", os.path.join(B.CSRC, "mfma_gemm_template.hip"), "-o", str(out)] +
                   ["-DHRN_%s=%d" % kv for kv in dict(DEFINES, OP=op).items()], check=True, capture_output=True)
    sizes = re.findall(r"\.size: +(\d+)\n +\.value_kind: +by_value", out.read_text())
    assert sizes and {int(s) for s in sizes} == {library().args_bytes(op)}


def test_a_product_carries_no_conv():
    assert library().args_bytes(0) + 150 <= library().args_bytes(1)
