"""Suites of single instances on the very tiles their instances name.  In their own files a default module launches what its callers
get: another tile of the instance wherever the grid leaves CUs idle, which most shapes there do."""
import functools

import pytest

import test_gpu_parity
from heron_amd import backend as B
from test_gpu_channels_first import test_equals_the_separate_passes  # noqa: F401
from test_gpu_deep import test_channels_first, test_conv_images_in_one_launch_and_apart, test_equals_the_plain_kernel  # noqa: F401
from test_gpu_direct_epilogue import test_rows_and_starts  # noqa: F401
from test_gpu_fuzz import test_sampled_instance  # noqa: F401
from test_gpu_parity import (test_bmm_f16, test_bmm_u8s8, test_caller_supplied_column_sums, test_conv2d_nhwc_f16,  # noqa: F401
                             test_conv2d_nhwc_u8s8_bit_exact, test_conv2d_u8s8_extremes_and_blocked_filter, test_conv_1x1_is_gemm,
                             test_gemm_f16_exact_cases, test_gemm_f16_within_tolerance, test_gemm_u8s8_bit_exact,
                             test_gemm_u8s8_extremes, test_template_variants)
from test_gpu_phased import test_k_tiles  # noqa: F401

pytestmark = pytest.mark.gpu
_mods = {}


@pytest.fixture(autouse=True)
def own(monkeypatch):
    monkeypatch.setattr(B, "Module", functools.partial(B.Module, own_tiles=True))
    monkeypatch.setattr(test_gpu_parity, "_mods", _mods)
