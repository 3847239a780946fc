"""The largest launches that vtdge_region_step is taken for, class of rows by class, against the separate operators bit for bit;
one sample more is refused."""
import pytest
import torch

import test_gpu_region_step as step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,C,dtype,mode", [(144, 384, "bf16", "records"), (512, 192, "bf16", "norm"), (256, 768, "bf16", "norm"),
                                            (700, 192, "f32", "norm"), (128, 384, "f32", "norm"), (48, 768, "f32", "norm")])
def test_the_most_regions(dev, B, C, dtype, mode):
    from vtpack_amd import _lib
    step.test_against_the_separate_operators(dev, B, 4, 4, C, 1, dtype, mode, B % 32 == 0)
    code = _lib.BF16 if dtype == "bf16" else _lib.F32
    assert _lib.load().vtdge_region_step_fits(B + 1, 16, 16, C, 1, code) == 0
