"""Shapes of linear_lora_bwd's fake results: empty where a gradient is not asked for."""

import itertools

import pytest
import torch
from torch._subclasses import FakeTensorMode

from ojasx_amd import ops


@pytest.mark.parametrize("need", itertools.product((False, True), repeat=3))
@pytest.mark.parametrize("shape", [(6,), (2, 3)])
def test_fake_shapes(need, shape):
    n, k, r, gs = 48, 64, 4, 16
    with FakeTensorMode(allow_non_fake_inputs=False):
        bf16 = torch.bfloat16
        gx, ga, gb = ops.linear_lora_bwd(
            torch.empty(*shape, k, dtype=bf16), torch.empty(*shape, n, dtype=bf16),
            torch.empty(n * k * 3 // 16, dtype=torch.uint8),
            torch.empty(n * k // gs, dtype=torch.float16), torch.empty(k, r, dtype=bf16),
            torch.empty(r, n, dtype=bf16), 1.0, ops.FMT_TERNARY, n, k, gs, *need)
    assert gx.shape == ((6, k) if need[0] else (0, k))
    assert ga.shape == ((k, r) if need[1] else (0, r))
    assert gb.shape == ((r, n) if need[2] else (r, 0))
    assert gx.dtype == ga.dtype == gb.dtype == torch.bfloat16
