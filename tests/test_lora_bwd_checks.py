"""linear_lora_bwd refuses operands that do not fit the layer before anything is launched.

The op's body runs on CPU tensors here, with the device check let through and the library
replaced by one that records its calls.
"""

import contextlib

import pytest
import torch

from ojasx_amd import _native as N
from ojasx_amd import ops

OUT, IN, GS, R, ROWS = 48, 64, 16, 4, 6
CODE_BYTES = {ops.FMT_TERNARY: OUT * IN * 3 // 16, ops.FMT_E8: OUT * IN // 4,
              ops.FMT_ROOT: OUT * IN // 8}


class _Library:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *args: self.calls.append(name) or 0


@pytest.fixture
def library(monkeypatch):
    fake = _Library()
    monkeypatch.setattr(N, "lib", lambda: fake)
    monkeypatch.setattr(N, "require_device", lambda *tensors: torch.device("cpu"))
    monkeypatch.setattr(N, "stream_handle", lambda device: 0)
    monkeypatch.setattr(torch.cuda, "device", lambda device: contextlib.nullcontext())
    return fake


def _operands(fmt):
    bf16 = torch.bfloat16
    return dict(x=torch.zeros(ROWS, IN, dtype=bf16), grad_y=torch.zeros(ROWS, OUT, dtype=bf16),
                packed_weight=torch.zeros(CODE_BYTES[fmt], dtype=torch.uint8),
                block_scales=torch.zeros(OUT * IN // GS, dtype=torch.float16),
                lora_a=torch.zeros(IN, R, dtype=bf16), lora_b=torch.zeros(R, OUT, dtype=bf16),
                scaling=1.0, fmt=fmt, out_features=OUT, in_features=IN, group_size=GS,
                need_x=True, need_a=True, need_b=True)


@pytest.mark.parametrize("fmt", sorted(CODE_BYTES))
@pytest.mark.parametrize("shape", [(ROWS,), (2, 3)])
def test_operands_that_fit_are_taken(library, fmt, shape):
    args = _operands(fmt)
    args["x"] = args["x"].view(*shape, IN)
    args["grad_y"] = args["grad_y"].view(*shape, OUT)
    gx, ga, gb = ops.linear_lora_bwd(**args)
    assert gx.shape == (ROWS, IN) and ga.shape == (IN, R) and gb.shape == (R, OUT)
    assert library.calls == ["ojx_gemm_bwd_lora_workspace_bytes", "ojx_gemm_bwd_lora"]


@pytest.mark.parametrize("fmt", sorted(CODE_BYTES))
@pytest.mark.parametrize("name,change", [
    ("packed_weight", lambda t: t[:-1]),
    ("packed_weight", lambda t: t.to(torch.int32)),
    ("block_scales", lambda t: t[:-1]),
    ("block_scales", lambda t: t.view(torch.int16)),
    ("x", lambda t: t[:-1]),
    ("x", lambda t: t[:, :-1]),
    ("x", lambda t: t.view(2 * ROWS, IN // 2)),
    ("x", lambda t: t.float()),
    ("x", lambda t: t.half()),
    ("grad_y", lambda t: t[:-1]),
    ("grad_y", lambda t: t[:0]),
    ("grad_y", lambda t: t[:, :-1]),
    ("grad_y", lambda t: t.float()),
    ("grad_y", lambda t: t.double()),
    ("lora_a", lambda t: t[:-1]),
    ("lora_a", lambda t: t[:, :-1]),
    ("lora_a", lambda t: t.t()),
    ("lora_a", lambda t: t.float()),
    ("lora_b", lambda t: t[:-1]),
    ("lora_b", lambda t: t[:, :-1]),
    ("lora_b", lambda t: t.half()),
    ("group_size", lambda v: 0),
    ("group_size", lambda v: 6),
    ("fmt", lambda v: 3),
    ("out_features", lambda v: v + 1),
    ("in_features", lambda v: 2 * v),
])
def test_operands_that_do_not_fit_are_refused(library, fmt, name, change):
    args = _operands(fmt)
    args[name] = change(args[name])
    with pytest.raises(RuntimeError):
        ops.linear_lora_bwd(**args)
    assert not library.calls


def test_rank_is_bounded(library):
    for r in (0, ops.LORA_MAX_RANK + 1):
        args = _operands(ops.FMT_TERNARY)
        args["lora_a"], args["lora_b"] = args["lora_a"].new_zeros(IN, r), args["lora_b"].new_zeros(r, OUT)
        with pytest.raises(RuntimeError):
            ops.linear_lora_bwd(**args)
    assert not library.calls
