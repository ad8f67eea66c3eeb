"""linear_lora_bwd, the registered op of the adapter gradients, which compiled and traced
training reaches: the same bits as the eager extension's call for every choice of gradients,
and what a compiled layer and a backward under a dispatch mode run.
"""

import itertools

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import ojasx_amd
from ojasx_amd import _native as N
from ojasx_amd import ops

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
FMT = {1.5: ops.FMT_TERNARY, 2.0: ops.FMT_E8, 1.0: ops.FMT_ROOT}


def _layer(bitrate, dtype=torch.bfloat16, n=96, k=320, rank=8):
    torch.manual_seed(11)
    lin = torch.nn.Linear(k, n, bias=True).to(DEV).to(dtype)
    layer = ojasx_amd.E8LatticeLinear.from_linear(lin, rank=rank, group_size=32, bitrate=bitrate)
    with torch.no_grad():
        layer.lora_B.normal_(std=0.05)
    return layer


class Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.ops = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.ops.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("bitrate", sorted(FMT))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_op_equals_the_extension(bitrate, dtype):
    layer = _layer(bitrate, dtype)
    n, k, r = 96, 320, 8
    a, b = layer.lora_A.detach(), layer.lora_B.detach()
    base = torch.randn(3, 7, k, device=DEV).to(dtype)
    gy = torch.randn(3, 7, n, device=DEV).to(dtype)
    for x in (base, base.transpose(0, 1).contiguous().transpose(0, 1)):
        for need in itertools.product((False, True), repeat=3):
            args = (x, gy, layer.packed_weight, layer.block_scales, a, b, 2.0, FMT[bitrate], n, k,
                    layer.group_size, *need)
            print(f"lora bwd op bitrate={bitrate} {dtype} need={need}", flush=True)
            with torch.no_grad():
                got, ref = N.eager().linear_lora_bwd(*args), ops.linear_lora_bwd(*args)
            shapes = [(21 if need[0] else 0, k), (k, r) if need[1] else (0, r),
                      (r, n) if need[2] else (r, 0)]
            for g, o, want, shape in zip(got, ref, need, shapes):
                assert o.shape == shape
                assert (g is None) != want
                assert not want or torch.equal(g.reshape(o.shape), o)


@pytest.mark.parametrize("bitrate", sorted(FMT))
def test_backward_under_a_dispatch_mode_runs_the_op(bitrate):
    layer = _layer(bitrate)
    x = torch.randn(9, 320, device=DEV).bfloat16().requires_grad_(True)
    gy = torch.randn(9, 96, device=DEV).bfloat16()
    wrt = [x, layer.lora_A, layer.lora_B, layer.bias]
    ref = torch.autograd.grad(layer(x), wrt, gy)
    with Seen() as seen:
        got = torch.autograd.grad(layer(x), wrt, gy)
    assert any("ojasx_e8t.linear_lora." in o for o in seen.ops)
    assert any("ojasx_e8t.linear_lora_bwd" in o for o in seen.ops)
    for g, r in zip(got, ref):
        assert torch.equal(g, r)


@pytest.mark.parametrize("frozen", [(), ("lora_A",), ("bias", "lora_B")])
def test_compiled_layer_with_an_adapter(frozen):
    """One graph, forward and backward, with the eager layer's bits."""
    layer = _layer(1.5)
    for name in frozen:
        getattr(layer, name).requires_grad_(False)
    torch._dynamo.reset()
    compiled = torch.compile(layer, backend="aot_eager", fullgraph=True)
    for shape in ((9, 320), (2, 5, 320)):
        x = torch.randn(*shape, device=DEV).bfloat16().requires_grad_(True)
        wrt = [x] + [p for p in layer.parameters() if p.requires_grad]
        y, ref = compiled(x), layer(x)
        gy = torch.randn_like(ref)
        assert torch.equal(y, ref)
        for g, r in zip(torch.autograd.grad(y, wrt, gy), torch.autograd.grad(ref, wrt, gy)):
            assert torch.equal(g, r)
