"""The eager extension (csrc/e8t_torch.cpp) against the registered ops: the same bits for
every call it takes, and None (the caller's route to the op) for every call it must not.

Nothing here depends on a tolerance: both routes enqueue the same kernels on the same data.
"""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import ojasx_amd
from ojasx_amd import _native as N
from ojasx_amd import ops

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
LINEAR = {1.5: ops.e8t_linear, 2.0: ops.e8_linear, 1.0: ops.e8r_linear}
BWD = {1.5: ops.e8t_linear_bwd_dx, 2.0: ops.e8_linear_bwd_dx, 1.0: ops.e8r_linear_bwd_dx}
FMT = {1.5: ops.FMT_TERNARY, 2.0: ops.FMT_E8, 1.0: ops.FMT_ROOT}


def _layer(bitrate, dtype=torch.bfloat16, rank=0, bias=True, n=96, k=320):
    torch.manual_seed(3)
    lin = torch.nn.Linear(k, n, bias=bias).to(DEV).to(dtype)
    layer = ojasx_amd.E8LatticeLinear.from_linear(lin, rank=rank, group_size=32, bitrate=bitrate)
    if rank:
        with torch.no_grad():
            layer.lora_B.normal_(std=0.05)
    return layer


def _call(layer, x):
    return N.eager().linear(x, layer.packed_weight, layer.block_scales, layer.bias,
                            layer.out_features, layer.in_features, layer.group_size,
                            FMT[layer.bitrate])


def _op(layer, x):
    return LINEAR[layer.bitrate](x, layer.packed_weight, layer.block_scales, layer.bias,
                                 layer.out_features, layer.in_features, layer.group_size)


@pytest.mark.parametrize("bitrate", [1.5, 2.0, 1.0])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_forward_forms(bitrate, dtype):
    layer = _layer(bitrate, dtype)
    base = torch.randn(7, 320, device=DEV).to(dtype)
    forms = [base, base[3], base.view(7, 1, 320), base.t().contiguous().t(), base[::2],
             base[:0], base.expand(2, 7, 320), torch.randn(7, 321, device=DEV).to(dtype)[:, 1:],
             torch.randn(40, 320, device=DEV).to(dtype)]
    with torch.no_grad():
        for x in forms:
            y, ref = _call(layer, x), _op(layer, x)
            assert y is not None and y.shape == ref.shape and torch.equal(y, ref)
            assert torch.equal(layer(x), ref) and not y.requires_grad
            gy = torch.randn_like(ref)
            gx = N.eager().linear_bwd(gy, layer.packed_weight, layer.block_scales, 96, 320,
                                      layer.group_size, FMT[bitrate])
            assert torch.equal(gx, BWD[bitrate](gy, layer.packed_weight, layer.block_scales, 96,
                                                320, layer.group_size))


@pytest.mark.parametrize("bitrate", [1.5, 2.0, 1.0])
@pytest.mark.parametrize("rank", [0, 8])
def test_gradients_equal_the_ops(bitrate, rank):
    layer = _layer(bitrate, rank=rank)
    x = torch.randn(2, 9, 320, device=DEV).bfloat16().requires_grad_(True)
    gy = torch.randn(2, 9, 96, device=DEV).bfloat16()
    wrt = [x] + [p for p in (layer.bias, layer.lora_A, layer.lora_B) if p is not None]
    y = layer(x)
    got = torch.autograd.grad(y, wrt, gy)
    if rank:
        ref = ops.linear_lora(x, layer.packed_weight, layer.block_scales, layer.bias, layer.lora_A,
                              layer.lora_B, float(layer.scaling), FMT[bitrate], 96, 320,
                              layer.group_size)
    else:
        ref = _op(layer, x)
    assert torch.equal(y, ref)
    for a, b in zip(got, torch.autograd.grad(ref, wrt, gy)):
        assert torch.equal(a, b)
    # under hooks that replace what is saved
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t.clone(),
                                                  lambda t: t):
        y = layer(x)
    assert seen
    for a, b in zip(got, torch.autograd.grad(y, wrt, gy)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("fmt,pack,enc,dec", [
    (ops.FMT_TERNARY, ojasx_amd.TernaryE8LatticePacker, ops.encode, ops.decode),
    (ops.FMT_E8, ojasx_amd.E8LatticePacker, ops.encode2, ops.decode2),
    (ops.FMT_ROOT, ojasx_amd.RootE8LatticePacker, ops.encode1, ops.decode1)])
def test_codec(fmt, pack, enc, dec):
    for w in (torch.randn(33, 40, device=DEV), torch.randn(64, 50, device=DEV).half().t(),
              torch.randn(5, 7, device=DEV).bfloat16(), torch.randn(3, 16, device=DEV).double()):
        codes, scales, shape = pack.pack(w, group_size=16)
        ref = enc(w, 16)
        assert torch.equal(codes, ref[0]) and torch.equal(scales, ref[1])
        for dtype in (torch.float32, torch.float16, torch.bfloat16):
            out = pack.unpack(codes, scales, shape, dtype=dtype)
            assert torch.equal(out.view(-1), dec(codes, scales, w.numel(), 16, dtype))


def test_calls_left_to_the_op():
    layer = _layer(1.5)
    x = torch.randn(4, 320, device=DEV).bfloat16()
    with torch.no_grad():
        assert _call(layer, x) is not None
        assert _call(layer, x.cpu()) is None
        assert _call(layer, x.double()) is None
        assert _call(layer, x[:, :319]) is None
        assert _call(layer, torch._neg_view(x)) is None
        assert _call(layer.float(), x) is None          # bias and scales cast away
        layer = _layer(1.5)

        class Seen(TorchDispatchMode):
            def __init__(self):
                super().__init__()
                self.ops = []

            def __torch_dispatch__(self, func, types, args=(), kwargs=None):
                self.ops.append(str(func))
                return func(*args, **(kwargs or {}))

        with Seen() as seen:
            assert _call(layer, x) is None
            layer(x)
        assert any("ojasx_e8t.e8t_linear" in o for o in seen.ops)

        with torch._subclasses.FakeTensorMode() as mode:
            assert _call(layer, mode.from_tensor(x)) is None
        with torch.autograd.forward_ad.dual_level():
            assert _call(layer, torch.autograd.forward_ad.make_dual(x, x)) is None
        torch.func.vmap(lambda t: (_call(layer, t) is None or pytest.fail("under vmap"), t)[1])(x)
        with torch.inference_mode():
            assert torch.equal(_call(layer, x), _op(layer, x))
    assert _call(layer, x.clone().requires_grad_(True)) is None  # gradients to record
    traced = torch.jit.trace(layer, (x,), check_trace=False)
    assert "e8t_linear" in str(traced.inlined_graph) or "PythonOp" in str(traced.inlined_graph) \
        or "_FusedE8GEMMFunction" in str(traced.inlined_graph)
    other = torch.randn(4, 320, device=DEV).bfloat16()
    assert torch.equal(traced(other), layer(other))


def test_captured_and_streams():
    layer = _layer(1.5, rank=8).requires_grad_(False)
    x = torch.randn(300, 320, device=DEV).bfloat16()
    ref = layer(x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = layer(x)
    torch.cuda.synchronize()
    assert torch.equal(y, ref)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        y = layer(x)
    for _ in range(3):
        x.copy_(torch.randn(300, 320, device=DEV).bfloat16())
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, layer(x))
