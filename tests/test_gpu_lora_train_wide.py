"""Training an adapter on a layer of 2^23 outputs, past the fused gradients' widths: the torch
products, as where the gradients are themselves differentiated."""

import pytest
import torch

from ojasx_amd import _native as N
from ojasx_amd import ops

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def test_wide_layer():
    M, N_out, K, r = 3, 1 << 23, 16, 2
    g = torch.Generator(device=DEV).manual_seed(5)

    def rand(*shape):
        return torch.randn(*shape, generator=g, device=DEV).bfloat16()

    pk = torch.zeros(N_out * K * 3 // 16, dtype=torch.uint8, device=DEV)
    sc = torch.ones(N_out, dtype=torch.float16, device=DEV)
    x, gy = rand(M, K), rand(M, N_out)
    a, b = rand(K, r).requires_grad_(True), rand(r, N_out).requires_grad_(True)

    def grads(**kw):
        y = ops.linear_lora(x, pk, sc, None, a, b, 2.0, ops.FMT_TERNARY, N_out, K, 16)
        return torch.autograd.grad(y, (a, b), gy, **kw)

    for got, ref in zip(grads(), grads(create_graph=True)):
        assert torch.equal(got, ref)
    with pytest.raises(RuntimeError, match="adapter gradients need"):
        ops.linear_lora_bwd(x, gy, pk, sc, a.detach(), b.detach(), 2.0, ops.FMT_TERNARY, N_out, K,
                            16, False, True, True)
    assert b"adapter gradients need" in N.lib().ojx_e8t_last_error()
