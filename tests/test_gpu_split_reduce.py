"""The reduction of a K split's fp32 partial sums: every split count from 2 to 16 (its loads go
out five splits at a time), with and without bias, rows of odd widths, an output of odd alignment.

The operands are small integers and powers of two, so every product and every sum is exact in
fp32 and the result is exact in the activation dtype: equality, no tolerance.
"""

import pytest
import torch

from ojasx_amd import _native as N
from ojasx_amd import ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


@pytest.mark.parametrize("splits", range(1, 17))
@pytest.mark.parametrize("n", [64, 131])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_split_count(splits, n, dtype):
    k, m, gs = 256 * splits, 33, 32
    g = torch.Generator().manual_seed(splits)
    packed, scales, _ = O.encode((torch.randn(n, k, generator=g) * 0.02).numpy(), gs)
    scales = torch.full((n * k // gs,), 0.5, dtype=torch.float16)
    w = torch.from_numpy(O.decode(packed, scales.view(torch.int16).numpy().view("uint16"), n * k,
                                  gs, O.DT_F32).copy()).view(n, k).double()
    x = torch.zeros(m, k)
    at = torch.randint(0, k, (m, 40), generator=g)  # up to 40 products of +-0.5: exact in 16 bits
    x.scatter_(1, at, torch.randint(-1, 2, (m, 40), generator=g).float())
    bias = torch.randint(-8, 9, (n,), generator=g).double()
    pk, sc = torch.from_numpy(packed).to(DEV), scales.to(DEV)
    xd = x.to(DEV, dtype)
    print(f"splits={splits} n={n} {dtype}", flush=True)
    ref = x.double() @ w.t()
    assert torch.equal(ops.e8t_linear(xd, pk, sc, None, n, k, gs).cpu().double(), ref)
    bd = bias.to(DEV, dtype)
    y = ops.e8t_linear(xd, pk, sc, bd, n, k, gs)
    assert torch.equal(y.cpu().double(), ref + bias)
    # the C ABI with an output two bytes off
    store = torch.zeros(m * n + 1, dtype=dtype, device=DEV)
    ws = torch.empty(16 * (m * n + 64) * 4, dtype=torch.uint8, device=DEV)
    with torch.cuda.device(DEV):
        N.check(N.lib().ojx_e8t_gemm_fwd(
            N.ptr(xd), N.ptr(pk), N.ptr(sc), N.ptr(bd), store.data_ptr() + 2, m, n, k, gs,
            N.DTYPE_CODE[dtype], N.ptr(ws), ws.numel(), N.stream_handle(DEV)), "gemm_fwd")
    assert torch.equal(store[1:].view(m, n).cpu().double(), ref + bias)
