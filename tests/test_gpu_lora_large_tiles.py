"""grad_x of the low-bit formats on large tiles (at least 192 of 256 x 256), where layers with and
without an adapter run kernels of their own, unsplit and with a K split: against float64 on
the oracle's decoded weights, to the bound of the other adapter gradients.
"""

import pytest
import torch

from ojasx_amd import ops
from test_gpu_lora_train import DEV, _case, _check, bf16, f16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,gs", [(ops.FMT_E8, 8), (ops.FMT_E8, 64), (ops.FMT_ROOT, 16)])
@pytest.mark.parametrize("M,N,K,dtype", [
    (1030, 64, 12416, bf16), (1030, 192, 12416, f16),  # 5 x 49 tiles
    (1000, 2048, 6144, bf16),                          # 4 x 24 tiles, split in two over N
])
@pytest.mark.parametrize("rank", [0, 5, 16])
def test_grad_x(fmt, gs, M, N, K, dtype, rank):
    t, pk, sc, w = _case(fmt, M, N, K, gs, max(rank, 1), dtype)
    print(f"large tiles fmt={fmt} M={M} N={N} K={K} gs={gs} r={rank} {dtype}", flush=True)
    gy, a, b = (t[k].to(DEV) for k in ("gy", "a", "b"))
    w, gyd = w.to(DEV), gy.double()
    ref, mag = gyd @ w, gyd.abs() @ w.abs()
    if rank:
        gx = ops.linear_lora_bwd(t["x"].to(DEV), gy, pk, sc, a, b, 0.5, fmt, N, K, gs, True, False,
                                 False)[0]
        ad, bt = a.double().t().contiguous(), b.double().t().contiguous()
        ref += 0.5 * (gyd @ bt) @ ad
        mag += 0.5 * (gyd.abs() @ bt.abs()) @ ad.abs()
    else:
        bwd = ops.e8_linear_bwd_dx if fmt == ops.FMT_E8 else ops.e8r_linear_bwd_dx
        gx = bwd(gy, pk, sc, N, K, gs)
    _check(gx, ref.cpu(), mag.cpu(), 2 * N + rank, dtype, "x")
