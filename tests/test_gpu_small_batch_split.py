"""16-bit linears of 17 to 128 rows (and the backward of fewer), whose K splits go down to
four 64-k steps: every element against float64 on the oracle's decoded weights.

Bound: fp32 sums of n products in any order, (n + 2) 2^-24 sum |a b|, and one rounding to bf16
(2^-8 of the result).
"""

import numpy as np
import pytest
import torch

from ojasx_amd import ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _layer(N, K, gs):
    g = torch.Generator().manual_seed(N + K)
    packed, scales, _ = O.e8b_encode((torch.randn(N, K, generator=g) * 0.02).numpy(), gs)
    dense = O.bf16_bits_to_f32(np.asarray(O.e8b_decode(packed, scales, N * K, gs, O.DT_BF16)))
    sc = torch.from_numpy(np.asarray(scales).view(np.int16)).view(torch.float16).to(DEV)
    return (torch.from_numpy(packed).to(DEV), sc,
            torch.from_numpy(dense.astype(np.float64)).view(N, K))


def _check(out, ref, mag, terms):
    err = (out.cpu().double() - ref).abs()
    assert (err <= (terms + 2) * 2.0 ** -24 * mag + 2.0 ** -8 * ref.abs() + 1e-30).all()


@pytest.mark.parametrize("M", [1, 17, 127, 128, 129])
@pytest.mark.parametrize("N,K", [(256, 192), (512, 256), (320, 576), (130, 1088), (4160, 832),
                                 (16512, 512)])
def test_split_rows(M, N, K):
    pk, sc, w = _layer(N, K, 8)
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16()
    print(f"split M={M} N={N} K={K}", flush=True)
    _check(ops.e8_linear(x.to(DEV), pk, sc, None, N, K, 8), x.double() @ w.t(),
           x.double().abs() @ w.abs().t(), K)
    gy = torch.randn(M, N, generator=g).bfloat16()
    _check(ops.e8_linear_bwd_dx(gy.to(DEV), pk, sc, N, K, 8), gy.double() @ w,
           gy.double().abs() @ w.abs(), N)
