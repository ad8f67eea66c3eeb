"""u = scaling * (x @ A) and the adapter gradients at the ranks, dtypes and row counts that pick
each form of the down-projection: a workgroup per row (fewer than 512 rows, factors readable
in 16-byte pieces), tiles of 16 rows with 1, 2 or 4 column tiles of ranks, staged through LDS,
read along K or read value by value, and the general kernel.

Bound per fp32 output: (K + 3) 2^-24 times the sum of the term magnitudes (products of 16-bit
values are exact in fp32; fp32 products round once more), on float64 references.
"""

import pytest
import torch

from ojasx_amd import _native as N
from ojasx_amd import ops

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
f32, f16, bf16 = torch.float32, torch.float16, torch.bfloat16
ROUND = {f32: 2.0 ** -24, f16: 2.0 ** -11, bf16: 2.0 ** -8}
RANKS = [1, 8, 16, 17, 32, 33, 40, 48, 63, 64]


def _rand(g, rows, cols, scale, dtype):
    return (torch.randn(rows, cols, generator=g) * scale).to(dtype)


def _down(x, a, s):
    M, K = x.shape
    r = a.shape[1]
    u = torch.full((M, r), float("nan"), device=DEV)
    N.check(N.lib().ojx_lora_down(N.ptr(x), N.ptr(a), M, K, r, s, N.DTYPE_CODE[x.dtype], N.ptr(u),
                                  N.stream_handle(DEV)), "lora_down")
    return u


@pytest.mark.parametrize("dtype", [bf16, f16, f32])
@pytest.mark.parametrize("rank", RANKS)
@pytest.mark.parametrize("M,K", [
    (512, 1024), (530, 136),   # staged tiles, the second with a batch that ends inside K
    (513, 100), (40, 100),     # value by value
    (16, 520), (15, 520),      # ranks that no 16-byte piece fits: tiles from 16 rows, general below
    (511, 520), (3, 64),       # a workgroup per row where the rank allows
])
def test_down_projection(M, K, rank, dtype):
    g = torch.Generator().manual_seed(M + K + rank)
    x, a = _rand(g, M, K, 1.0, dtype), _rand(g, K, rank, 0.1, dtype)
    print(f"lora down M={M} K={K} r={rank} {dtype}", flush=True)
    u = _down(x.to(DEV), a.to(DEV), 0.5).cpu().double()
    ref, mag = 0.5 * (x.double() @ a.double()), 0.5 * (x.double().abs() @ a.double().abs())
    assert ((u - ref).abs() <= (K + 3) * 2.0 ** -24 * mag + 1e-30).all()


def _check(out, ref, mag, terms, what):
    err = (out.cpu().double() - ref).abs()
    bound = (terms + 3) * 2.0 ** -24 * mag + ROUND[out.dtype] * ref.abs() + 2.0 ** -25
    assert (err <= bound).all(), f"{what}: error {(err / bound).max().item():.2f} of the bound"


@pytest.mark.parametrize("dtype", [bf16, f16, f32])
@pytest.mark.parametrize("rank", [8, 20, 33, 64])
@pytest.mark.parametrize("M,N_out,K", [(700, 136, 144), (520, 90, 80), (24, 136, 144)])
def test_factor_gradients(M, N_out, K, rank, dtype):
    g = torch.Generator().manual_seed(M + K + rank)
    x, gy = _rand(g, M, K, 1.0, dtype), _rand(g, M, N_out, 0.1, dtype)
    a, b = _rand(g, K, rank, 0.1, dtype), _rand(g, rank, N_out, 0.1, dtype)
    pk = torch.zeros(N_out * K * 3 // 16, dtype=torch.uint8, device=DEV)
    sc = torch.zeros(N_out * K // 16, dtype=f16, device=DEV)
    print(f"factor grads M={M} N={N_out} K={K} r={rank} {dtype}", flush=True)
    gx, ga, gb = ops.linear_lora_bwd(x.to(DEV), gy.to(DEV), pk, sc, a.to(DEV), b.to(DEV), 2.0,
                                     ops.FMT_TERNARY, N_out, K, 16, True, True, True)
    x, gy, a, b = (t.double() for t in (x, gy, a, b))
    u, v = 2 * x @ a, 2 * gy @ b.t()
    mu, mv = 2 * x.abs() @ a.abs(), 2 * gy.abs() @ b.abs().t()
    # (zero scales: W is 0, so grad_x is the adapter's term alone)
    _check(gx, v @ a.t(), mv @ a.abs().t(), N_out + rank, "x")
    _check(ga, x.t() @ v, x.abs().t() @ mv, N_out + M, "lora_a")
    _check(gb, u.t() @ gy, mu.t() @ gy.abs(), K + M, "lora_b")
