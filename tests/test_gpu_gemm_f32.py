"""The fused linear on the fp32 matrix instruction (csrc/e8t_gemm_f32.hip) against the oracle's
decoded weights in float64: fp32 activations, and the 16-bit shapes outside the 64-wide
kernels, at the edges of its tiles (16-row tiles of either operand, 32-k blocks, 16-row
groups of the reduction, columns of 128) and of its row and wave splits.

Bound: fp32 sums of n exact-input products differ from the exact sum by at most
(n + 2) 2^-24 sum |a b| in any order of summation; 16-bit outputs add one rounding (2^-8 of
the result in bf16, 2^-11 in fp16).  The weights are the oracle's decoded ones, so no
weight rounding enters.
"""

import numpy as np
import pytest
import torch

from ojasx_amd import ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
DT_CODE = {torch.float32: O.DT_F32, torch.float16: O.DT_F16, torch.bfloat16: O.DT_BF16}
ROUND = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
FMT = {"ternary": (O.encode, O.decode, ops.e8t_linear, ops.e8t_linear_bwd_dx),
       "2bit": (O.e8b_encode, O.e8b_decode, ops.e8_linear, ops.e8_linear_bwd_dx),
       "1bit": (O.e8r_encode, O.e8r_decode, ops.e8r_linear, ops.e8r_linear_bwd_dx)}
f32, f16, bf16 = torch.float32, torch.float16, torch.bfloat16


def _layer(fmt, N, K, gs, dtype):
    enc, dec, fwd, bwd = FMT[fmt]
    g = torch.Generator().manual_seed(N * 7 + K + gs)
    w = (torch.randn(N, K, generator=g) * 0.02).numpy()
    packed, scales, _ = enc(w, gs)
    dense = np.asarray(dec(packed, scales, N * K, gs, DT_CODE[dtype]))
    if dense.dtype == np.uint16:  # 16-bit weights come back as bits
        dense = (O.bf16_bits_to_f32 if dtype == bf16 else O.f16_bits_to_f32)(dense)
    pk = torch.from_numpy(packed).to(DEV)
    sc = torch.from_numpy(np.asarray(scales).view(np.int16)).view(torch.float16).to(DEV)
    return pk, sc, torch.from_numpy(dense.astype(np.float64)).view(N, K), fwd, bwd


def _check(out, ref, mag, terms, dtype, what):
    err = (out.detach().cpu().double() - ref).abs()
    bound = (terms + 2) * 2.0 ** -24 * mag + ROUND[dtype] * ref.abs() + 1e-30
    if dtype == f16:
        bound += 2.0 ** -25  # below the normal range
    worst = (err / bound).max().item()
    assert worst <= 1.0, f"{what}: error {worst:.2f} of the bound"


SHAPES = [
    ("ternary", 1, 4096, 1024, 32, f32, True),
    ("ternary", 1, 33, 8208, 16, f32, False),       # ragged rows, K tail of half a block
    ("ternary", 16, 8200, 256, 64, f32, True),      # two row tiles per wave, ragged
    ("ternary", 17, 130, 320, 32, f32, False),      # one row past a tile, idle waves
    ("ternary", 33, 100, 544, 32, f32, True),
    ("ternary", 64, 16400, 128, 128, f32, False),   # four row tiles per wave
    ("ternary", 70, 96, 48, 16, f32, True),         # a second block of rows, blocks < waves
    ("ternary", 5, 48, 16, 16, f32, True),          # a single code pair per row
    ("2bit", 1, 100, 1000, 8, f32, True),           # K % 32 == 8
    ("2bit", 9, 257, 456, 8, bf16, True),
    ("2bit", 40, 65, 72, 8, f16, False),
    ("2bit", 3, 40, 64, 64, f32, False),
    ("1bit", 1, 72, 1992, 8, f32, True),
    ("1bit", 18, 129, 416, 32, bf16, False),
    ("1bit", 66, 31, 104, 8, f16, True),
    ("ternary", 6, 1536, 4448, 32, f16, True),
    ("ternary", 300, 200, 96, 32, bf16, False),
    # rows of whole words (one load per eight codes), the last 256-k chunk cut off
    ("ternary", 4, 200, 704, 16, f32, True),
    ("ternary", 20, 8210, 320, 64, f32, False),
    ("ternary", 50, 5000, 576, 32, f32, True),
    ("2bit", 16, 100, 1008, 8, f32, True),
    ("2bit", 70, 530, 544, 16, f32, False),
    ("2bit", 2, 72, 2304, 256, f32, False),
    ("2bit", 3, 50, 1000, 8, bf16, False),
    ("1bit", 2, 40, 288, 16, f32, True),
    ("1bit", 40, 70, 1056, 8, f32, False),
    ("1bit", 1, 100, 4128, 32, f16, True),
]


@pytest.mark.parametrize("fmt,M,N,K,gs,dtype,bias", SHAPES)
def test_forward(fmt, M, N, K, gs, dtype, bias):
    pk, sc, w, fwd, _ = _layer(fmt, N, K, gs, dtype)
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn(M, K, generator=g).to(dtype)
    b = torch.randn(N, generator=g).to(dtype) if bias else None
    print(f"f32 fwd {fmt} M={M} N={N} K={K} gs={gs} {dtype}", flush=True)
    y = fwd(x.to(DEV), pk, sc, None if b is None else b.to(DEV), N, K, gs)
    ref = x.double() @ w.t()
    mag = x.double().abs() @ w.abs().t()
    if bias:
        ref, mag = ref + b.double(), mag + b.double().abs()
    _check(y, ref, mag, K, dtype, "forward")


@pytest.mark.parametrize("fmt,M,N,K,gs,dtype,bias", SHAPES + [
    ("ternary", 16, 14336, 256, 64, f32, False),    # rows split over workgroups and waves
    ("ternary", 1, 14330, 128, 32, f32, False),     # ... N % 4 != 0: scalar loads
    ("1bit", 50, 4100, 200, 8, f32, False),
    ("2bit", 20, 2049, 264, 8, bf16, False),
])
def test_backward_dx(fmt, M, N, K, gs, dtype, bias):
    pk, sc, w, _, bwd = _layer(fmt, N, K, gs, dtype)
    gy = torch.randn(M, N, generator=torch.Generator().manual_seed(M + N)).to(dtype)
    print(f"f32 bwd {fmt} M={M} N={N} K={K} gs={gs} {dtype}", flush=True)
    gx = bwd(gy.to(DEV), pk, sc, N, K, gs)
    _check(gx, gy.double() @ w, gy.double().abs() @ w.abs(), N, dtype, "backward")


@pytest.mark.parametrize("K,N", [(40, 20), (264, 33), (32, 4)])
def test_rows_stay_apart(K, N):
    """An infinite row of activations (gradients) reaches its own outputs only: the tails of
    the other rows' last blocks never read it."""
    pk, sc, w, fwd, bwd = _layer("2bit", N, K, 8, f32)
    for op, width in ((lambda t: fwd(t, pk, sc, None, N, K, 8), K),
                      (lambda t: bwd(t, pk, sc, N, K, 8), N)):
        a = torch.randn(5, width, generator=torch.Generator().manual_seed(K))
        clean = op(a.to(DEV)).cpu()
        a[2] = float("inf")
        out = op(a.to(DEV)).cpu()
        keep = [0, 1, 3, 4]
        assert torch.equal(out[keep], clean[keep])
        assert not torch.isfinite(out[2]).any()
