"""Adapter gradients at the ends of their size range: rows whose activations pass 2^31 bytes
per wave, a caller without a workspace, and layers too wide for the fused kernels.

Bound per output: (n + 2) 2^-24 times the sum of the term magnitudes for the fp32 sums over n
terms, plus one rounding of the result to its dtype.
"""

import ctypes

import pytest
import torch

from ojasx_amd import _native as N
from ojasx_amd import ops

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
bf16, f16 = torch.bfloat16, torch.float16
ROUND = {bf16: 2.0 ** -8, f16: 2.0 ** -11}


def _operands(M, N_out, K, r, dtype):
    g = torch.Generator(device=DEV).manual_seed(M + N_out + K)

    def rand(rows, cols, scale):
        return (torch.randn(rows, cols, generator=g, device=DEV, dtype=dtype)).mul_(scale)

    return (rand(M, K, 1.0), rand(M, N_out, 0.1), rand(K, r, 0.05), rand(r, N_out, 0.05),
            torch.zeros(N_out * K * 3 // 16, dtype=torch.uint8, device=DEV),
            torch.zeros(N_out * K // 16, dtype=f16, device=DEV))


def _check(out, ref, mag, terms, what):
    err = (out.double() - ref).abs()
    bound = (terms + 2) * 2.0 ** -24 * mag + ROUND[out.dtype] * ref.abs() + 2.0 ** -25
    assert (err <= bound).all(), f"{what}: error {(err / bound).max().item():.2f} of the bound"


def _check_factors(ga, gb, x, gy, a, b, s):
    """Against float64, a few rows at a time."""
    M, K = x.shape
    N_out, r = gy.shape[1], a.shape[1]
    ref = [torch.zeros(2, K, r, dtype=torch.float64, device=DEV),
           torch.zeros(2, r, N_out, dtype=torch.float64, device=DEV)]
    a, b = a.double(), b.double()
    for m in range(0, M, 2048):
        xd, yd = x[m:m + 2048].double(), gy[m:m + 2048].double()
        u, v = s * xd @ a, s * yd @ b.t().contiguous()
        ref[0][0] += xd.t().contiguous() @ v
        ref[1][0] += u.t().contiguous() @ yd
        xd, yd = xd.abs_(), yd.abs_()
        u, v = s * xd @ a.abs(), s * yd @ b.abs().t().contiguous()
        ref[0][1] += xd.t().contiguous() @ v
        ref[1][1] += u.t().contiguous() @ yd
    _check(ga, ref[0][0], ref[0][1], N_out + M, "lora_a")
    _check(gb, ref[1][0], ref[1][1], K + M, "lora_b")


# one wave's rows hold just under and over 2^31 bytes as fp32 (8 waves, no row splits), the
# second with a ragged last group of rows
@pytest.mark.parametrize("M,N_out,K", [(33440, 128256, 16), (65475, 65536, 32)])
def test_many_rows(M, N_out, K):
    x, gy, a, b, pk, sc = _operands(M, N_out, K, 8, bf16)
    print(f"rows M={M} N={N_out} K={K}", flush=True)
    _, ga, gb = ops.linear_lora_bwd(x, gy, pk, sc, a, b, 2.0, ops.FMT_TERNARY, N_out, K, 16,
                                    False, True, True)
    _check_factors(ga, gb, x, gy, a, b, 2.0)


@pytest.mark.parametrize("M,N_out,K,r,dtype", [
    (80007, 16384, 64, 20, bf16),
    (9001, 2500, 80, 33, f16),  # by single values
])
def test_without_workspace(M, N_out, K, r, dtype):
    x, gy, a, b, pk, sc = _operands(M, N_out, K, r, dtype)
    ga, gb = torch.empty_like(a), torch.empty_like(b)
    uv = torch.empty(2, M, r, device=DEV)
    print(f"no workspace M={M} N={N_out} K={K} r={r}", flush=True)
    N.check(N.lib().ojx_gemm_bwd_lora(
        ops.FMT_TERNARY, N.ptr(x), N.ptr(gy), N.ptr(pk), N.ptr(sc), N.ptr(a), N.ptr(b), r, 0.5,
        N.ptr(uv), 0, N.ptr(ga), N.ptr(gb), M, N_out, K, 16, N.DTYPE_CODE[dtype], 0,
        ctypes.c_size_t(0), N.stream_handle(DEV)), "gemm_bwd_lora")
    _check_factors(ga, gb, x, gy, a, b, 0.5)
