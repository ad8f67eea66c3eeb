"""Adapters of training-sized calls, where the adapter term is added on the matrix unit:
forward outputs and gradients of linear_lora against float64 on the oracle's decoded weights.

Bound per output: (n + 2) 2^-24 times the sum of the term magnitudes for every fp32 sum over n
terms, plus one rounding of the result to its dtype (2^-8 in bf16, 2^-11 in fp16).  The
16-bit kernels contract decoded 16-bit weights whose products are exact in fp32.
"""

import numpy as np
import pytest
import torch

from ojasx_amd import ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
f32, f16, bf16 = torch.float32, torch.float16, torch.bfloat16
DT_CODE = {f32: O.DT_F32, f16: O.DT_F16, bf16: O.DT_BF16}
ROUND = {f32: 2.0 ** -24, f16: 2.0 ** -11, bf16: 2.0 ** -8}
CODEC = {ops.FMT_TERNARY: (O.encode, O.decode), ops.FMT_E8: (O.e8b_encode, O.e8b_decode),
         ops.FMT_ROOT: (O.e8r_encode, O.e8r_decode)}


def _case(fmt, M, N, K, gs, r, dtype):
    enc, dec = CODEC[fmt]
    g = torch.Generator().manual_seed(M + 3 * N + K + r)
    packed, scales, _ = enc((torch.randn(N, K, generator=g) * 0.02).numpy(), gs)
    dense = np.asarray(dec(packed, scales, N * K, gs, DT_CODE[dtype]))
    if dense.dtype == np.uint16:
        dense = (O.bf16_bits_to_f32 if dtype == bf16 else O.f16_bits_to_f32)(dense)
    t = dict(x=torch.randn(M, K, generator=g).to(dtype),
             a=(torch.randn(K, r, generator=g) * 0.05).to(dtype),
             b=(torch.randn(r, N, generator=g) * 0.05).to(dtype),
             gy=(torch.randn(M, N, generator=g) * 0.1).to(dtype),
             bias=torch.randn(N, generator=g).to(dtype))
    pk = torch.from_numpy(packed).to(DEV)
    sc = torch.from_numpy(np.asarray(scales).view(np.int16)).view(f16).to(DEV)
    return t, pk, sc, torch.from_numpy(dense.astype(np.float64)).view(N, K)


def _check(out, ref, mag, terms, dtype, what):
    err = (out.detach().cpu().double() - ref).abs()
    bound = (terms + 2) * 2.0 ** -24 * mag + ROUND[dtype] * ref.abs() + 1e-30
    if dtype == f16:
        bound += 2.0 ** -25
    worst = (err / bound).max().item()
    assert worst <= 1.0, f"{what}: error {worst:.2f} of the bound"


SHAPES = [
    (ops.FMT_TERNARY, 600, 512, 2048, 32, 8, bf16),     # K split over small tiles
    (ops.FMT_TERNARY, 2048, 4096, 1024, 64, 8, bf16),   # large tiles, split
    (ops.FMT_TERNARY, 1030, 12416, 256, 32, 16, bf16),  # large tiles, unsplit
    (ops.FMT_E8, 33, 130, 320, 8, 3, f16),              # a rank under four
    (ops.FMT_ROOT, 260, 1000, 512, 32, 21, bf16),       # ranks over several fours, ragged
    (ops.FMT_E8, 130, 448, 1024, 16, 64, bf16),
    (ops.FMT_TERNARY, 17, 200, 96, 32, 5, bf16),        # the fp32 kernel's 16-bit shapes
    (ops.FMT_TERNARY, 16, 1504, 1024, 64, 8, f32),
    (ops.FMT_TERNARY, 70, 72, 48, 16, 30, f32),
    (ops.FMT_ROOT, 1, 33, 40, 8, 1, f32),
]


@pytest.mark.parametrize("fmt,M,N,K,gs,r,dtype", SHAPES)
def test_forward(fmt, M, N, K, gs, r, dtype):
    t, pk, sc, w = _case(fmt, M, N, K, gs, r, dtype)
    s = 2.0
    print(f"lora fwd fmt={fmt} M={M} N={N} K={K} gs={gs} r={r} {dtype}", flush=True)
    y = ops.linear_lora(t["x"].to(DEV), pk, sc, t["bias"].to(DEV), t["a"].to(DEV),
                        t["b"].to(DEV), s, fmt, N, K, gs)
    x, a, b, bias = (t[k].double() for k in ("x", "a", "b", "bias"))
    ref = x @ w.t() + s * (x @ a) @ b + bias
    mag = x.abs() @ w.abs().t() + s * (x.abs() @ a.abs()) @ b.abs() + bias.abs()
    _check(y, ref, mag, K + r, dtype, "forward")


def _grads(t, pk, sc, s, fmt, N, K, gs, need=("x", "a", "b"), **kw):
    d = {k: v.to(DEV).requires_grad_(k in need) for k, v in t.items() if k not in ("gy", "bias")}
    y = ops.linear_lora(d["x"], pk, sc, None, d["a"], d["b"], s, fmt, N, K, gs)
    return torch.autograd.grad(y, [d[k] for k in need], t["gy"].to(DEV), **kw)


@pytest.mark.parametrize("fmt,M,N,K,gs,r,dtype", SHAPES + [
    (ops.FMT_TERNARY, 4100, 320, 256, 32, 12, bf16),   # row splits with fp32 partial sums
    (ops.FMT_E8, 300, 100, 24, 24, 9, f16),            # the SIMT kernel (group size 24)
])
def test_gradients(fmt, M, N, K, gs, r, dtype):
    t, pk, sc, w = _case(fmt, M, N, K, gs, r, dtype)
    s = 0.5
    print(f"lora bwd fmt={fmt} M={M} N={N} K={K} gs={gs} r={r} {dtype}", flush=True)
    gx, ga, gb = _grads(t, pk, sc, s, fmt, N, K, gs)
    x, a, b, gy = (t[k].double() for k in ("x", "a", "b", "gy"))
    v, u = s * gy @ b.t(), s * x @ a
    mv, mu = s * gy.abs() @ b.abs().t(), s * x.abs() @ a.abs()
    _check(gx, gy @ w + v @ a.t(), gy.abs() @ w.abs() + mv @ a.abs().t(), 2 * N + r, dtype, "x")
    _check(ga, x.t() @ v, x.abs().t() @ mv, N + M, dtype, "lora_a")
    _check(gb, u.t() @ gy, mu.t() @ gy.abs(), K + M, dtype, "lora_b")


@pytest.mark.parametrize("need", [("x",), ("a",), ("b",), ("a", "b"), ("x", "b")])
def test_gradients_of_some(need):
    """Frozen operands: the others' gradients are the ones of the full call, bit for bit."""
    fmt, M, N, K, gs, r = ops.FMT_TERNARY, 1500, 256, 512, 32, 8
    t, pk, sc, _ = _case(fmt, M, N, K, gs, r, bf16)
    full = dict(zip(("x", "a", "b"), _grads(t, pk, sc, 2.0, fmt, N, K, gs)))
    some = dict(zip(need, _grads(t, pk, sc, 2.0, fmt, N, K, gs, need=need)))
    for k, v in some.items():
        if k == "x" or len(need) > 1:
            assert torch.equal(v, full[k])
        else:  # one factor alone may split its rows differently: fp32 sums in another order
            assert (v.float() - full[k].float()).abs().max() <= 2 ** -7 * full[k].float().abs().max()


def test_gradients_other_callers():
    """A transposed view of x, a batch of sequences, no rows, and gradients that are themselves
    to be differentiated (these keep the torch products)."""
    fmt, N, K, gs, r = ops.FMT_TERNARY, 96, 256, 32, 8
    t, pk, sc, _ = _case(fmt, 24, N, K, gs, r, bf16)
    ref = _grads(t, pk, sc, 2.0, fmt, N, K, gs)
    view = dict(t, x=t["x"].t().contiguous().t())
    assert all(torch.equal(p, q) for p, q in zip(ref, _grads(view, pk, sc, 2.0, fmt, N, K, gs)))
    batch = dict(t, x=t["x"].view(4, 6, K), gy=t["gy"].view(4, 6, N))
    out = _grads(batch, pk, sc, 2.0, fmt, N, K, gs)
    assert out[0].shape == (4, 6, K)
    assert all(torch.equal(p.reshape(q.shape), q) for p, q in zip(out, ref))
    none = dict(t, x=t["x"][:0], gy=t["gy"][:0])
    out = _grads(none, pk, sc, 2.0, fmt, N, K, gs)
    assert out[0].shape == (0, K) and not out[1].any() and not out[2].any()
    out = _grads(t, pk, sc, 2.0, fmt, N, K, gs, create_graph=True)
    assert out[1].requires_grad and out[2].requires_grad
    for p, q in zip(out, ref):  # three bf16 roundings more than the fused gradients
        assert (p.float() - q.float()).abs().max() <= 2 ** -6 * q.float().abs().max()
