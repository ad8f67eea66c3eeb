"""The decoders at the edges of their 16-byte runs, pieces and blocks, and at group sizes that
are no power of two: bits equal to the oracle's (exact; the packers' decode rule)."""

import numpy as np
import pytest
import torch

from ojasx_amd import ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
DT = {torch.float32: O.DT_F32, torch.float16: O.DT_F16, torch.bfloat16: O.DT_BF16}
FMT = {"ternary": (O.encode, O.decode, ops.decode), "2bit": (O.e8b_encode, O.e8b_decode, ops.decode2),
       "1bit": (O.e8r_encode, O.e8r_decode, ops.decode1)}


@pytest.mark.parametrize("fmt", FMT)
@pytest.mark.parametrize("dtype", list(DT))
@pytest.mark.parametrize("numel,gs", [(1, 16), (8, 16), (13, 48), (4096, 32), (4097, 16), (8191, 48),
                                      (8192, 64), (3 * 8192 + 5, 32), (40001, 16),
                                      (2200003, 16), (4194304, 48)])
def test_decode_bits(fmt, dtype, numel, gs):
    enc, dec, op = FMT[fmt]
    w = torch.randn(1, numel, generator=torch.Generator().manual_seed(numel + gs))
    packed, scales, _ = enc((w * 0.02).numpy(), gs)
    scales = np.array(scales)
    scales[::7] = 0  # zero scales keep the coordinates' signs
    print(f"decode {fmt} {dtype} numel={numel} gs={gs}", flush=True)
    ref = np.asarray(dec(packed, scales, numel, gs, DT[dtype])).reshape(-1)
    sc = torch.from_numpy(scales.view(np.int16)).view(torch.float16).to(DEV)
    out = op(torch.from_numpy(packed).to(DEV), sc, numel, gs, dtype).cpu()
    bits = out.view(torch.int32 if dtype == torch.float32 else torch.int16).numpy()
    want = ref.view(np.int32) if ref.dtype == np.float32 else ref.view(np.int16)
    assert bits.dtype == want.dtype and np.array_equal(bits, want)
