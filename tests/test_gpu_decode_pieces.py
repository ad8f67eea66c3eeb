"""Decodes with two and four 16-byte pieces per lane (results from 32 and 256 MB) against decodes of
a million weights at a time, which take one piece and are checked against the oracle
elsewhere: the same bits.  And the time of a result too small for several pieces."""

import pytest
import torch

from ojasx_amd import ops

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
CODE_BYTES = {ops.decode: 3 / 16, ops.decode2: 1 / 4, ops.decode1: 1 / 8}
DTYPES = [torch.float32, torch.float16, torch.bfloat16]


def _packed(op, numel, gs):
    padded = -(-numel // gs) * gs
    g = torch.Generator(device=DEV).manual_seed(numel)
    top = 52 if op is ops.decode else 256  # (ternary codes stay below 3281)
    packed = torch.randint(0, top, (int(padded * CODE_BYTES[op]),), generator=g, device=DEV,
                           dtype=torch.uint8)
    scales = torch.randn(padded // gs, generator=g, device=DEV).half()
    scales[::5] = 0
    return packed, scales


@pytest.mark.parametrize("op", list(CODE_BYTES))
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("blocks,extra,gs", [(8191, 7, 32), (8192, 9, 32), (12001, 1, 48),
                                             (65535, 1, 64), (65537, 2049, 32)])
def test_pieces(op, dtype, blocks, extra, gs):
    numel = blocks * 256 * (16 // dtype.itemsize) + extra
    packed, scales = _packed(op, numel, gs)
    print(f"decode pieces {op} {dtype} blocks={blocks} gs={gs}", flush=True)
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    out = op(packed, scales, numel, gs, dtype).view(bits)
    assert out.numel() == numel
    part = gs * 16 * 1365
    for at in range(0, numel, part):
        n = min(part, numel - at)
        c = int(at * CODE_BYTES[op])
        ref = op(packed[c:], scales[at // gs:], n, gs, dtype).view(bits)
        assert torch.equal(out[at:at + n], ref)


@pytest.mark.parametrize("op", list(CODE_BYTES))
def test_time_grows_with_the_size(op):
    """Half as many weights are not slower."""
    sizes, graphs = [(1 << 20) - 8, 1 << 21], []
    for numel in sizes:
        packed, scales = _packed(op, numel, 32)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            op(packed, scales, numel, 32, torch.float16)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            keep = [op(packed, scales, numel, 32, torch.float16) for _ in range(12)]
        graphs.append((graph, packed, scales, keep))
    best = [float("inf")] * 2
    for _ in range(10):
        for i, g in enumerate(graphs):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            g[0].replay()
            b.record()
            torch.cuda.synchronize()
            best[i] = min(best[i], a.elapsed_time(b))
    print(f"decode {op} {best}", flush=True)
    assert best[1] < 1.24 * best[0]  # 1.1; 1.28 to 1.4 with four pieces per lane for the larger
