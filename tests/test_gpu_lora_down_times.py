"""Times of the adapter's down-projection against each other on one card: pairs of calls of
nearly the same work, one of which once took a form that did not fit it."""

import pytest
import torch

from ojasx_amd import _native as N

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
f32, f16, bf16 = torch.float32, torch.float16, torch.bfloat16


def _graph(M, K, rank, dtype, launches=12):
    x = torch.zeros(M, K, dtype=dtype, device=DEV)
    a = torch.zeros(K, rank, dtype=dtype, device=DEV)
    u = torch.empty(M, rank, device=DEV)

    def down():
        N.check(N.lib().ojx_lora_down(N.ptr(x), N.ptr(a), M, K, rank, 1.0, N.DTYPE_CODE[dtype],
                                      N.ptr(u), N.stream_handle(DEV)), "lora_down")

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        down()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        for _ in range(launches):
            down()
    return graph, (x, a, u)


def _ratio(first, second):
    """Time of the first call over the second's: the best of ten runs each, in turn."""
    graphs = [_graph(*first), _graph(*second)]
    best = [float("inf")] * 2
    for _ in range(10):
        for i, (graph, _) in enumerate(graphs):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            graph.replay()
            b.record()
            torch.cuda.synchronize()
            best[i] = min(best[i], a.elapsed_time(b))
    print(f"lora down {first} / {second}: {best[0] / best[1]:.2f}", flush=True)
    return best[0] / best[1]


@pytest.mark.parametrize("rank", [16, 24, 64])
def test_two_workgroups_per_cu_in_both_types(rank):
    # 1.01, 1.05 and 1.07; 1.24, 1.27 and 1.22 with one workgroup per CU in bfloat16
    assert _ratio((384, 4096, rank, bf16), (384, 4096, rank, f16)) < 1.15


@pytest.mark.parametrize("first,second,limit", [
    # rows of no whole 16-byte pieces against the next multiple of eight: value by value in a
    # workgroup per row, not in tiles of 16 rows
    ((64, 1001, 8, bf16), (64, 1008, 8, bf16), 2.2),  # 1.49; 4.9 in tiles
    ((300, 1001, 3, f32), (300, 1001, 4, f32), 0.98),  # 0.87; 1.09 with both in tiles
    ((300, 1001, 3, f32), (300, 1008, 8, f32), 1.8),  # 0.97; 2.5 in tiles
    # ranks of no whole pieces: a workgroup per row for few ranks, tiles for many
    ((64, 4096, 3, f32), (64, 4096, 8, f32), 1.4),  # 1.16; 1.85 in tiles
    ((64, 256, 3, bf16), (64, 256, 8, bf16), 1.1),  # 0.97; 1.22 in tiles
    ((64, 14336, 12, bf16), (64, 14336, 16, bf16), 2.2),  # 1.92, in tiles
    # 512 rows fill the CUs twice, as 448 do; 520 are in tiles
    ((512, 1024, 16, bf16), (448, 1024, 16, bf16), 1.15),  # 1.01; 1.36 as 513 rows
    ((520, 14336, 16, bf16), (448, 14336, 16, bf16), 1.35),  # 1.15
])
def test_forms_by_size(first, second, limit):
    assert _ratio(first, second) < limit
