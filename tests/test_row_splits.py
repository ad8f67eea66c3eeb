"""K splits of one row of small GEMM tiles (17 to 128 rows; the backward also fewer), read off the
workspace query: at measured shapes the choice is within 5% of the best time.

Times: us from a graph on one MI355X, ternary group 32 in bf16, by split count.
"""

import ctypes

import pytest

from ojasx_amd import _native as N
from ojasx_amd import ops

# (backward, M, columns, reduction): {splits: us}
TIMES = {
    (0, 17, 1024, 4096): {1: 58.8, 8: 14.9, 16: 12.4},
    (0, 64, 1024, 1024): {2: 15.0, 4: 11.9},
    (0, 17, 8192, 4096): {1: 58.3, 2: 34.3, 3: 26.4, 4: 21.6, 5: 22.9, 6: 21.1, 7: 19.9, 8: 18.1,
                          10: 24.7},
    (0, 64, 8192, 4096): {1: 59.6, 2: 35.7, 3: 27.9, 4: 23.3, 5: 24.5, 6: 23.0, 7: 22.0, 8: 20.7,
                          10: 28.0},
    (0, 64, 9216, 3072): {1: 46.8, 2: 30.6, 3: 25.4, 4: 27.0, 5: 25.9, 6: 25.0, 7: 25.1, 8: 31.9},
    (0, 64, 6144, 4096): {1: 59.7, 2: 36.4, 3: 29.1, 4: 25.0, 5: 23.4, 6: 25.6, 7: 25.5, 8: 24.2,
                          10: 24.4, 12: 30.8},
    (0, 64, 11008, 4096): {2: 38.4, 5: 28.4, 6: 38.7},
    (0, 17, 4096, 11008): {1: 146.3, 2: 78.8, 4: 43.9, 8: 27.5, 10: 29.3, 12: 26.7, 14: 25.0,
                           16: 23.6},
    (1, 64, 1024, 1024): {1: 22.6, 4: 13.0},
    (1, 1, 11008, 4096): {2: 40.0, 4: 32.2, 5: 28.1},
    (1, 64, 11008, 4096): {2: 42.4, 4: 35.9, 5: 32.6},
    (1, 64, 4096, 8192): {1: 125.6, 2: 69.5, 4: 40.8, 8: 27.8, 10: 31.6, 12: 29.5, 14: 28.1,
                          16: 26.7},
    (1, 64, 4096, 11008): {1: 165.7, 2: 90.1, 4: 50.6, 8: 32.3, 10: 36.8, 12: 33.8, 14: 31.4,
                           16: 30.0},
}


def _splits(bwd, M, cols, red):
    n, k = (red, cols) if bwd else (cols, red)
    nbytes = ctypes.c_size_t(0)
    N.check(N.lib().ojx_gemm_workspace_bytes(ops.FMT_TERNARY, bwd, M, n, k, 32, N.BF16,
                                             ctypes.byref(nbytes)), "gemm_workspace_bytes")
    return max(1, nbytes.value // (4 * M * cols))


@pytest.mark.parametrize("case", sorted(TIMES))
def test_measured_shapes(case):
    times = TIMES[case]
    assert times[_splits(*case)] <= 1.05 * min(times.values())


@pytest.mark.parametrize("bwd", [0, 1])
def test_bounds(bwd):
    """At least four 64-k steps per split and at most two workgroups per CU."""
    for M in (1, 17, 64, 128):
        if M < 17 and not bwd:
            continue
        for cols in (64, 320, 1024, 4096, 6144, 11008, 16384):
            for red in (64, 192, 256, 512, 576, 1088, 4096, 14336):
                s = _splits(bwd, M, cols, red)
                if -(-cols // 256) * 16 >= 192:
                    continue  # large tiles can be split far enough
                assert s == 1 or red // 64 // s >= 4
                assert s == 1 or s * -(-cols // 128) <= 512
