"""The host's share of a batched 3-bit call: choosing the kernel (hq_q3_workspace_need makes the launch's own choice).  Host
arithmetic only - no GPU."""
import ctypes
import time

import pytest

from hecbench_amd import _lib


def _us(lib, K, N, M):
    f, c = ctypes.c_int64(), ctypes.c_int64()
    pf, pc = ctypes.byref(f), ctypes.byref(c)
    fn = ctypes.CDLL(lib._name).hq_q3_workspace_need  # without argument types, whose checks would be half of the time
    best = float("inf")
    for _ in range(60):
        t = time.perf_counter()
        for _ in range(500):
            fn(256, K, N, M, pf, pc)
        best = min(best, (time.perf_counter() - t) / 500)
    return best * 1e6


@pytest.mark.parametrize("K,N,M", [(4096, 4096, 8), (1024, 512, 16)])
def test_a_batch_that_keeps_its_row_blocks_makes_no_other_plan(K, N, M):
    """Calls of a few microseconds, bound by the host.  Making the one-launch kernel's plan in order to reject it took these as
    long again as all else (0.33 us with the call through ctypes, four rows, which no other kernel competes for; 0.61 with it)."""
    lib = _lib.load()
    assert _us(lib, K, N, M) <= 1.4 * _us(lib, K, N, 4)
