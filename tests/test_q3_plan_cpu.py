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


@pytest.mark.parametrize("M,K,N,kernel", [(5, 4096, 11008, "block"), (6, 4096, 11008, "block"), (5, 8192, 8192, "block"),
                                          (6, 11008, 4096, "block"), (8, 8192, 8192, "block"), (7, 7680, 6328, "block"),
                                          (5, 5184, 5008, "direct"), (6, 5440, 5372, "direct"), (8, 8608, 4376, "direct"),
                                          (9, 4096, 11008, "direct"), (5, 4224, 14336, "direct")])
def test_five_to_eight_rows_of_a_large_matrix_stay_with_the_block_kernel(M, K, N, kernel):
    """On 256 compute units: its passes and row blocks take 2 to 17 % less than the one-launch kernel while four rows would have a
    compute unit for every workgroup (not the last: 448 of them) and the matrix has 3.5e7 weights and more (seven and eight rows: 4e7)."""
    choose = getattr(_lib.load(), "_Z18hq_q3_batch_kerneliiii")
    assert ("block", "direct", "rows64", "tiles")[choose(256, K, N, M)] == kernel


@pytest.mark.parametrize("M,K,N,kernel", [(8, 4160, 19972, "direct"), (7, 4960, 24904, "direct"), (5, 5120, 13824, "direct"),
                                          (6, 15936, 12176, "block"), (8, 15936, 12176, "direct"), (6, 10976, 12176, "direct"),
                                          (5, 12128, 17920, "direct"), (5, 12128, 16384, "block"), (6, 15936, 10176, "direct"),
                                          (8, 4096, 19648, "block"), (8, 4096, 19652, "direct"), (7, 8256, 8500, "block"),
                                          (7, 8704, 8500, "direct"), (8, 16416, 9000, "block")])
def test_five_to_eight_rows_in_more_workgroups_than_compute_units(M, K, N, kernel):
    """7e7 weights and more, on either side of each line: up to a fifth more workgroups than compute units (307 of 64 columns; a last
    range of K that is nearly empty counts for nothing), five and six rows of K >= 11000 in evenly filled rounds, K beyond 16384."""
    choose = getattr(_lib.load(), "_Z18hq_q3_batch_kerneliiii")
    assert ("block", "direct", "rows64", "tiles")[choose(256, K, N, M)] == kernel


@pytest.mark.parametrize("M,K,N,kernel", [(8, 3680, 19904, "block"), (8, 4064, 24576, "block"), (8, 4064, 24580, "direct"), (5, 10368, 10116, "block"),
                                          (5, 15872, 15488, "block"), (5, 7968, 21376, "block"), (5, 6976, 21376, "direct"),
                                          (5, 7968, 25000, "direct"), (6, 7968, 21376, "direct")])
def test_more_workgroups_than_compute_units_that_stay(M, K, N, kernel):
    """On either side of each line: a K of less than a round in up to half as many workgroups again; five rows of K >= 7000 in evenly
    filled rounds, or in up to three with a last range of K that is nearly whole."""
    choose = getattr(_lib.load(), "_Z18hq_q3_batch_kerneliiii")
    assert ("block", "direct", "rows64", "tiles")[choose(256, K, N, M)] == kernel


@pytest.mark.parametrize("M,K,N,tiles_us,cut", [(263, 2240, 13548, 28.2, False), (1848, 288, 9420, 21.6, False), (135, 3584, 25704, 42.1, False),
                                                (1024, 2048, 8448, 45.9, True), (1902, 1056, 13184, 62.4, True), (129, 2304, 23920, 28.2, False)])
def test_columns_are_cut_off_where_that_gains_more_than_a_launch(M, K, N, tiles_us, cut):
    """The estimate of a call beside that of whole tiles (tiles_us, and the pre-pass): less by a microsecond and more, or the same."""
    import ctypes
    us = getattr(_lib.load(), "_Z14hq_q3_tiles_usiiii")
    us.restype = ctypes.c_float
    whole = tiles_us + 3.2 + 0.0002 * K + M * K * 4 / 4.5e6
    assert (us(256, K, N, M) < whole - 1) if cut else abs(us(256, K, N, M) - whole) < 0.1


@pytest.mark.parametrize("M,K,N,kernel", [(576, 1280, 14524, "direct"), (1999, 960, 4492, "direct"), (1179, 1216, 7208, "direct"),
                                          (1654, 2144, 5056, "tiles"), (324, 2432, 23040, "tiles"), (1992, 768, 16592, "tiles")])
def test_cut_tiles_beside_the_one_launch_kernel(M, K, N, kernel):
    """The estimate of tiles with their last columns cut off stands against that of the one-launch kernel for all columns."""
    choose = getattr(_lib.load(), "_Z18hq_q3_batch_kerneliiii")
    assert ("block", "direct", "rows64", "tiles")[choose(256, K, N, M)] == kernel
