"""hq_reserve_workspace promises that calls up to (max_K, max_N) never allocate: its bound (hq_reserve_need) must
cover the workspace need of every smaller call (hq_q3_workspace_need, computed by the launch's own plan
functions).  Host arithmetic only - no GPU."""
import ctypes
import random

import pytest

from hecbench_amd import _lib


def _need(lib, cus, K, N, M):
    f, c = ctypes.c_int64(), ctypes.c_int64()
    rc = lib.hq_q3_workspace_need(cus, K, N, M, ctypes.byref(f), ctypes.byref(c))
    assert rc == 0, (rc, cus, K, N, M)
    return f.value, c.value


def _bound(lib, cus, K, N):
    f, c = ctypes.c_int64(), ctypes.c_int64()
    assert lib.hq_reserve_need(cus, K, N, ctypes.byref(f), ctypes.byref(c)) == 0
    return f.value, c.value


BATCHES = (1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 13, 16, 24, 32, 33, 48, 64, 65, 72, 128)


@pytest.mark.parametrize("cus", [256, 304, 120, 64])
@pytest.mark.parametrize("max_K,max_N", [(8192, 28672), (16384, 65536), (4096, 4096), (49152, 12288), (1024, 256),
                                         (32768, 1024), (65536, 4096)])
def test_reserve_covers_every_smaller_call(cus, max_K, max_N):
    lib = _lib.load()
    bf, bc = _bound(lib, cus, max_K, max_N)
    rng = random.Random(cus * 1000003 + max_K * 31 + max_N)
    Ks = {max_K, 32, 4096, 8192, 2048, 1024, 128, 14336, 11008, 16384, 28672, 36864, 40960} | \
         {rng.randrange(1, max_K // 32 + 1) * 32 for _ in range(12)}
    Ns = {max_N, 4, 64, 128, 256, 1024, 2048, 4096, 4100, 8192, 11008, 12288, 22016} | \
         {rng.randrange(1, max_N // 4 + 1) * 4 for _ in range(12)}
    worst = (0, (0, 0, 0))
    for K in sorted(k for k in Ks if k <= max_K):
        for N in sorted(n for n in Ns if n <= max_N):
            for M in BATCHES:
                f, c = _need(lib, cus, K, N, M)
                assert f <= bf, ("floats", cus, K, N, M, f, bf)
                assert c <= bc, ("counters", cus, K, N, M, c, bc)
                worst = max(worst, (f, (K, N, M)))
    assert worst[0] > 0 or max_K < 2048


@pytest.mark.parametrize("cus", [256, 304, 64])
@pytest.mark.parametrize("max_K,max_N", [(512, 512), (1024, 4096), (1920, 4096), (4096, 11008), (16384, 16384), (49152, 12288)])
def test_reserve_is_close_to_the_largest_need(cus, max_K, max_N):
    """Batches of any size are covered, and no more is reserved than a quarter beyond what the largest of them takes (a layer of
    512 x 512 once reserved 68 MiB for a need of 8)."""
    lib = _lib.load()
    bf, bc = _bound(lib, cus, max_K, max_N)
    rng = random.Random(max_K + cus)
    worst = 0
    for i in range(6000):
        K = max_K if i % 2 else rng.randrange(1, max_K // 32 + 1) * 32
        N = max_N if i % 3 else rng.randrange(1, max_N // 4 + 1) * 4
        M = int(2 ** rng.uniform(6, 15))
        f, c = _need(lib, cus, K, N, M)
        assert f <= bf and c <= bc, (cus, K, N, M, f, bf, c, bc)
        worst = max(worst, f)
    assert bf <= 1.25 * worst


def test_the_array_of_the_call_that_allocates_nothing_holds_every_batch():
    """hq_q3_matvec_noalloc takes the tiles' plan at every batch as long as its fixed array holds it (68 MiB + 64 KiB, 16128
    arrival counters; 256 compute units, K <= 16384): there is no batch beyond 64 rows that it does not hold."""
    lib = _lib.load()
    rng = random.Random(17)
    for i in range(20000):
        K = (16384, 2080, rng.randrange(1, 513) * 32)[i % 3]   # the longest, one that pads much, any
        N = rng.randrange(1, 16385) * 4
        f, c = _need(lib, 256, K, N, int(2 ** rng.uniform(6.03, 15)))
        assert f * 4 <= (68 << 20) + (64 << 10) and c <= 16128, (K, N, f, c)


def test_the_case_that_used_to_fall_short():
    # 256 compute units: a reservation for (8192, 28672) must hold M=72, K=8192, N=4096, whose 32 column tiles
    # split K eight ways (re-ordered activations 262,144 floats + 128 + 32 x 8 x 64 x 128 raw sums)
    lib = _lib.load()
    f, _ = _need(lib, 256, 8192, 4096, 72)
    assert f == 262144 + 128 + 32 * 8 * 64 * 128
    bf, _ = _bound(lib, 256, 8192, 28672)
    assert bf >= f
    f2, _ = _need(lib, 256, 16384, 2048, 72)
    assert _bound(lib, 256, 16384, 65536)[0] >= f2


@pytest.mark.parametrize("M,K,N,shares,rows", [(1, 8192, 640, 2, 40), (1, 8192, 28672, 2, 448), (1, 28672, 4096, 7, 64), (4, 8192, 8256, 2, 129 * 4),
                                               (7, 8192, 640, 2, 10 * 8)])
def test_the_slots_of_a_few_shares_are_told(M, K, N, shares, rows):
    """A few shares of K meet in slots, of two counters each: a row of 64 per column tile (16 columns, where they are few), share but
    one and row of results (whole row blocks of four)."""
    lib = _lib.load()
    f, c = _need(lib, 256, K, N, M)
    assert f == rows * shares * 64 and c == 2 * rows * (shares - 1) * 64


@pytest.mark.parametrize("M,K,N,counters", [(1, 28672, 8192, 128), (3, 32768, 8192, 128), (2, 24576, 8192, 128), (1, 32768, 5696, 89),
                                            (1, 32768, 5632, 2 * 88 * 7 * 64)])
def test_many_workgroups_of_many_shares_count(M, K, N, counters):
    """Six to eight shares in more than two and three quarters workgroups per compute unit (the last: just not): arrival counters,
    and no slots."""
    assert _need(_lib.load(), 256, K, N, M)[1] == counters


def test_a_reservation_for_very_many_columns_has_slots_for_fewer():
    """Beyond 32 MiB of slots a call does without; a reservation that would take more holds those 32 MiB."""
    lib = _lib.load()
    assert _bound(lib, 256, 65536, 2000000)[1] == 2 * (4 << 20) + 256 // 8  # (and the arrival counters of AQLM calls in slices)
    assert _need(lib, 256, 20480, 65536, 1)[1] == 2 * 1024 * 4 * 64
    assert _need(lib, 256, 20480, 1200000, 1)[1] == 18750  # arrival counters


def test_bad_arguments():
    lib = _lib.load()
    f, c = ctypes.c_int64(), ctypes.c_int64()
    assert lib.hq_q3_workspace_need(256, 100, 64, 1, ctypes.byref(f), ctypes.byref(c)) < 0
    assert lib.hq_q3_workspace_need(0, 128, 64, 1, ctypes.byref(f), ctypes.byref(c)) < 0
    assert lib.hq_reserve_need(256, -1, 64, ctypes.byref(f), ctypes.byref(c)) < 0
    assert lib.hq_reserve_need(256, 128, 64, None, ctypes.byref(c)) < 0
