"""Calls on different streams use different workspaces and may overlap: interleaved split-K
matvecs and batched GEMMs on two streams give the results of the same calls on one stream."""
import ctypes

import numpy as np
import pytest

from tests import oracle_api as oa

pytestmark = pytest.mark.gpu


def test_two_streams_interleaved(hq, oracle, tunable):
    import torch
    dev = torch.device("cuda:0")
    tunable("HQ_Q3_KSPLIT", 4)          # force the cross-workgroup reduction (workspace + counters)
    tunable("HQ_Q3_WAVES", 4)
    tunable("HQ_Q3_STEPS", 1)
    K, N, M = 2048, 512, 24
    problems = []
    for seed in (1, 2):
        codes, scales, zeros, x = oa.make_q3_problem(100 + seed, K, N)
        mat = oracle.q3_pack(codes)
        A = np.random.default_rng(seed).standard_normal((M, K)).astype(np.float16)
        problems.append(tuple(torch.from_numpy(t).to(dev) for t in (x, mat, scales, zeros, A)))
    # one stream, one call at a time
    want = []
    for x, mat, s, z, A in problems:
        want.append((hq.q3_matvec(x, mat, s, z).clone(), hq.q3_gemm(A, mat, s, z).clone()))
    torch.cuda.synchronize()
    # two streams, many interleaved calls in flight
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [[], []]
    for rep in range(20):
        for i, st in enumerate(streams):
            x, mat, s, z, A = problems[i]
            with torch.cuda.stream(st):
                outs[i].append((hq.q3_matvec(x, mat, s, z), hq.q3_gemm(A, mat, s, z)))
    torch.cuda.synchronize()
    for i in range(2):
        for y, g in outs[i]:
            assert torch.equal(y, want[i][0])
            assert torch.equal(g, want[i][1])


def test_a_reservation_allocates_what_it_names(hq):
    """Memory of a stream's reservation: what hq_reserve_need tells, rounded to the allocator's units and not to a power of two."""
    import torch
    from hecbench_amd import _lib
    lib = _lib.load()
    cus = hq.device_info()["compute_units"]
    stream = torch.cuda.Stream()
    for K, N in ((512, 512), (4096, 11008)):     # the second one replaces the first one's buffer, which stays
        f, c = ctypes.c_int64(), ctypes.c_int64()
        assert lib.hq_reserve_need(cus, K, N, ctypes.byref(f), ctypes.byref(c)) == 0
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        assert lib.hq_reserve_workspace(ctypes.c_void_p(stream.cuda_stream), K, N) == 0
        taken = free - torch.cuda.mem_get_info()[0]
        assert taken <= f.value * 4 + c.value * 4 + (6 << 20), (K, N, taken, f.value * 4)


def test_a_reservation_is_enough_for_the_lut_kernels(hq):
    """Whatever the split of K and the meeting of its shares: no call of those sizes allocates."""
    import torch
    from hecbench_amd import _lib
    lib = _lib.load()
    torch.cuda.synchronize()
    assert lib.hq_shutdown() == 0
    stream = torch.cuda.Stream()
    maxK, maxN = 8192, 9000
    buf = torch.zeros(maxK * maxN // 8 * 4, dtype=torch.uint8, device="cuda:0")
    alpha = torch.zeros(maxK // 32 * 4 * maxN, dtype=torch.float16, device="cuda:0")
    x, y = torch.zeros(maxK, device="cuda:0").half(), torch.zeros(maxN, device="cuda:0").half()
    vp = lambda t: ctypes.c_void_p(t.data_ptr())
    call = lambda K, N, nb, G, s: lib.hq_lut_gemv(vp(buf), vp(alpha), None, vp(x), vp(y), K, N, nb, G, ctypes.c_void_p(s))
    shapes = [(K, N, nb, G) for K in (1152, 2304, 4224, 8192) for N in (64, 700, 2166, 4096, 9000) for nb, G in ((1, 128), (3, 128), (2, 64), (4, 32))]
    for s in shapes:
        assert call(*s, 0) == 0  # (code objects, and the default stream's workspace)
    with torch.cuda.stream(stream):
        y.zero_()  # (the stream's own queue)
    torch.cuda.synchronize()
    assert lib.hq_reserve_workspace(ctypes.c_void_p(stream.cuda_stream), maxK, maxN) == 0
    free = torch.cuda.mem_get_info()[0]
    for s in shapes:
        assert call(*s, stream.cuda_stream) == 0
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] < 4 << 20  # (to grow is to take 8 MiB)
