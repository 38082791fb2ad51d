"""Parity of hq_aqlm_matvec with the CPU oracle (and, where built, the
reference's own kernel), through the C ABI."""
import ctypes

import numpy as np
import pytest

from tests import oracle_api as oa
from tests.tol import FLOOR_F16, TOL_F16_ACC, rel_err

pytestmark = pytest.mark.gpu


def _run(hq, codes, codebooks, scales, x, sizes, stride=65536):
    import torch
    dev = torch.device("cuda:0")
    t = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    y = hq.code1x16_matvec(t(codes), t(x), t(codebooks), sizes, stride, scales=t(scales))
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("M,K,seed", [(4096, 4096, 1), (64, 256, 2), (1000, 1024, 3), (7, 8192, 4), (3, 64, 5)])
def test_vs_oracle(hq, oracle, M, K, seed):
    codes, cb, scales, x = oa.make_aqlm_problem(seed, M, K)
    y = _run(hq, codes, cb, scales, x, (M, 0, 0, 0))
    _, ref64 = oracle.aqlm_matvec(codes, cb, scales, x, (M, 0, 0, 0), 65536, mode=0)
    assert rel_err(y, ref64) <= 2e-3
    ref16, _ = oracle.aqlm_matvec(codes, cb, scales, x, (M, 0, 0, 0), 65536, mode=1)
    assert rel_err(y, ref16.astype(np.float64), FLOOR_F16) <= TOL_F16_ACC


@pytest.mark.parametrize("M,K,rows", [(5, 8192, 1), (5, 8256, 1), (9, 24576, 2), (9, 24640, 4), (11, 4160, 4), (4, 4096, 2), (6, 8128, 4), (2049, 64, 1),
                                      (1, 64, 11), (3, 512, 12), (5, 1600, 11), (7, 2112, 12), (9, 24576, 12), (4, 24640, 11)])
def test_activations_in_lds_and_not(hq, oracle, tunable, M, K, rows):
    """Either side of the longest row whose activations go through LDS, chunks of 512 codes whole and cut, the last workgroup
    with waves that have no row; waves that share rows (11, 12), some without a chunk."""
    tunable("HQ_AQLM_ROWS", rows)
    codes, cb, scales, x = oa.make_aqlm_problem(M + K, M, K)
    y = _run(hq, codes, cb, scales, x, (M, 0, 0, 0))
    _, ref64 = oracle.aqlm_matvec(codes, cb, scales, x, (M, 0, 0, 0), 65536, mode=0)
    assert rel_err(y, ref64, FLOOR_F16) <= 2e-3


@pytest.mark.parametrize("M,K", [(2049, 4096), (2048, 4160), (1001, 8256), (4097, 8320), (8193, 576)])
def test_default_rules(hq, oracle, M, K):
    codes, cb, scales, x = oa.make_aqlm_problem(M + 2 * K, M, K)
    y = _run(hq, codes, cb, scales, x, (M, 0, 0, 0))
    _, ref64 = oracle.aqlm_matvec(codes, cb, scales, x, (M, 0, 0, 0), 65536, mode=0)
    assert rel_err(y, ref64, FLOOR_F16) <= 2e-3


@pytest.mark.parametrize("sub", [0, 1, 2])
@pytest.mark.parametrize("M,K,ncb", [(1, 64, 1), (31, 1024, 1), (33, 1088, 3), (2049, 2112, 1), (2100, 4096, 3), (8193, 1600, 1), (70, 15872, 3)])
def test_code_book_in_slices(hq, oracle, tunable, M, K, ncb, sub):
    """Groups of rows without rows, of one and of several trips, the last with waves that have none; rows of one run of lanes and of
    several, the last cut; the longest K; groups with rows of several code books, one of them empty."""
    codes, cb, scales, x = oa.make_aqlm_problem(M + 3 * K, M, K, ncb=ncb)
    sizes = (M, 0, 0, 0) if ncb == 1 else (M // 3, M // 3, M // 2, M)
    if ncb == 3:
        cb = np.concatenate([cb, cb[:1] * np.float16(2)])
    tunable("HQ_AQLM_ROWS", 20 + sub)
    y = _run(hq, codes, cb, scales, x, sizes)
    _, ref64 = oracle.aqlm_matvec(codes, cb, scales, x, sizes, 65536, mode=0)
    assert rel_err(y, ref64, FLOOR_F16) <= 2e-3
    assert np.array_equal(y.view(np.uint16), _run(hq, codes, cb, scales, x, sizes).view(np.uint16))


def test_groups_without_rows_of_several_code_books(hq, oracle, tunable):
    test_code_book_in_slices(hq, oracle, tunable, 20, 128, 3, 0)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_slices_and_numbers_that_are_none(hq, tunable, bad):
    """An infinity or NaN among the activations, or in a code book, reaches the outputs that it reaches without slices, as it does there."""
    M, K = 300, 640
    codes, cb, scales, x = oa.make_aqlm_problem(77, M, K)
    for in_x in (True, False):
        xs, cbs = x.copy(), cb.copy()
        if in_x:
            xs[K // 2] = bad
            cbs[0, codes[5, K // 16].astype(np.uint16), (K // 2) % 8] = 0  # times zero: NaN there
        else:
            cbs[0, codes[7, 3].astype(np.uint16), 2] = bad
            xs[8 * np.arange(K // 8)[codes[9] == codes[7, 3]] + 2] = 0
        got = []
        for knob in (1, 21):
            tunable("HQ_AQLM_ROWS", knob)
            got.append(_run(hq, codes, cbs, scales, xs, (M, 0, 0, 0)).astype(np.float64))
        fin = np.isfinite(got[0])
        assert not fin.all() and np.array_equal(got[0][~fin], got[1][~fin], equal_nan=True)
        assert not fin.any() or rel_err(got[1][fin], got[0][fin], FLOOR_F16) <= 2e-3


def test_default_takes_slices_but_not_under_capture(hq, tunable):
    import torch
    M, K = 8192, 4096
    codes, cb, scales, x = oa.make_aqlm_problem(8, M, K)
    t = [torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0") for a in (codes, x, cb, scales)]
    call = lambda: hq.code1x16_matvec(t[0], t[1], t[2], (M, 0, 0, 0), 65536, scales=t[3])
    y = call()
    want = {}
    for knob in (2, 22):
        tunable("HQ_AQLM_ROWS", knob)
        want[knob] = call()
    assert torch.equal(y, call())           # as forced: in slices
    assert not torch.equal(want[2], want[22])  # (sums in another order round differently somewhere among 8192)
    from hecbench_amd import _lib
    _lib.load().hq_set_tunable(b"HQ_AQLM_ROWS", 0, 1)
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            out = call()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert rel_err(out.cpu().numpy(), y.cpu().numpy().astype(np.float64), FLOOR_F16) <= 2e-3
        assert torch.equal(call(), y)


def _many_codes(seed, M=8192, K=4096):
    import torch
    codes, cb, scales, x = oa.make_aqlm_problem(seed, M, K)
    t = [torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0") for a in (codes, cb, scales, x)]
    y = torch.zeros(M, dtype=torch.float16, device="cuda:0")
    sizes = (ctypes.c_int * 4)(M, M, M, M)
    vp = lambda a: ctypes.c_void_p(a.data_ptr())

    def call(stream):
        from hecbench_amd import _lib
        assert _lib.load().hq_aqlm_matvec(vp(t[0]), vp(t[1]), vp(t[2]), vp(t[3]), vp(y), M, K, sizes, 65536, ctypes.c_void_p(stream)) == 0
        return y
    return call


def test_slices_beside_replays_of_the_same_stream(hq, tunable):
    """A graph with a divided K captured on a stream, replayed on another one beside eager calls in slices on the first: neither
    touches what the other leaves in memory.  The same with calls of this operator in the graph."""
    import torch
    torch.cuda.synchronize()
    call = _many_codes(12)
    K, N = 8192, 28672
    mat = torch.randint(-2 ** 31, 2 ** 31 - 1, (3 * K // 32, N), dtype=torch.int32, device="cuda:0")
    s = torch.full((N,), 0.01, device="cuda:0")
    x = torch.randn(K, device="cuda:0")
    captured, other = torch.cuda.Stream(), torch.cuda.Stream()
    want_q3 = hq.q3_matvec(x, mat, s, 4 * s)
    with torch.cuda.stream(captured):
        captured.wait_stream(torch.cuda.default_stream())
        hq.q3_matvec(x, mat, s, 4 * s)
        y = call(captured.cuda_stream)
    torch.cuda.synchronize()
    want, outs = y.clone(), [torch.zeros_like(want_q3) for _ in range(8)]
    beside = _many_codes(13)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=captured):
        for o in outs:
            hq.q3_matvec(x, mat, s, 4 * s, out=o)
            y_beside = beside(captured.cuda_stream)
    with torch.cuda.stream(other):
        graph.replay()
    torch.cuda.synchronize()
    want_beside = y_beside.clone()
    assert not torch.equal(want, want_beside)
    for rep in range(30):
        with torch.cuda.stream(other):
            graph.replay()
        got = []
        with torch.cuda.stream(captured):
            for _ in range(8):
                got.append(call(captured.cuda_stream).clone())
        torch.cuda.synchronize()
        assert all(torch.equal(o, want_q3) for o in outs) and torch.equal(y_beside, want_beside), rep
        assert all(torch.equal(g, want) for g in got), rep


def test_the_first_call_in_slices_beside_a_capture(hq):
    """A stream's first call of millions of codes, while another stream is being captured: it runs, and the capture is whole."""
    import torch
    from hecbench_amd import _lib
    call, inside = _many_codes(14), _many_codes(15)
    call(0), inside(0)
    torch.cuda.synchronize()
    assert _lib.load().hq_shutdown() == 0
    want, want_inside = call(0).clone(), inside(0).clone()
    captured, eager = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=captured):
        y = inside(captured.cuda_stream)
        got = call(eager.cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert rel_err(y.cpu().numpy(), want_inside.cpu().numpy().astype(np.float64), FLOOR_F16) <= 2e-3


def test_a_reservation_inside_a_relaxed_capture(hq):
    """Where a capture allows allocations, a reservation of the captured stream is no part of the graph: the stream's eager calls
    find their counters at zero although nothing is ever replayed."""
    import torch
    from hecbench_amd import _lib
    lib = _lib.load()
    call = _many_codes(16)
    call(0)
    torch.cuda.synchronize()
    assert lib.hq_shutdown() == 0  # torch hands streams out again: none has a workspace from here on
    want = call(0).clone()
    torch.cuda.synchronize()
    used = []
    for n in (1 << 16, 1 << 18, 1 << 20, 1 << 21) * 8:  # what the reservation is likely to be given: not zero
        p = ctypes.c_void_p()
        assert lib.hipMalloc(ctypes.byref(p), ctypes.c_size_t(n)) == 0 and lib.hipMemset(p, 0xff, ctypes.c_size_t(n)) == 0
        used.append(p)
    torch.cuda.synchronize()
    for p in used:
        assert lib.hipFree(p) == 0
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
        want + 1
        assert lib.hq_reserve_workspace(ctypes.c_void_p(stream.cuda_stream), 4096, 8192) == 0
    torch.cuda.synchronize()
    for _ in range(3):
        got = call(0).zero_()
        torch.cuda.synchronize()
        call(stream.cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(got, want)


def test_three_codebooks_and_no_scale(hq, oracle):
    """Reference default geometry: 3 code books of 4096 rows each, no scale."""
    M, K = 12288, 1024
    codes, cb, _, x = oa.make_aqlm_problem(11, M, K, ncb=3)
    sizes = (4096, 8192, 12288, 122880)
    y = _run(hq, codes, cb, None, x, sizes)
    _, ref64 = oracle.aqlm_matvec(codes, cb, None, x, sizes, 65536, mode=0)
    assert rel_err(y, ref64) <= 2e-3
    # partition boundaries: constant code books make the row's code book visible
    cbc = np.zeros((3, 65536, 8), np.float16)
    cbc[0], cbc[1], cbc[2] = 1.0, 2.0, 3.0
    xs = np.ones(K, np.float16) / 8
    y = _run(hq, codes, cbc, None, xs, sizes)
    assert (y[:4096] == K / 8).all() and (y[4096:8192] == 2 * K / 8).all() and (y[8192:] == 3 * K / 8).all()


def test_signed_codes_and_gather(hq, oracle):
    """-1 -> entry 65535, -32768 -> entry 32768; one-hot entries gather x."""
    M, K = 4, 64
    cb = np.zeros((1, 65536, 8), np.float16)
    cb[0, 65535, 0] = 1.0
    cb[0, 32768, 7] = 1.0
    cb[0, 5, 3] = 1.0
    codes = np.zeros((M, K // 8), np.int16)
    codes[0, :] = -1
    codes[1, :] = -32768
    codes[2, :] = 5
    x = (np.arange(K) + 1).astype(np.float16)
    y = _run(hq, codes, cb, None, x, (M, 0, 0, 0))
    assert y[0] == x[0::8].astype(np.float64).sum()
    assert y[1] == x[7::8].astype(np.float64).sum()
    assert y[2] == x[3::8].astype(np.float64).sum()
    assert y[3] == 0


def test_vs_reference_kernel(hq, oracle):
    import torch
    ref = oa.load_ref_hip()
    if ref is None:
        pytest.skip("oracle/_ref/libhecref_hip.so not built")
    dev = torch.device("cuda:0")
    M, K = 12288, 4096
    codes, cb, _, x = oa.make_aqlm_problem(31, M, K, ncb=3)
    sizes = (4096, 8192, 12288, 122880)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    dc, dcb, dx = t(codes), t(cb), t(x)
    out = torch.zeros(M, dtype=torch.float16, device=dev)
    vp = lambda a: ctypes.c_void_p(a.data_ptr())
    ref.ref_code1x16_launch(vp(dc), vp(dx), vp(out), vp(dcb), M, K, (ctypes.c_int * 4)(*sizes), 65536, None)
    torch.cuda.synchronize()
    y = hq.code1x16_matvec(dc, dx, dcb, sizes, 65536)
    torch.cuda.synchronize()
    r = out.cpu().numpy()
    assert rel_err(y.cpu().numpy(), r, FLOOR_F16) <= TOL_F16_ACC
    # the oracle's restatement of the reference arithmetic matches the real kernel bit for bit
    ref16, _ = oracle.aqlm_matvec(codes[:256], cb, None, x, sizes, 65536, mode=1)
    assert np.array_equal(ref16.view(np.uint16), r[:256].view(np.uint16))
