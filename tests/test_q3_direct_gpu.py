"""The one-launch kernel of the batched 3-bit product (q3_direct.hip): every form, undivided and divided along K, at the edges of
tiles, steps and k-groups, against the oracle row by row; and the library's own choice of it."""
import ctypes

import numpy as np
import pytest

from tests import oracle_api as oa
from tests.q3_kernel import kernel_of
from tests.tol import FLOOR_F16, rel_err

pytestmark = pytest.mark.gpu


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def _check(y, exact):
    for m in range(len(y)):
        if exact[m].any():
            assert rel_err(y[m], exact[m], FLOOR_F16) <= 1e-4, m
        else:
            assert not y[m].any(), m


@pytest.mark.parametrize("kind,shares", [(3, 1), (3, 2), (3, 8), (4, 1), (4, 3), (5, 1), (5, 2), (5, 5), (6, 1), (6, 2)])
@pytest.mark.parametrize("M,K,N", [(2, 32, 4), (31, 96, 132), (32, 1024, 128), (33, 2080, 260), (65, 4128, 68), (13, 1376, 1028)])
def test_forms_and_shares(hq, oracle, tunable, kind, shares, M, K, N):
    codes, scales, zeros, A = oa.make_q3_problem(M + K + N, K, N, x_dtype=np.float16, batch=M)
    plain = np.ones(M, bool)
    if M > 10:
        A[5] *= np.float16(2.0 ** -14)     # rows of other magnitudes, down to subnormal numbers, a zero row, an outlier
        A[7] = 0
        A[9, K // 64 * 32 + 3] = np.float16(4096.0)
        plain[[7, 9]] = False
    mat = oracle.q3_pack(codes)
    tunable("HQ_Q3_TILES", kind + 10 * shares)
    y = hq.q3_gemm(_t(A), _t(mat), _t(scales), _t(zeros))
    again = hq.q3_gemm(_t(A), _t(mat), _t(scales), _t(zeros))
    assert np.array_equal(y.cpu().numpy(), again.cpu().numpy())  # shares are added in a fixed order
    exact = oracle.q3_gemm(A, mat, scales, zeros, mode=0)
    y = y.cpu().numpy()
    _check(y, exact)
    # codes and activations are exact operands and the row sums are fp32: what is left is the scatter of the matrix
    # instruction's cuts, 2e-7 of the result at K=4096 in 2-norm (short sums lose less)
    d = y[plain].astype(np.float64) - exact[plain]
    assert np.linalg.norm(d) <= 1e-6 * np.linalg.norm(exact[plain])


@pytest.mark.parametrize("kind", [3, 4, 5, 6])
def test_error_does_not_grow_with_an_offset(hq, oracle, tunable, kind):
    """Odd parts of K enter negated, so that the matrix instruction's cuts, all towards minus infinity, cancel."""
    M, K, N = 40, 8192, 260
    codes, scales, zeros, A = oa.make_q3_problem(77, K, N, x_dtype=np.float16, batch=M)
    mat = oracle.q3_pack(codes)
    tunable("HQ_Q3_TILES", kind)
    y = hq.q3_gemm(_t(A), _t(mat), _t(scales), _t(zeros)).cpu().numpy().astype(np.float64)
    exact = oracle.q3_gemm(A, mat, scales, zeros, mode=0)
    err = (y - exact) / scales
    assert np.linalg.norm(y - exact) <= 5e-7 * np.linalg.norm(exact)
    assert abs(err.mean()) <= 0.25 * np.sqrt(np.mean(err ** 2))


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_infinities_and_nan_stay_in_their_row(hq, oracle, tunable, bad):
    M, K, N = 35, 352, 136       # the last step of K is cut short in every form: what it loads instead is taken as zero
    codes, scales, zeros, A = oa.make_q3_problem(5, K, N, x_dtype=np.float16, batch=M)
    A[3, K - 1] = bad
    mat = oracle.q3_pack(codes)
    good = np.arange(M) != 3
    exact = oracle.q3_gemm(A[good], mat, scales, zeros, mode=0)
    for kind in (3, 4, 5, 6):
        tunable("HQ_Q3_TILES", kind)
        y = hq.q3_gemm(_t(A), _t(mat), _t(scales), _t(zeros)).cpu().numpy()
        assert not np.isfinite(y[3]).any()
        _check(y[good], exact)


@pytest.mark.parametrize("M,K,N", [(16, 5120, 3068), (45, 3648, 5028), (70, 4096, 4096), (341, 4416, 644), (80, 9216, 1000)])
def test_default_plans(hq, oracle, M, K, N):
    """Problems that the library gives to this kernel by itself (more precise than any other of the batched product), and the call
    that allocates nothing, which returns the same bits; with and without accumulation."""
    import torch
    from hecbench_amd import _lib
    lib = _lib.load()
    assert kernel_of(M, K, N) == "direct"
    codes, scales, zeros, A = oa.make_q3_problem(M + K, K, N, x_dtype=np.float16, batch=M)
    mat = oracle.q3_pack(codes)
    a, w, s, z = _t(A), _t(mat), _t(scales), _t(zeros)
    cols = np.unique(np.concatenate([np.arange(0, 70), np.arange(N - 70, N)]))
    exact = oracle.q3_gemm(A, np.ascontiguousarray(mat[:, cols]), scales[cols], zeros[cols], mode=0)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    got = {}
    for flags in (0, 1):
        for fn in (lib.hq_q3_matvec, lib.hq_q3_matvec_noalloc):
            y = torch.full((M, N), 3.0, device="cuda:0")
            assert fn(a.data_ptr(), 1, w.data_ptr(), s.data_ptr(), z.data_ptr(), y.data_ptr(), K, N, M, flags, stream) == 0
            torch.cuda.synchronize()
            got[flags, fn is lib.hq_q3_matvec] = y
        assert torch.equal(got[flags, True], got[flags, False])
    y = got[0, True].cpu().numpy()[:, cols].astype(np.float64)
    assert np.linalg.norm(y - exact) <= 5e-7 * np.linalg.norm(exact)
    assert torch.equal(got[1, True], got[0, True] + 3.0)


@pytest.mark.parametrize("M,K,N", [(33, 11008, 8192), (64, 6016, 16380), (64, 16352, 5632)])
def test_default_plans_where_the_other_kernel_would_cut_k(hq, oracle, M, K, N):
    test_default_plans(hq, oracle, M, K, N)


@pytest.mark.parametrize("M,K,N,kernel", [(39, 4160, 1176, "direct"), (39, 4160, 1176, "rows64"), (6, 11008, 4096, "block"),
                                          (8, 8192, 8192, "block")])
def test_capture_without_any_workspace(hq, oracle, tunable, M, K, N, kernel):
    """Under capture nothing can be allocated: on a stream that has no workspace the call divides no tile, and replays give the
    eager result's values to the last bits but the order of the sums.  The same for a batch of the 64-row kernel, whose re-ordered
    activations have no place there, and for the block kernel where it would divide K."""
    import torch
    if kernel == "rows64":
        tunable("HQ_Q3_SMALL_BATCH", 0)
        tunable("HQ_Q3_TILES", 9)
    assert kernel_of(M, K, N) == kernel
    codes, scales, zeros, A = oa.make_q3_problem(11, K, N, x_dtype=np.float16, batch=M)
    mat = oracle.q3_pack(codes)
    a, w, s, z = _t(A), _t(mat), _t(scales), _t(zeros)
    out = torch.zeros((M, N), device="cuda:0")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        hq.q3_gemm(a, w, s, z, out=out)
    exact = oracle.q3_gemm(A, mat, scales, zeros, mode=0)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        _check(out.cpu().numpy(), exact)
        eager = hq.q3_gemm(a, w, s, z)
        assert (eager - out).abs().max() <= 1e-5 * eager.abs().max()
