"""The tiled kernels of the batched 3-bit GEMM (many rows): every tile kind, undivided and divided along K, at the edges of
tiles, steps and k-groups, against the oracle row by row."""
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


def _check(y, exact, rows=True):
    # as for the 64-row kernel: the only error is the matrix cores' fp32 accumulation, 1.8e-6 of the RMS - of the row's
    # own, as every row is a sum of its own magnitude (an outlier's products cancel in single results, not in the row)
    for m in range(len(y)) if rows else [slice(None)]:
        if exact[m].any():
            assert rel_err(y[m], exact[m]) <= 5e-3, m
            assert rel_err(y[m], exact[m], FLOOR_F16) <= 1e-4, m
        else:
            assert not y[m].any(), m


@pytest.mark.parametrize("kind,shares", [(0, 1), (0, 2), (0, 5), (1, 1), (1, 2), (1, 3), (2, 1), (2, 2), (2, 8)])
@pytest.mark.parametrize("M,K,N", [(97, 32, 4), (128, 1024, 256), (129, 2080, 260), (193, 1376, 132), (300, 96, 1028),
                                   (98, 4128, 516)])
def test_kinds_and_shares(hq, oracle, tunable, kind, shares, M, K, N):
    codes, scales, zeros, A = oa.make_q3_problem(M + K + N, K, N, x_dtype=np.float16, batch=M)
    A[5] *= np.float16(2.0 ** -10)     # rows of other magnitudes, a zero row, an outlier
    A[7] = 0
    # An outlier at k = 3 of its k-group, whose code lies at bit 5 of its operand: what the matrix instruction cuts off the
    # products next to it is 2^-5 of what it cuts at k = 0, where 1e-4 of such a row's RMS does not hold (the bound that holds
    # at every k, here and in the 64-row kernel: test_outlier_at_any_code).
    A[9, K // 64 * 32 + 3] = np.float16(4096.0)
    mat = oracle.q3_pack(codes)
    tunable("HQ_Q3_TILES", kind + 10 * shares)
    y = hq.q3_gemm(_t(A), _t(mat), _t(scales), _t(zeros))
    again = hq.q3_gemm(_t(A), _t(mat), _t(scales), _t(zeros))
    assert np.array_equal(y.cpu().numpy(), again.cpu().numpy())  # shares are added in a fixed order
    exact = oracle.q3_gemm(A, mat, scales, zeros, mode=0)
    _check(y.cpu().numpy(), exact)


@pytest.mark.parametrize("M,K,N,kind", [(1024, 96, 8196, 0), (1000, 1376, 8452, 0), (97, 416, 66052, 0), (1090, 288, 7684, 0), (512, 1056, 8452, 1),
                                        (300, 2080, 13316, 1)])
def test_columns_beyond_the_last_round(hq, oracle, tunable, M, K, N, kind):
    """Columns cut off for the one-launch kernel: four columns, a tile of 256 and four, 516 behind whole rounds that row tiles do
    not divide, and on top of what is in the output.  Bounds of the tiles."""
    import torch
    from hecbench_amd import _lib
    lib = _lib.load()
    codes, scales, zeros, A = oa.make_q3_problem(M + K + N, K, N, x_dtype=np.float16, batch=M)
    mat = oracle.q3_pack(codes)
    a, w, s, z = _t(A), _t(mat), _t(scales), _t(zeros)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    tunable("HQ_Q3_TILES", 100 + kind)
    y = hq.q3_gemm(a, w, s, z)
    for fn in (lib.hq_q3_matvec, lib.hq_q3_matvec_noalloc):
        on_top = torch.full((M, N), 3.0, device="cuda:0")
        assert fn(a.data_ptr(), 1, w.data_ptr(), s.data_ptr(), z.data_ptr(), on_top.data_ptr(), K, N, M, 1, stream) == 0
        assert torch.allclose(on_top - 3.0, y, rtol=0, atol=2.0 ** -22 * float(y.abs().max() + 3))  # one rounding of the sum and one back
    row_tiles = -(-M // (128 >> kind))
    cut = 256 // row_tiles * 256 if N // 256 * row_tiles < 512 else 512 // row_tiles * 256
    cols = np.r_[0:40, cut - 40:min(cut + 40, N), N - 4:N]
    _check(y[:, cols].cpu().numpy(), oracle.q3_gemm(A, np.ascontiguousarray(mat[:, cols]), scales[cols], zeros[cols], mode=0), rows=False)


@pytest.mark.parametrize("M,K,N", [(40, 2080, 516), (64, 8192, 132), (129, 2080, 260), (300, 1024, 1028)])
@pytest.mark.parametrize("k,pos", [(0, 0), (19, 0), (29, 0), (14, 1), (3, 5)])
@pytest.mark.parametrize("amp", [64.0, 4096.0, -60000.0])
def test_outlier_at_any_code(hq, oracle, tunable, M, K, N, k, pos, amp):
    """What an outlier costs its row, in the 64-row kernel and in the tiles.  A code at bit pos of its operand is a subnormal
    number: the matrix instruction aligns its product as if the code were 2^(10 - pos), and cuts the other fifteen products and
    the sum so far below the 24th bit of that: 17 cuts of at most 2^(10 - pos) * 2^-24 of the outlier's power of two, times the
    column's scale (seen: a quarter of that).  The rest of the row: 1e-5 of its RMS."""
    tunable("HQ_Q3_SMALL_BATCH", 0)
    tunable("HQ_Q3_TILES", 9)
    assert kernel_of(M, K, N) == ("rows64" if M <= 64 else "tiles")
    codes, scales, zeros, A = oa.make_q3_problem(M + K + N, K, N, x_dtype=np.float16, batch=M)
    A[9, K // 64 * 32 + k] = np.float16(amp)
    mat = oracle.q3_pack(codes)
    y = hq.q3_gemm(_t(A), _t(mat), _t(scales), _t(zeros)).cpu().numpy()[9].astype(np.float64)
    exact = oracle.q3_gemm(A[9:10], mat, scales, zeros, mode=0)[0]
    cut = 2.0 ** (np.floor(np.log2(abs(amp))) + 10 - pos - 24)
    assert np.all(np.abs(y - exact) <= 17 * cut * scales + 1e-5 * np.sqrt(np.mean(exact ** 2)))


@pytest.mark.parametrize("M,K,N,default", [(100, 4096, 4096, 0), (700, 512, 3000, 0), (1030, 16416, 8, 0), (70, 256, 8200, 0),
                                           (100, 6112, 17848, 1), (1100, 5376, 4468, 1), (72, 576, 49700, 1), (1100, 16384, 4100, 1),
                                           (163, 8416, 10948, 1)])
def test_default_plans(hq, oracle, tunable, M, K, N, default):
    """The library's own choice of the tiles' plan: few tiles, several full rounds with a rest, several passes over the rows,
    65 ... 96 rows of a wide matrix; problems that the tiles serve by default, and smaller ones that are the one-launch kernel's.
    Rows of one magnitude: the RMS of the whole result is the measure, as in the 64-row kernel's tests (a few columns of one row
    are no sample of it)."""
    if not default:
        tunable("HQ_Q3_TILES", 9)
    assert kernel_of(M, K, N) == "tiles"
    codes, scales, zeros, A = oa.make_q3_problem(M + K, K, N, x_dtype=np.float16, batch=M)
    mat = oracle.q3_pack(codes)
    y = hq.q3_gemm(_t(A), _t(mat), _t(scales), _t(zeros)).cpu().numpy()
    cols = np.unique(np.concatenate([np.arange(0, min(N, 70)), np.arange(max(0, N - 70), N)]))
    _check(y[:, cols], oracle.q3_gemm(A, np.ascontiguousarray(mat[:, cols]), scales[cols], zeros[cols], mode=0), rows=False)


def test_accumulate_and_the_call_that_allocates_nothing(hq, oracle, tunable):
    import torch
    from hecbench_amd import _lib
    lib = _lib.load()
    M, K, N = 200, 1024, 516
    tunable("HQ_Q3_TILES", 9)
    assert kernel_of(M, K, N) == "tiles"
    codes, scales, zeros, A = oa.make_q3_problem(3, K, N, x_dtype=np.float16, batch=M)
    mat = oracle.q3_pack(codes)
    exact = oracle.q3_gemm(A, mat, scales, zeros, mode=0)
    a, w, s, z = _t(A), _t(mat), _t(scales), _t(zeros)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for fn in (lib.hq_q3_matvec, lib.hq_q3_matvec_noalloc):
        y = torch.full((M, N), 3.0, device="cuda:0")
        assert fn(a.data_ptr(), 1, w.data_ptr(), s.data_ptr(), z.data_ptr(), y.data_ptr(), K, N, M, 1, stream) == 0
        torch.cuda.synchronize()
        _check(y.cpu().numpy() - 3.0, exact)


def test_capture_with_the_workspace_of_a_smaller_call(hq, oracle, tunable):
    """Under capture nothing can be allocated: where the stream's workspace holds what 64 rows need and not what all do, the
    call goes 64 rows at a time, and gives the bits of such calls."""
    tunable("HQ_Q3_TILES", 9)  # the workspace of the 64-row kernel, which this matrix is too small to take by itself
    tunable("HQ_Q3_SMALL_BATCH", 0)
    import torch
    M, K, N = 1000, 4096, 16512
    codes, scales, zeros, A = oa.make_q3_problem(11, K, N, x_dtype=np.float16, batch=M)
    mat = oracle.q3_pack(codes)
    a, w, s, z = _t(A), _t(mat), _t(scales), _t(zeros)
    out = torch.zeros((M, N), device="cuda:0")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        hq.q3_gemm(a[:32].contiguous(), w, s, z)
        first, last = hq.q3_gemm(a[:64].contiguous(), w, s, z), hq.q3_gemm(a[960:].contiguous(), w, s, z)
    assert kernel_of(64, K, N) == "rows64" and kernel_of(M, K, N) == "tiles"
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        hq.q3_gemm(a, w, s, z, out=out)
    cols = np.concatenate([np.arange(0, 40), np.arange(N - 40, N)])
    exact = oracle.q3_gemm(A, np.ascontiguousarray(mat[:, cols]), scales[cols], zeros[cols], mode=0)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        _check(out.cpu().numpy()[:, cols], exact, rows=False)
        assert torch.equal(out[:64], first) and torch.equal(out[960:], last)
