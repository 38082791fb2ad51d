"""hq_q3_matvec_noalloc, the entry point that allocates nothing: through the C ABI, bit-identical with
hq_q3_matvec (same kernels, scratch in a fixed device array instead of the stream's workspace) on two
calls in a row, the second with a smaller input, for the split-K matvec and for the batched path."""
import ctypes

import numpy as np
import pytest

from tests import oracle_api as oa
from tests.q3_kernel import kernel_of
from tests.tol import rel_err

pytestmark = pytest.mark.gpu


def _problem(oracle, seed, K, N, M):
    import torch
    dev = torch.device("cuda:0")
    codes, scales, zeros, x = oa.make_q3_problem(seed, K, N)
    mat = oracle.q3_pack(codes)
    A = np.random.default_rng(seed).standard_normal((M, K)).astype(np.float16)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    return dict(K=K, N=N, M=M, x=t(x), mat=t(mat), s=t(scales), z=t(zeros), A=t(A),
                host=(x, mat, scales, zeros, A))


def _call(fn, p, batch):
    import torch
    vp = lambda t: ctypes.c_void_p(t.data_ptr())
    act = p["A"] if batch > 1 else p["x"]
    y = torch.full((batch, p["N"]), float("nan"), device="cuda:0")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = fn(vp(act), 1 if batch > 1 else 0, vp(p["mat"]), vp(p["s"]), vp(p["z"]), vp(y), p["K"], p["N"], batch, 0, stream)
    assert rc == 0, rc
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.fixture(params=["default", "pre-pass"])
def pre_pass(request, tunable):
    """Once as the library chooses, and once with the kernels behind a pre-pass in place of the one-launch kernel."""
    if request.param == "pre-pass":
        tunable("HQ_Q3_TILES", 9)
    return request.param == "pre-pass"


def test_noalloc_matches_workspace_path(hq, oracle, pre_pass):
    from hecbench_amd import _lib
    lib = _lib.load()
    # 32 and 8 column tiles: far fewer than half the compute units, so both calls split K across
    # workgroups and use the partial sums and the arrival counters
    big = _problem(oracle, 301, 8192, 2048, 70)
    small = _problem(oracle, 302, 2048, 512, 66)
    for p in (big, small):                      # two calls in a row, the second with a smaller input
        # the matvec (narrow tiles), the small-batch kernel with one workgroup per tile and with two, three and
        # ten row blocks, the one-launch kernel, the GEMM (64 rows and the rest)
        for batch in (1, 2, 6, 11, 40, p["M"]):
            want = _call(lib.hq_q3_matvec, p, batch)
            got = _call(lib.hq_q3_matvec_noalloc, p, batch)
            assert np.array_equal(got, want), (p["K"], p["N"], batch)
            x, mat, scales, zeros, A = p["host"]
            if batch == 1:
                assert rel_err(got[0], oracle.q3_matvec_f64(x, mat, scales, zeros)) <= 1e-4
            else:
                assert rel_err(got, oracle.q3_gemm(A[:batch], mat, scales, zeros, mode=0)) <= 5e-3
    # and again in the other order: the array keeps the last call's contents
    for p in (small, big, small):
        assert np.array_equal(_call(lib.hq_q3_matvec_noalloc, p, 1), _call(lib.hq_q3_matvec, p, 1))


@pytest.mark.parametrize("K,N,M", [(4096, 11008, 65), (8192, 4096, 72), (1024, 2048, 97), (4096, 4096, 128), (8192, 28672, 200),
                                   (16384, 6148, 300), (512, 260, 9000), (2080, 1028, 1100), (4160, 28672, 1030)])
def test_many_rows_give_the_bits_of_the_workspace_path(hq, oracle, pre_pass, K, N, M):
    """Batches that hq_q3_matvec takes in tiles (and one that it takes 64 rows at a time): whole rounds, divided rests, several
    passes over the rows, the longest K; the smaller of them on the one-launch kernel by default."""
    import torch
    from hecbench_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device="cuda:0").manual_seed(M)
    dev = "cuda:0"
    A = torch.empty((M, K), dtype=torch.float16, device=dev).normal_(generator=g)
    w = torch.randint(-2 ** 31, 2 ** 31, (3 * K // 32, N), dtype=torch.int32, device=dev, generator=g)
    s = torch.rand(N, device=dev, generator=g).mul_(0.01).add_(0.002)
    p = dict(K=K, N=N, M=M, x=None, mat=w, s=s, z=s * 3, A=A)
    want = _call(lib.hq_q3_matvec, p, M)
    assert np.isfinite(want).all()
    for _ in range(2):
        assert np.array_equal(_call(lib.hq_q3_matvec_noalloc, p, M), want)


class _Scratch(ctypes.Structure):  # HqQ3Scratch of csrc/hq_internal.h
    _fields_ = [("partial", ctypes.c_void_p), ("partial_floats", ctypes.c_size_t), ("rows", ctypes.c_void_p),
                ("counters", ctypes.c_void_p), ("ncounters", ctypes.c_size_t), ("sums", ctypes.c_void_p),
                ("sums_floats", ctypes.c_size_t), ("tiles", ctypes.c_void_p), ("tiles_floats", ctypes.c_size_t)]


@pytest.mark.parametrize("K,N,M", [(4096, 516, 40), (8192, 516, 20), (8192, 2048, 64), (4096, 4096, 70), (8192, 512, 66),
                                   (4096, 1028, 130)])
def test_batched_call_after_one_that_was_cut_short(hq, oracle, tunable, pre_pass, K, N, M):
    """A call that does not finish leaves its arrival counters part of the way up.  The next call must not count on from
    there: the library's own launch function with a scratch of the test's, counters as such a call leaves them; one-launch kernel,
    64-row kernel (K split, sums by the last workgroup and, eight splits of 64 rows, by the second kernel) and tiles."""
    import torch
    from hecbench_amd import _lib
    if pre_pass:
        tunable("HQ_Q3_SMALL_BATCH", 0)
        assert kernel_of(M, K, N) == ("tiles" if M > 96 else "rows64")
    launch = getattr(_lib.load(), "_Z17hq_q3_gemm_launchPKvPKiPKfS4_PfiiijP12ihipStream_tPK11HqQ3Scratch")
    p = _problem(oracle, 303, K, N, M)
    dev = "cuda:0"
    partial = torch.zeros(1 << 19, device=dev)
    rows = torch.zeros(256, device=dev)
    sums = torch.zeros(1 << 21, device=dev)
    tiles = torch.zeros(1 << 22, device=dev)
    counters = torch.full((4096,), 100, dtype=torch.int32, device=dev)  # of a call with more parts
    vp = lambda t: ctypes.c_void_p(t.data_ptr())
    s = _Scratch(partial.data_ptr(), partial.numel(), rows.data_ptr(), counters.data_ptr(), counters.numel(), sums.data_ptr(),
                 sums.numel(), tiles.data_ptr(), tiles.numel())
    want = oracle.q3_gemm(p["host"][4], *p["host"][1:4], mode=0)
    for _ in range(2):
        y = torch.full((M, N), float("nan"), device=dev)
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert launch(vp(p["A"]), vp(p["mat"]), vp(p["s"]), vp(p["z"]), vp(y), K, N, M, 0, stream, ctypes.byref(s)) == 0
        torch.cuda.synchronize()
        assert rel_err(y.cpu().numpy(), want) <= 5e-3


def test_noalloc_rejects_beyond_its_limits(hq):
    import torch
    from hecbench_amd import _lib
    lib = _lib.load()
    dev = torch.device("cuda:0")
    K, N, M = 32768, 64, 65                     # the batched GEMM's activations would need 4 MiB
    A = torch.zeros((M, K), dtype=torch.float16, device=dev)
    w = torch.zeros((3 * K // 32, N), dtype=torch.int32, device=dev)
    s = torch.zeros(N, device=dev)
    y = torch.zeros((M, N), device=dev)
    vp = lambda t: ctypes.c_void_p(t.data_ptr())
    assert lib.hq_q3_matvec_noalloc(vp(A), 1, vp(w), vp(s), vp(s), vp(y), K, N, M, 0, None) == -6
    assert lib.hq_q3_matvec(vp(A), 1, vp(w), vp(s), vp(s), vp(y), K, N, M, 0, None) == 0
    torch.cuda.synchronize()
    assert lib.hq_q3_matvec_noalloc(None, 0, None, None, None, None, 64, 8, 1, 0, None) == -1
