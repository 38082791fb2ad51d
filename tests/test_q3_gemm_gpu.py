"""Parity of the batched GPTQ 3-bit GEMM (hq_q3_matvec with batch_M > 1) with the
CPU oracle, through the C ABI.  The reference has no batched kernel: the oracle is
the matvec formula applied row by row (parity unpinned by the reference)."""
import numpy as np
import pytest

from tests import oracle_api as oa
from tests.q3_kernel import kernel_of
from tests.tol import FLOOR_F16, TOL_F16_ACC, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _the_gemm_kernel_only(tunable):
    """Most problems of these sizes would take the matvec's four-rows-per-workgroup kernel (tests/test_q3_small_batch_gpu.py
    covers that) or the one-launch kernel (tests/test_q3_direct_gpu.py): this file is about the MFMA GEMM behind a pre-pass, so
    every batch takes it, up to 64 rows on the 64-row kernel, more on the tiles (or 64 at a time)."""
    tunable("HQ_Q3_SMALL_BATCH", 0)
    tunable("HQ_Q3_TILES", 9)


def _run(hq, A, mat, scales, zeros):
    import torch
    M, K, N = len(A), A.shape[1], mat.shape[1]
    assert kernel_of(M, K, N) in (("rows64",) if M <= 64 else ("rows64", "tiles")), (M, K, N)
    dev = torch.device("cuda:0")
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    y = hq.q3_gemm(t(A), t(mat), t(scales), t(zeros))
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("M,K,N,seed", [(16, 256, 256, 1), (64, 1024, 512, 2), (33, 512, 132, 3), (100, 512, 260, 4),
                                        (17, 96, 8, 5), (64, 2048, 1000, 6)])
def test_small_shapes_vs_oracle(hq, oracle, M, K, N, seed):
    codes, scales, zeros, A = oa.make_q3_problem(seed, K, N, x_dtype=np.float16, batch=M)
    mat = oracle.q3_pack(codes)
    y = _run(hq, A, mat, scales, zeros)
    exact = oracle.q3_gemm(A, mat, scales, zeros, mode=0)
    w16 = oracle.q3_gemm(A, mat, scales, zeros, mode=1)
    # contract: within 2e-2 of the dequantise-to-fp16 formulation ...
    assert rel_err(y, w16, FLOOR_F16) <= TOL_F16_ACC
    # ... and in fact close to the exact result: the only error source is the matrix cores' truncating fp32
    # accumulation (1.8e-6 of the RMS; up to 1.5e-5 in single results, 1.5e-5 / 1% floor = 1.5e-3)
    assert rel_err(y, exact) <= 5e-3
    assert rel_err(y, exact, FLOOR_F16) <= 1e-4


@pytest.mark.parametrize("M,K,N,seed", [(16, 4096, 512, 11), (64, 8192, 260, 12), (40, 14336, 1024, 13), (13, 2048, 128, 14),
                                        (100, 4096, 4096, 15)])
def test_small_n_splits_k(hq, oracle, M, K, N, seed):
    """Few column tiles: K is cut into ranges (one workgroup each) whose raw sums a second kernel adds up."""
    codes, scales, zeros, A = oa.make_q3_problem(seed, K, N, x_dtype=np.float16, batch=M)
    mat = oracle.q3_pack(codes)
    y = _run(hq, A, mat, scales, zeros)
    assert np.array_equal(y, _run(hq, A, mat, scales, zeros))      # the sums are added in a fixed order
    cols = np.unique(np.concatenate([np.arange(0, min(N, 130)), np.arange(max(0, N - 130), N)]))
    exact = oracle.q3_gemm(A, np.ascontiguousarray(mat[:, cols]), scales[cols], zeros[cols], mode=0)
    assert rel_err(y[:, cols], exact) <= 5e-3
    assert rel_err(y[:, cols], exact, FLOOR_F16) <= 1e-4


@pytest.mark.parametrize("M,K,N", [(23, 1952, 12980), (24, 16384, 4096), (33, 12288, 5000), (64, 4096, 11008), (20, 16384, 6148)])
def test_split_sums_by_the_last_workgroup(hq, oracle, M, K, N):
    """Two to eight shares per tile, one and two row blocks, a last tile of any width."""
    import torch
    codes, scales, zeros, A = oa.make_q3_problem(M + N, K, N, x_dtype=np.float16, batch=M)
    mat = oracle.q3_pack(codes)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    args = t(A), t(mat), t(scales), t(zeros)
    assert kernel_of(M, K, N) == "rows64"
    y = hq.q3_gemm(*args)
    for _ in range(3):
        assert torch.equal(y, hq.q3_gemm(*args))
    cols = np.unique(np.concatenate([np.arange(0, 130), np.arange(N - 130, N)]))
    exact = oracle.q3_gemm(A, np.ascontiguousarray(mat[:, cols]), scales[cols], zeros[cols], mode=0)
    assert rel_err(y.cpu().numpy()[:, cols], exact, FLOOR_F16) <= 1e-4


@pytest.mark.parametrize("M,K,N", [(40, 8192, 1000), (64, 4096, 132), (70, 4096, 2048), (128, 8192, 516), (300, 4096, 260)])
def test_error_has_no_offset(hq, oracle, M, K, N):
    """The matrix instruction cuts its sums towards minus infinity.  With every product entering with its own sign that was an
    offset of all results, 9e-6 (K=4096) and 1.3e-5 (K=8192) of them in 2-norm, and grew with K; with the cuts of two halves of
    opposite sign cancelling, what is left is their scatter, 1.8e-6 whatever K.  64-row kernel and tiles, K whole and split."""
    codes, scales, zeros, A = oa.make_q3_problem(M + N, K, N, x_dtype=np.float16, batch=M)
    mat = oracle.q3_pack(codes)
    y = _run(hq, A, mat, scales, zeros).astype(np.float64)
    exact = oracle.q3_gemm(A, mat, scales, zeros, mode=0)
    err = (y - exact) / scales           # in units of the raw sums, as the offset is
    assert np.linalg.norm(y - exact) <= 4e-6 * np.linalg.norm(exact)
    assert abs(err.mean()) <= 0.25 * np.sqrt(np.mean(err ** 2))


@pytest.mark.parametrize("scale_exp", [-16, -12, -8, 0, 4])
def test_dynamic_range(hq, oracle, scale_exp):
    """Accuracy must not depend on the magnitude of the activations: whole problem scaled by a power of
    two (down to where fp16 inputs are subnormal), rows of very different magnitude in one batch, an
    all-zero row and a row with one large outlier.  Every row is held to the bound the N(0,1) cases meet,
    measured against that row's own RMS."""
    M, K, N = 40, 2048, 260
    codes, scales, zeros, A = oa.make_q3_problem(70 + scale_exp, K, N, x_dtype=np.float16, batch=M)
    rng = np.random.default_rng(7)
    A = A.astype(np.float32) * np.float32(2.0 ** scale_exp)
    A[3] = 0.0                                            # an all-zero row
    A[5] *= np.float32(2.0 ** -6)                         # rows of other magnitudes in the same batch
    A[6] *= np.float32(2.0 ** 5)
    A[7, 100] = np.float32(2.0 ** min(15, scale_exp + 12))   # one large outlier (4096 sigma) in a row
    A[8] = rng.standard_normal(K).astype(np.float32) * np.float32(2.0 ** scale_exp) * \
        np.exp2(rng.integers(-8, 1, K)).astype(np.float32)    # magnitudes spread over 2^8 inside a row
    A = A.astype(np.float16)
    mat = oracle.q3_pack(codes)
    y = _run(hq, A, mat, scales, zeros)
    exact = oracle.q3_gemm(A, mat, scales, zeros, mode=0)
    assert np.all(y[3] == 0.0)
    for m in range(M):
        if m == 3:
            continue
        assert rel_err(y[m], exact[m]) <= 5e-3, (scale_exp, m)
        assert rel_err(y[m], exact[m], FLOOR_F16) <= 1e-4, (scale_exp, m)
    # a row of the batch equals the batch-1 matvec on that row
    import torch
    dev = torch.device("cuda:0")
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    for m in (0, 5, 7):
        yv = hq.q3_matvec(t(A[m]), t(mat), t(scales), t(zeros)).cpu().numpy()
        assert rel_err(y[m], yv) <= 5e-3, (scale_exp, m)


@pytest.mark.parametrize("M,K,N", [(40, 16384, 8192), (48, 24576, 4096)])
def test_divided_by_default(hq, oracle, tunable, M, K, N):
    """Without any knob: 33 to 64 rows of 9e7 weights and more whose column tiles leave compute units idle; four shares of K
    summed by the last workgroup, eight by the kernel behind."""
    import torch
    from hecbench_amd import _lib
    for knob in (b"HQ_Q3_SMALL_BATCH", b"HQ_Q3_TILES"):
        assert _lib.load().hq_set_tunable(knob, 0, 1) == 0
    assert kernel_of(M, K, N) == "rows64"
    g = torch.Generator(device="cuda:0").manual_seed(K)
    mat = torch.randint(-2 ** 31, 2 ** 31, (3 * K // 32, N), dtype=torch.int32, device="cuda:0", generator=g)
    scales = torch.rand(N, device="cuda:0", generator=g).mul_(0.01).add_(0.002)
    A = torch.empty((M, K), dtype=torch.float16, device="cuda:0").normal_(generator=g)
    y = hq.q3_gemm(A, mat, scales, scales * 3)
    assert torch.equal(y, hq.q3_gemm(A, mat, scales, scales * 3))
    cols = np.unique(np.concatenate([np.arange(0, 68), np.arange(N // 2, N // 2 + 8), np.arange(N - 68, N)]))
    sc = scales.cpu().numpy()[cols]
    exact = oracle.q3_gemm(A.cpu().numpy(), np.ascontiguousarray(mat.cpu().numpy()[:, cols]), sc, (scales * 3).cpu().numpy()[cols], mode=0)
    assert rel_err(y.cpu().numpy()[:, cols], exact, FLOOR_F16) <= 1e-4


def test_config4_sampled_columns(hq, oracle):
    """M=64, K=8192, N=28672: all outputs computed on the GPU, 384 sampled columns checked."""
    M, K, N = 64, 8192, 28672
    rng = np.random.default_rng(44)
    mat = rng.integers(-2 ** 31, 2 ** 31, size=(3 * K // 32, N), dtype=np.int64).astype(np.int32)
    scales = rng.uniform(0.005, 0.02, size=N).astype(np.float32)
    zeros = (scales * rng.integers(3, 5, size=N)).astype(np.float32)
    A = rng.standard_normal((M, K)).astype(np.float16)
    y = _run(hq, A, mat, scales, zeros)
    cols = np.unique(np.concatenate([np.arange(0, 132), np.arange(N - 132, N), rng.integers(0, N, 120)]))
    sub = np.ascontiguousarray(mat[:, cols])
    exact = oracle.q3_gemm(A, sub, scales[cols], zeros[cols], mode=0)
    assert rel_err(y[:, cols], exact) <= 5e-3
    assert rel_err(y[:, cols], exact, FLOOR_F16) <= 1e-4
    # every row of the batch equals the batch-1 matvec on that row (same library, other kernel)
    import torch
    dev = torch.device("cuda:0")
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    dm, ds, dz = t(mat), t(scales), t(zeros)
    for m in (0, 31, 63):
        yv = hq.q3_matvec(t(A[m]), dm, ds, dz)
        torch.cuda.synchronize()
        assert rel_err(y[m], yv.cpu().numpy()) <= 5e-3


def test_batch_needs_fp16(hq):
    import torch
    dev = torch.device("cuda:0")
    from hecbench_amd import _lib
    A = torch.zeros((16, 64), device=dev)
    w = torch.zeros((6, 8), dtype=torch.int32, device=dev)
    s = torch.zeros(8, device=dev)
    y = torch.zeros((16, 8), device=dev)
    rc = _lib.load().hq_q3_matvec(A.data_ptr(), 0, w.data_ptr(), s.data_ptr(), s.data_ptr(), y.data_ptr(), 64, 8, 16, 0, None)
    assert rc == -3
