"""A K divided among up to eight workgroups: their sums meet two and two by exchange.  The same bits as through partial sums and a
count (formal fences, and the entry point that allocates nothing), on every call: the slots are empty again after each."""
import ctypes

import numpy as np
import pytest

from tests import oracle_api as oa
from tests.tol import FLOOR_F16, rel_err

pytestmark = pytest.mark.gpu


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


@pytest.mark.parametrize("M", [1, 2, 4, 7])
@pytest.mark.parametrize("shares,N", [(2, 4), (2, 1028), (3, 260), (4, 196), (5, 68), (6, 4100), (7, 132), (8, 36), (9, 100)])
def test_shares_meet(oracle, tunable, shares, N, M):
    import torch
    from hecbench_amd import _lib
    lib = _lib.load()
    K = 4096 * (shares - 1) + (32 if shares % 2 else 2080)
    codes, scales, zeros, x = oa.make_q3_problem(shares * 100 + N + M, K, N, x_dtype=np.float16, batch=M)
    mat = oracle.q3_pack(codes)
    dx, dm, ds, dz = _t(x), _t(mat), _t(scales), _t(zeros)
    y0 = torch.linspace(-1.0, 1.0, M * N, device="cuda:0").reshape(M, N)
    vp = lambda t: ctypes.c_void_p(t.data_ptr())

    def call(flags=0, fn=lib.hq_q3_matvec):
        y = y0.clone() if flags else torch.full((M, N), 7.0, device="cuda:0")
        assert fn(vp(dx), 1, vp(dm), vp(ds), vp(dz), vp(y), K, N, M, flags, None) == 0
        torch.cuda.synchronize()
        return y

    y = call()
    rows = oracle.q3_gemm(x, mat, scales, zeros, mode=0) if M > 1 else oracle.q3_matvec_f64(x, mat, scales, zeros)
    assert rel_err(y.cpu().numpy().reshape(np.shape(rows)), rows, FLOOR_F16) <= 1e-3
    for _ in range(3):
        assert torch.equal(call(), y)
        assert torch.equal(call(1), y0 + y)  # accumulated: one addition to the finished sum
    assert torch.equal(call(fn=lib.hq_q3_matvec_noalloc), y)
    tunable("HQ_SPLITK_FENCES", 1)
    assert torch.equal(call(), y)


def test_a_nan_is_not_an_empty_slot(hq, oracle):
    """Every sum NaN, whatever its bits: the call after it finds the slots empty."""
    K, N = 8192, 512
    codes, scales, zeros, x = oa.make_q3_problem(5, K, N)
    mat = oracle.q3_pack(codes)
    bad = x.copy()
    bad[[0, K - 1]] = np.array([0xffffffff, 0x7f800001], np.uint32).view(np.float32)
    dm, ds, dz = _t(mat), _t(scales), _t(zeros)
    y = hq.q3_matvec(_t(x), dm, ds, dz)
    assert bool(hq.q3_matvec(_t(bad), dm, ds, dz).isnan().all())
    assert bool((hq.q3_matvec(_t(x), dm, ds, dz) == y).all())
