"""Guard on the choice between the two walks over K of hq_lut_gemv (several quads per wave and round, or one quad and a workgroup per
round): on problems where one of them takes a tenth longer and more, the library's own choice is the faster one."""
import ctypes

import pytest

from tests.test_q3_policy_gpu import _time

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N,nb,group", [(13312, 192, 5, 32), (5888, 5562, 4, 32), (17664, 1814, 6, 32), (4480, 26432, 2, 64),
                                          (14208, 10688, 2, 32), (8320, 384, 3, 128), (8704, 256, 6, 128), (11392, 1778, 2, 128),
                                          (512, 11964, 3, 64), (512, 23848, 2, 32), (256, 10475, 4, 64), (512, 40000, 3, 32)])
def test_own_choice_is_the_faster_walk(hq, tunable, K, N, nb, group):
    import torch
    from hecbench_amd import _lib
    lib = _lib.load()
    g = torch.Generator(device="cuda:0")
    g.manual_seed(K + N)
    nbuf = min(32, int(560e6 // (K * N * nb // 8)) + 1)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (nbuf, K // 32, nb, N), dtype=torch.int32, device="cuda:0", generator=g)
    alpha = torch.rand(nbuf, K // group, nb, N, device="cuda:0", generator=g).mul_(0.02).half()
    x = torch.randn(K, device="cuda:0", generator=g).half()
    y = torch.empty(N, dtype=torch.float16, device="cuda:0")
    vp = lambda t: ctypes.c_void_p(t.data_ptr())
    pw, pa, px, py = [vp(w) for w in bW], [vp(a) for a in alpha], vp(x), vp(y)

    def call(i):
        assert lib.hq_lut_gemv(pw[i], pa[i], None, px, py, K, N, nb, group, None) == 0

    torch.cuda.synchronize()
    _time(lib, call, nbuf)
    own = _time(lib, call, nbuf)
    forced = []
    for knob in (0, 1):
        tunable("HQ_LUT_FINE", knob)
        forced.append(_time(lib, call, nbuf))
    print(f"{K}x{N} {nb} planes group {group}: own {own:.2f} us, several quads {forced[0]:.2f}, one {forced[1]:.2f}")
    assert own <= 1.08 * min(forced)
