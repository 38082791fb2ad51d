"""Device-side packers and the 4-bit quantiser against the CPU oracle (bit-exact), and
round trips through the matvec / dequant kernels, through the C ABI."""
import numpy as np
import pytest

from tests import oracle_api as oa
from tests.tol import rel_err

pytestmark = pytest.mark.gpu


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


@pytest.mark.parametrize("K,N", [(4096, 1024), (32, 4), (96, 37), (1024, 11008)])
def test_q3_pack_bit_exact_and_round_trip(hq, oracle, K, N):
    import torch
    rng = np.random.default_rng(K + N)
    codes = rng.integers(0, 8, size=(K, N), dtype=np.uint8)
    got = hq.q3_pack(_t(codes))
    torch.cuda.synchronize()
    want = oracle.q3_pack(codes)
    assert np.array_equal(got.cpu().numpy(), want)
    assert np.array_equal(oracle.q3_unpack(got.cpu().numpy(), K), codes)
    if N % 4 == 0:
        x = rng.integers(-8, 9, size=K).astype(np.float32)
        y = hq.q3_matvec(_t(x), got, _t(np.ones(N, np.float32)), _t(np.zeros(N, np.float32)))
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy().astype(np.int64), x.astype(np.int64) @ codes.astype(np.int64))


@pytest.mark.parametrize("K,N,nb", [(1024, 256, 3), (32, 5, 1), (256, 130, 8)])
def test_bcq_pack_bit_exact(hq, oracle, K, N, nb):
    import torch
    rng = np.random.default_rng(K + N + nb)
    signs = (rng.integers(0, 2, size=(K, nb, N)) * 2 - 1).astype(np.int8)
    got = hq.bcq_pack(_t(signs))
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy().view(np.uint32), oracle.bcq_pack(signs))


@pytest.mark.parametrize("table", [0, 1])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("n,blocksize", [(4096 * 64, 64), (1000, 64), (999, 64), (4096, 128), (256, 2), (96, 32)])
def test_quantize_4bit_bit_exact_and_round_trip(hq, oracle, n, blocksize, dtype, table):
    import torch
    rng = np.random.default_rng(n + blocksize + table)
    x = (rng.standard_normal(n) * rng.uniform(0.01, 10)).astype(dtype)
    packed, absmax = hq.quantize_4bit(_t(x), blocksize, table)
    torch.cuda.synchronize()
    wp, wa = oracle.quantize_4bit(x, blocksize, table)
    assert np.array_equal(absmax.cpu().numpy(), wa)
    assert np.array_equal(packed.cpu().numpy(), wp)
    # round trip: dequantise on the GPU, compare with the oracle's dequantisation of the same codes
    deq = hq.dequant_4bit(packed, absmax, n, blocksize, table)
    torch.cuda.synchronize()
    want = oracle.dequant_4bit(wp, wa, n, blocksize, table)
    assert np.array_equal(deq.cpu().numpy().view(np.uint16), want.view(np.uint16))
    # and the round trip error is bounded by half the widest code gap times absmax
    err = np.abs(deq.cpu().numpy().astype(np.float32) - x.astype(np.float32))
    assert np.all(err <= 0.17 * np.repeat(wa, blocksize)[:n] + 1e-3 * np.abs(x.astype(np.float32)))


def test_zero_block_and_midpoint_ties(hq, oracle):
    import torch
    # an all-zero block has absmax 0 and code 7 (the zero entry); values exactly on a midpoint
    # take the lower code
    t = oracle.nf4_table
    mids = ((t[:-1] + t[1:]) * np.float32(0.5)).astype(np.float32)
    x = np.concatenate([np.zeros(64, np.float32), np.array([1.0], np.float32), mids, np.zeros(64 - 16, np.float32)])
    packed, absmax = hq.quantize_4bit(_t(x), 64, 0)
    torch.cuda.synchronize()
    wp, wa = oracle.quantize_4bit(x, 64, 0)
    assert np.array_equal(packed.cpu().numpy(), wp) and np.array_equal(absmax.cpu().numpy(), wa)
    codes = np.stack([wp >> 4, wp & 15], 1).reshape(-1)
    assert (codes[:64] == 7).all() and codes[64] == 15
    assert np.array_equal(codes[65:80], np.arange(15))


@pytest.mark.parametrize("table", [0, 1])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("n,blocksize", [(1, 8), (8, 8), (513, 8), (2047, 16), (511, 512), (2049, 512), (1025, 1024), (6001, 2048),
                                        (4096, 4096), (20003, 4096), (2 ** 24 + 77, 64), (3000, 48)])
def test_quantize_4bit_units(hq, oracle, n, blocksize, dtype, table):
    """Edges of the lane units, of the waves and of blocks longer than a unit row, zero and denormal blocks, NaN and
    infinite values (codes as the comparisons of the definition give them): byte for byte the oracle's."""
    import torch
    rng = np.random.default_rng(n + blocksize)
    x = (rng.standard_normal(n) * 0.3).astype(dtype)
    if 2000 < n < 100000:
        x[5], x[17], x[70], x[n - 1] = np.nan, np.inf, -np.inf, -0.0
        x[100:n // 2] = 0
        x[n // 2:n // 2 + 64] = 1e-40 if dtype == np.float32 else 6e-8
    packed, absmax = hq.quantize_4bit(_t(x), blocksize, table)
    torch.cuda.synchronize()
    wp, wa = oracle.quantize_4bit(x, blocksize, table)
    assert np.array_equal(absmax.cpu().numpy(), wa)
    assert np.array_equal(packed.cpu().numpy(), wp)


@pytest.mark.parametrize("table", [0, 1])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("blocksize", [1024, 2048, 4096])
def test_blocks_shared_by_waves(hq, oracle, blocksize, dtype, table):
    """Blocks that the waves of a workgroup share: the largest magnitude in every wave's part in turn, a block of zeros,
    NaN and infinite elements, and lengths that end in any part of the last block."""
    import torch
    rng = np.random.default_rng(blocksize + table)
    x = rng.standard_normal(17 * blocksize).astype(dtype)
    for b in range(8):  # one peak per eighth of a block
        x[b * blocksize + (2 * b + 1) * blocksize // 16] = 9.0 + b
    x[8 * blocksize:9 * blocksize] = 0
    x[10 * blocksize + 3], x[11 * blocksize - 1] = np.nan, np.inf
    for n in (17 * blocksize, 16 * blocksize + 1, 12 * blocksize + blocksize // 4 + 5, 9 * blocksize + blocksize // 2, blocksize - 8):
        got, amax = hq.quantize_4bit(torch.from_numpy(x[:n]).cuda(), blocksize, table)
        want, wmax = oracle.quantize_4bit(x[:n], blocksize, table)
        assert np.array_equal(got.cpu().numpy(), want) and np.array_equal(amax.cpu().numpy(), wmax), n
