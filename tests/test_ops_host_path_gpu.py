"""The native host path of the operators: results come back as the caller's own tensor or a new one of the right
shape and type, library errors as HqError, and calls go to the current stream."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _q3(dev, K=512, N=128):
    w = torch.randint(-2**31, 2**31, (3 * K // 32, N), dtype=torch.int32, device=dev)
    return torch.randn(K, device=dev), w, torch.rand(N, device=dev), torch.rand(N, device=dev)


def test_given_and_new_results(hq):
    dev = torch.device("cuda:0")
    x, w, s, z = _q3(dev)
    out = torch.empty(128, device=dev)
    assert hq.q3_matvec(x, w, s, z, out=out) is out
    y = hq.q3_matvec(x, w, s, z)
    assert y.shape == (128,) and y.dtype == torch.float32 and y.device == dev and torch.equal(y, out)
    q, sc, azp = hq.dynamic_scaled_int8_quant(torch.randn(3, 40, device=dev), with_azp=True)
    assert (q.shape, q.dtype, sc.dtype, azp.dtype) == ((3, 40), torch.int8, torch.float32, torch.int32)
    assert hq.dynamic_scaled_int8_quant(torch.randn(3, 40, device=dev))[2] is None
    h = torch.randn(2, 3, 32, device=dev, dtype=torch.bfloat16)
    assert hq.mxfp4_qdq(h).shape == h.shape and hq.mxfp4_qdq(h).dtype == h.dtype


def test_library_errors(hq):
    dev = torch.device("cuda:0")
    x, w, s, z = _q3(dev)
    with pytest.raises(hq.HqError, match="hq_q3_matvec: hq: pointer not aligned"):
        hq.q3_matvec(torch.randn(513, device=dev)[1:], w, s, z)
    with pytest.raises(hq.HqError, match="unknown dtype / table"):
        hq.quantize_4bit(x, 64, table=9)
    with pytest.raises(ValueError, match="device tensors only"):
        hq.q3_matvec(x, w, s, torch.rand(128))


def test_current_stream(hq):
    """A call inside a stream context runs behind that stream's earlier work: the operand written there is seen."""
    dev = torch.device("cuda:0")
    x, w, s, z = _q3(dev, 4096, 4096)
    want = hq.q3_matvec(x, w, s, z)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        late = torch.zeros_like(x)
        for _ in range(50):
            late.add_(0.0)
        late.copy_(x)
        y = hq.q3_matvec(late, w, s, z)
    side.synchronize()
    assert torch.equal(y, want)


def test_integers_beyond_32_bits(hq):
    """A zero point counts by its low 32 bits; a code book's row bound beyond them holds for every row."""
    dev = torch.device("cuda:0")
    x = torch.randn(4, 64, device=dev)
    assert torch.equal(hq.static_scaled_int8_quant(x, 0.05, 2 ** 32 + 7), hq.static_scaled_int8_quant(x, 0.05, 7))
    assert torch.equal(hq.static_scaled_int8_quant(x, 0.05, -2 ** 63 - 3), hq.static_scaled_int8_quant(x, 0.05, -3))
    codes = torch.randint(-2 ** 15, 2 ** 15, (16, 8), dtype=torch.int16, device=dev)
    v, cb = torch.randn(64, device=dev).half(), torch.randn(2, 65536, 8, device=dev).half()
    assert torch.equal(hq.code1x16_matvec(codes, v, cb, (2 ** 32 + 5, 0, 0, 0), 65536),
                       hq.code1x16_matvec(codes, v, cb, (16, 0, 0, 0), 65536))
    assert torch.equal(hq.code1x16_matvec(codes, v, cb, (5, 2 ** 40, 0, 0), 65536),
                       hq.code1x16_matvec(codes, v, cb, (5, 16, 0, 0), 65536))
