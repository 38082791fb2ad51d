"""Operator-level wrappers: same names, argument meaning and error behaviour as
the reference launch wrappers, over the C ABI.  No arithmetic happens here and no checks: the native host
path behind each of them (csrc/pyops.cpp) checks dtype, element count, contiguity and device of every tensor
against the problem sizes (the C ABI sees raw pointers and cannot), allocates the result the caller did not pass
and makes one library call on the current stream."""
import ctypes

import torch

from . import _lib

NF4 = 0
FP4 = 1
_native = _lib.native_ops()


def init():
    _lib.check(_lib.load().hq_init(), "hq_init")


def device_info():
    lib = _lib.load()
    v = [ctypes.c_int() for _ in range(5)]
    name = ctypes.create_string_buffer(256)
    _lib.check(lib.hq_device_info(*[ctypes.byref(x) for x in v], name, 256), "hq_device_info")
    return {"compute_units": v[0].value, "wavefront_size": v[1].value, "lds_bytes_per_cu": v[2].value,
            "memory_clock_khz": v[3].value, "memory_bus_bits": v[4].value, "name": name.value.decode()}


def q3_matvec(x, qweight, scales, zeros, out=None, accumulate=False):
    """y[n] = sum_k x[k]*(scales[n]*q[k][n] - zeros[n]); x fp32 or fp16 [K]."""
    return _native.q3_matvec(x, qweight, scales, zeros, out, accumulate)


def vecquant3matmul(vec, mat, mul, scales, zeros, height=None, width=None):
    """Reference signature (src/quant3MatMul-hip/kernels.h:171-190): mul += vec @ W."""
    # view(-1) never copies: a non-contiguous mul raises instead of losing the "mul +=" result in a temporary
    q3_matvec(vec.reshape(-1), mat, scales, zeros, out=_flat_inplace(mul, "mul"), accumulate=True)


def _flat_inplace(t, name):
    if not isinstance(t, torch.Tensor) or not t.is_contiguous():
        raise ValueError(f"{name} must be a contiguous tensor (it is updated in place)")
    return t.view(-1)


def vecquant3matmul_faster(vec, mat, mul, scales, zeros, height=None, width=None):
    """Reference signature (src/quant3MatMul-hip/kernels.h:193-217): fp16 vec, mul += vec @ W."""
    if vec.dtype != torch.float16:
        raise ValueError("vecquant3matmul_faster takes an fp16 vector")
    q3_matvec(vec.reshape(-1), mat, scales, zeros, out=_flat_inplace(mul, "mul"), accumulate=True)


def q3_gemm(A, qweight, scales, zeros, out=None):
    """out[m][n] = sum_k A[m][k]*(scales[n]*q[k][n] - zeros[n]); A fp16 [M][K]."""
    return _native.q3_gemm(A, qweight, scales, zeros, out)


def dequant_4bit(packed, absmax, n_elems, blocksize, table=NF4, out=None):
    return _native.dequant_4bit(packed, absmax, n_elems, blocksize, table, out)


def dynamic_map():
    """The signed dynamic 8-bit map of bitsandbytes (7 exponent bits), 256 sorted fp32 values in [-1, 1]: the
    table the reference ships as a literal (src/quantBnB-cuda/code.h).  Returns a CPU tensor."""
    import numpy as np
    f32 = np.float32
    vals = []
    for i in range(7):
        items = (1 << i) + 1
        step = (f32(1.0) - f32(0.1)) / f32(items - 1)
        b = [f32(0.1) + step * f32(j) if j < items // 2 else f32(1.0) - step * f32(items - 1 - j) for j in range(items)]
        sc = f32(10.0 ** (-6 + i))
        for j in range(items - 1):
            mean = (b[j] + b[j + 1]) / f32(2.0)
            vals += [sc * mean, -(sc * mean)]
    vals += [f32(0.0), f32(1.0)]
    return torch.from_numpy(np.sort(np.array(vals, dtype=f32)))


def quantize_dynamic8(code, A, out=None):
    return _native.quantize_dynamic8(code, A, out)


def lut_matmul(x, bW, alpha, q_bias, group_size, out=None):
    """matmul(output, input, nqW, m) of src/lut-gemm-hip/kernels.cu:27-31.
    bW uint32/int32 [K/32][nb][N], alpha fp16 [K/G][nb][N], q_bias fp16 [K/G][N] or None."""
    return _native.lut_matmul(x, bW, alpha, q_bias, group_size, out)


def code1x16_matvec(codes, x, codebooks, codebook_a_sizes, codebook_stride_int4, scales=None, out=None):
    """code1x16_matvec of src/quantAQLM-hip/main.cu:103-139 (plus the optional row scale)."""
    return _native.code1x16_matvec(codes, x, codebooks, codebook_a_sizes, codebook_stride_int4, scales, out)


def q3_pack(codes):
    """codes uint8 [K][N] (0..7) -> qweight int32 [3K/32][N]."""
    return _native.q3_pack(codes)


def bcq_pack(signs):
    """signs int8 [K][nb][N] (> 0 means +1) -> bW int32 [K/32][nb][N]."""
    return _native.bcq_pack(signs)


def quantize_4bit(x, blocksize, table=NF4):
    """x fp32/fp16 [n] -> (packed uint8 [ceil(n/2)], absmax fp32 [ceil(n/blocksize)])."""
    return _native.quantize_4bit(x, blocksize, table)


def static_scaled_int8_quant(x, scale, azp=None, out=None):
    """static_scaled_int8_quant of src/quantVLLM-hip/main.cu:133-148; x [tokens][hidden]."""
    return _native.int8_quant_static(x, float(scale), None if azp is None else int(azp), out)


def dynamic_scaled_int8_quant(x, with_azp=False, out=None):
    """dynamic_scaled_int8_quant of src/quantVLLM-hip/main.cu:150-168; returns (out, scales, azp or None)."""
    return _native.int8_quant_dynamic(x, with_azp, out)


def gemv_fp16(mat, vec, out=None):
    """solve_gemv_with_params of src/gemv-hip/gemv.cu:94-133: res = mat @ vec (fp16 in, fp32 sums, fp16 out)."""
    return _native.gemv_fp16(mat, vec, out)


def gemv_int8(mat, vec, scale, zero_point, out=None):
    """solve_gemv_int8_quantized_with_params of src/gemv-hip/gemv.cu:52-92 (mat int8 [rows][n])."""
    return _native.gemv_int8(mat, vec, float(scale), float(zero_point), out)


def gemv_int4(mat, vec, scale, zero_point, out=None):
    """solve_gemv_int4_quantized_with_params of src/gemv-hip/gemv.cu:10-50 (mat uint8 [rows][n/2], low nibble
    first)."""
    return _native.gemv_int4(mat, vec, float(scale), float(zero_point), out)


def mxfp4_qdq(x, out=None):
    """mxfp4<T>() of src/mxfp4-hip/main.cu:144-171: microscaling fp4 quantise-dequantise of an fp16 / bf16 tensor
    whose element count is a multiple of 32."""
    return _native.mxfp4_qdq(x, out)
